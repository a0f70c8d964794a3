// What the streaming and the split-k kernel share: the routing tasks, the wait for
// a phase flag, the register transpose of row-major weights and the combine tasks.
#pragma once
#ifndef FMOE_PARAMS_IN_KERNARG
#define FMOE_PARAMS_IN_KERNARG 1
#endif
#include "moe_device.h"

namespace fmoe {

constexpr int ROUTER_KC = 256;   // k-chunk staged in LDS
constexpr int ROUTER_LD = ROUTER_KC + 4;  // LDS row stride in floats (bank spread)
constexpr int ROUTER_LDS_FLOATS = 2 * ROUTER_EXP * ROUTER_LD;  // per wave

extern __shared__ __align__(16) float lds_dyn[];  // ROUTER_LDS_FLOATS per wave

// The logits are computed by "dot" tasks: one wave takes 8 tokens x 8 experts,
// one (token, expert) chain per lane. Token rows and expert rows arrive with
// fully coalesced 16-byte loads, are converted to float once and staged in the
// wave's private LDS slice in k-chunks, and feed one sequential chain per lane
// (k ascending). Each chain ends as a candidate's ordered_bits in HBM. A "select"
// task per token waits for all of the token's expert groups and picks the
// winners. (bf16 layers of suitable shape run the chains on the matrix core: router_dot16_task.)
// post >= 0: its number among the routing posts, raised in the place of the tokens' counts.
template <typename DT>
__device__ __noinline__ void router_dot_task(ParamsRef pv, int tg, int eg, int post_in = -1, unsigned raised = 0u) {
  ParamsRef p = uniform_params(pv);
  const int post = __builtin_amdgcn_readfirstlane(post_in);
  typedef typename DT::elem elem;
  constexpr int EPV = DT::EPV;
  constexpr int CH_ROW = ROUTER_KC / EPV;               // 16-byte chunks per staged row
  constexpr int NLD = ROUTER_EXP * CH_ROW / 64;         // loads per lane per tile and chunk
  // Params is reached through a generic reference; keep what the loops need in
  // registers so that LDS stores do not force reloads.
  const int H = p.H, E = p.E, T = p.T;
  const int lane = lane_id();
  const int ti = lane >> 3, ei = lane & 7;
  const int t = tg * ROUTER_TOK + ti;
  const int e = eg * ROUTER_EXP + ei;
  float* ws = lds_dyn + (threadIdx.x >> 6) * ROUTER_LDS_FLOATS;  // [ROUTER_EXP][ROUTER_LD]
  float* xs = ws + ROUTER_EXP * ROUTER_LD;                       // [ROUTER_TOK][ROUTER_LD]
  const elem* gate = reinterpret_cast<const elem*>(p.gate);
  const elem* tokens = reinterpret_cast<const elem*>(p.tokens);

  // PF k-chunks of global loads are in flight ahead of the chunk being consumed
  constexpr int PF = 1;  // deeper prefetch measured slower (registers)
  uint4 wr[PF][NLD], xr[PF][NLD];
  auto issue = [&](uint4(&wq)[NLD], uint4(&xq)[NLD], int c0) {  // global -> registers
    if (c0 >= H) return;
    const int ch_row = min(ROUTER_KC, H - c0) / EPV;
#pragma unroll
    for (int i = 0; i < NLD; ++i) {
      // no branches around the loads: rows past the tile (short last chunk)
      // re-read the last row and are dropped when staging
      const int c = i * 64 + lane;
      const int row = min(c / ch_row, ROUTER_EXP - 1), col = c % ch_row;
      const int er = min(eg * ROUTER_EXP + row, E - 1);
      const int tr = min(tg * ROUTER_TOK + row, T - 1);
      wq[i] = ld16(gate + static_cast<size_t>(er) * H + c0 + col * EPV);
      xq[i] = ld16(tokens + static_cast<size_t>(tr) * H + c0 + col * EPV);
    }
  };
  auto stage = [&](const uint4(&wq)[NLD], const uint4(&xq)[NLD], int n) {  // -> float rows in LDS
    const int ch_row = n / EPV;
#pragma unroll
    for (int i = 0; i < NLD; ++i) {
      const int c = i * 64 + lane;
      const int row = c / ch_row, col = c % ch_row;
      if (row < ROUTER_EXP) {
        float wf[EPV], xf[EPV];
        unpack<DT>(wq[i], wf);
        unpack<DT>(xq[i], xf);
#pragma unroll
        for (int q = 0; q < EPV; q += 4) {
          *reinterpret_cast<float4*>(ws + row * ROUTER_LD + col * EPV + q) =
              make_float4(wf[q], wf[q + 1], wf[q + 2], wf[q + 3]);
          *reinterpret_cast<float4*>(xs + row * ROUTER_LD + col * EPV + q) =
              make_float4(xf[q], xf[q + 1], xf[q + 2], xf[q + 3]);
        }
      }
    }
  };

  float acc = 0.0f;
  const float* wrow = ws + ei * ROUTER_LD;
  const float* xrow = xs + ti * ROUTER_LD;
  auto consume = [&](int n) {
    // 32 k per block; the next block's LDS reads are in flight while this
    // block's chain runs (n is a multiple of 64)
    float4 wa[8], xa[8], wb[8], xb[8];
    auto lds_load = [&](float4(&w)[8], float4(&x)[8], int k) {
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        w[q] = *reinterpret_cast<const float4*>(wrow + k + 4 * q);
        x[q] = *reinterpret_cast<const float4*>(xrow + k + 4 * q);
      }
    };
    auto chain = [&](const float4(&w)[8], const float4(&x)[8]) {
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        if constexpr (EPV == 8) {
          acc = __builtin_fmaf(x[q].x, w[q].x, acc);
          acc = __builtin_fmaf(x[q].y, w[q].y, acc);
          acc = __builtin_fmaf(x[q].z, w[q].z, acc);
          acc = __builtin_fmaf(x[q].w, w[q].w, acc);
        } else {
          acc = __fadd_rn(acc, __fmul_rn(x[q].x, w[q].x));
          acc = __fadd_rn(acc, __fmul_rn(x[q].y, w[q].y));
          acc = __fadd_rn(acc, __fmul_rn(x[q].z, w[q].z));
          acc = __fadd_rn(acc, __fmul_rn(x[q].w, w[q].w));
        }
      }
    };
    if (n == ROUTER_KC) {
      // full chunk: straight-line code, so the two register sets simply
      // alternate and no copies are needed between blocks
      lds_load(wa, xa, 0);
#pragma unroll
      for (int k = 0; k < ROUTER_KC; k += 64) {
        lds_load(wb, xb, k + 32);
        chain(wa, xa);
        if (k + 64 < ROUTER_KC) lds_load(wa, xa, k + 64);
        chain(wb, xb);
      }
    } else {
      for (int k = 0; k < n; k += 32) {
        lds_load(wa, xa, k);
        chain(wa, xa);
      }
    }
  };

#pragma unroll
  for (int j = 0; j < PF; ++j) issue(wr[j], xr[j], j * ROUTER_KC);
  for (int c0 = 0; c0 < H; c0 += PF * ROUTER_KC) {
#pragma unroll
    for (int j = 0; j < PF; ++j) {
      const int cj = c0 + j * ROUTER_KC;
      if (cj < H) {
        const int n = min(ROUTER_KC, H - cj);
        stage(wr[j], xr[j], n);
        lds_wave_sync();
        issue(wr[j], xr[j], cj + PF * ROUTER_KC);
        consume(n);
        lds_wave_sync();
      }
    }
  }

  const bool valid = (t < T) && (e < E);
  if (valid) {
    float v = acc;
    if (p.bias != nullptr) v = __fadd_rn(v, as_global(p.bias)[e]);
    stc(&p.cand[static_cast<size_t>(t) * E + e], ordered_bits(v, true));
  }
  fence_release();
  if (post >= 0) {
    raise_post(p, POST_ROUTE, post, raised);
  } else if (ei == 0 && t < T) {
    add_relaxed(&p.tok_arrive[t], 1u);
  }
}

// The same chains on the matrix core, for bf16 layers: V_MFMA_F32_16X16X4_F32 adds
// its four products to the accumulator one after the other in k order, one
// rounding each, so a chain of them is the same sequential sum (and a dependent
// chain issues back to back, 32 cycles an instruction: 512 of them for H = 2048
// against 2048 dependent FMAs on the vector unit). A whole workgroup takes 16
// tokens x 16 experts: wave 0 only multiplies, four waves on the other SIMDs (the float matrix
// instructions and the vector unit of a SIMD take turns: with wave 4, which shares wave 0's, among them one
// token takes 45.0 us instead of 44.3) prepare its operands so that it has nothing else to do: they load 32 bytes of a row (16 k), widen them
// to float and leave them in LDS in the order the instruction wants them: the 16
// k of a group as [k % 4][row][k / 4], so lane l of the multiplying wave (row
// l % 16, k % 4 = l / 16) reads its operand of four consecutive instructions with
// one 16-byte read at 16 * l. Two stages of DOT16_KC k; one workgroup barrier per
// stage; the preparing waves hold the loads of eight stages in registers.
// Called by all eight waves of the workgroup.
constexpr int DOT16_GROUPS = DOT16_KC / 16;             // 16-k groups per stage
constexpr int DOT16_OP_BYTES = DOT16_GROUPS * 1024;     // one operand of one stage
constexpr int DOT16_STAGE_BYTES = 2 * DOT16_OP_BYTES;   // expert rows, then token rows
constexpr int DOT16_AHEAD = 8;                          // stages whose loads are in flight together (even)

__device__ __noinline__ void router_dot16_task(ParamsRef pv, int tg, int eg, int post_in = -1, unsigned raised = 0u) {
  ParamsRef p = uniform_params(pv);
  const int post = __builtin_amdgcn_readfirstlane(post_in);
  const int H = p.H, E = p.E, T = p.T;
  const int lane = lane_id();
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const int nc = H / DOT16_KC;
  unsigned char* lds = reinterpret_cast<unsigned char*>(lds_dyn);
  auto barrier = [] {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  if (wave == 0) {
    f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
    const unsigned char* mine = lds + lane * 16;
    float4 wc, xc, wn, xn;
    barrier();  // stage 0 is written
    wc = *reinterpret_cast<const float4*>(mine);
    xc = *reinterpret_cast<const float4*>(mine + DOT16_OP_BYTES);
    for (int c = 0; c < nc; ++c) {
      const unsigned char* st = mine + (c & 1) * DOT16_STAGE_BYTES;
      const unsigned char* st_next = mine + ((c + 1) & 1) * DOT16_STAGE_BYTES;
#pragma unroll
      for (int g = 0; g < DOT16_GROUPS; ++g) {
        if (g + 1 < DOT16_GROUPS) {
          wn = *reinterpret_cast<const float4*>(st + (g + 1) * 1024);
          xn = *reinterpret_cast<const float4*>(st + DOT16_OP_BYTES + (g + 1) * 1024);
        } else {
          // every read of this stage has returned: the stage may be refilled, and
          // the next one is complete once the others have arrived too
          barrier();
          if (c + 1 < nc) {
            wn = *reinterpret_cast<const float4*>(st_next);
            xn = *reinterpret_cast<const float4*>(st_next + DOT16_OP_BYTES);
          }
        }
        // the reads of the next group go out before this group's instructions, not after
        __builtin_amdgcn_sched_barrier(0);
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(wc.x, xc.x, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(wc.y, xc.y, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(wc.z, xc.z, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(wc.w, xc.w, acc, 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        wc = wn;
        xc = xn;
      }
    }
    // acc[v] of lane l: expert 16*eg + 4*(l/16) + v, token 16*tg + l%16
    const int t = tg * 16 + (lane & 15);
    const int e0 = eg * 16 + 4 * (lane >> 4);
    if (t < T) {
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int e = e0 + v;
        if (e < E) {
          float x = acc[v];
          if (p.bias != nullptr) x = __fadd_rn(x, as_global(p.bias)[e]);
          stc(&p.cand[static_cast<size_t>(t) * E + e], ordered_bits(x, true));
        }
      }
    }
    fence_release();
    if (post >= 0) {
      raise_post(p, POST_ROUTE, post, raised);
    } else if (lane < 16 && t < T) {
      add_relaxed(&p.tok_arrive[t], 1u);
    }
  } else if (wave <= 3 || wave == 5) {  // (waves w and w + 4 share a SIMD)
    // lane -> (row, group): four lanes cover 128 contiguous bytes of a row
    const int hl = min(wave - 1, 3) * 64 + lane;
    const int row = (hl & 63) >> 2;
    const int g = (hl >> 6) * 4 + (hl & 3);
    const unsigned short* wsrc = reinterpret_cast<const unsigned short*>(p.gate) +
                                 static_cast<size_t>(min(eg * 16 + row, E - 1)) * H + g * 16;
    const unsigned short* xsrc = reinterpret_cast<const unsigned short*>(p.tokens) +
                                 static_cast<size_t>(min(tg * 16 + row, T - 1)) * H + g * 16;
    unsigned char* dst = lds + g * 1024 + row * 16;
    struct Regs {
      uint4 w0, w1, x0, x1;
    };
    auto load = [&](Regs& r, int c) {
      const int k = min(c, nc - 1) * DOT16_KC;  // past the end: the last stage again, never written
      r.w0 = ld16(wsrc + k);
      r.w1 = ld16(wsrc + k + 8);
      r.x0 = ld16(xsrc + k);
      r.x1 = ld16(xsrc + k + 8);
    };
    auto widen = [](unsigned char* d, const uint4& a, const uint4& b) {
      // k % 4 = 0 and 1: low and high halves of the even words; 2 and 3: of the odd words
      *reinterpret_cast<uint4*>(d) = make_uint4(a.x << 16, a.z << 16, b.x << 16, b.z << 16);
      *reinterpret_cast<uint4*>(d + 256) =
          make_uint4(a.x & 0xFFFF0000u, a.z & 0xFFFF0000u, b.x & 0xFFFF0000u, b.z & 0xFFFF0000u);
      *reinterpret_cast<uint4*>(d + 512) = make_uint4(a.y << 16, a.w << 16, b.y << 16, b.w << 16);
      *reinterpret_cast<uint4*>(d + 768) =
          make_uint4(a.y & 0xFFFF0000u, a.w & 0xFFFF0000u, b.y & 0xFFFF0000u, b.w & 0xFFFF0000u);
    };
    // The loads of DOT16_AHEAD stages go out together (straight-line code, so each
    // stage waits for exactly its own four): a load takes 2 to 3 us to come back
    // here, three times what the multiplying wave spends on a stage.
    for (int c0 = 0; c0 < nc; c0 += DOT16_AHEAD) {
      Regs r[DOT16_AHEAD];
#pragma unroll
      for (int i = 0; i < DOT16_AHEAD; ++i) load(r[i], c0 + i);
#pragma unroll
      for (int i = 0; i < DOT16_AHEAD; ++i) {
        if (c0 + i < nc) {
          unsigned char* d = dst + (i & 1) * DOT16_STAGE_BYTES;
          widen(d, r[i].w0, r[i].w1);
          widen(d + DOT16_OP_BYTES, r[i].x0, r[i].x1);
          barrier();  // the stage is written; the multiplying wave is done with the one before
        }
      }
    }
    barrier();  // the multiplying wave has read everything: the LDS is free again
  } else {
    for (int c = 0; c <= nc; ++c) barrier();
  }
}

// All expert groups of token t have left their keys: pick the winners.
__device__ __noinline__ void router_select_task(ParamsRef pv, int t) {
  ParamsRef p = uniform_params(pv);
  constexpr int MAXEPL = MAX_EXPERTS / 64;
  const int lane = lane_id();
  unsigned val[MAXEPL];
#pragma unroll
  for (int j = 0; j < MAXEPL; ++j) {
    const int e = lane + 64 * j;
    val[j] = e < p.E ? ldc(&p.cand[static_cast<size_t>(t) * p.E + e]) : 0u;
  }
  if (lane == 0) stc(&p.tok_arrive[t], 0u);
  router_select_max(p, t, val,
                    reinterpret_cast<double*>(lds_dyn + (threadIdx.x >> 6) * ROUTER_LDS_FLOATS));
  const unsigned old = wave_arrive(&p.ctl->router_done.v);
  if (p.early && old == static_cast<unsigned>(p.T) - 1u) broadcast_flag(p, FLAG_ROUTED);
}

// LDS operations of this wave are done, then the workgroup barrier (loads from memory stay in flight)
__device__ __forceinline__ void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// ----------------------------------------------------------------------- waits
// Wave-uniform bounded wait for this workgroup's copy of a phase flag. Only one
// wave of the workgroup polls HBM; the others watch a word in LDS that the
// polling wave sets (1 = flag seen, 2 = failed).
__device__ __forceinline__ bool wait_flag(ParamsRef p, int which, unsigned* lds_flag,
                                          unsigned* lds_poller) {
  int ok = 1;
  if (lane_id() == 0) {
    while (true) {
      const unsigned f = __hip_atomic_load(&lds_flag[which], __ATOMIC_RELAXED,
                                           __HIP_MEMORY_SCOPE_WORKGROUP);
      if (f != 0u) {
        ok = f == 1u;
        break;
      }
      if (__hip_atomic_exchange(&lds_poller[which], 1u, __ATOMIC_RELAXED,
                                __HIP_MEMORY_SCOPE_WORKGROUP) == 0u) {
        // this wave polls for the workgroup
        const unsigned* g = &p.wgflags[blockIdx.x].f[which];
        const long long t0 = wall_clock64();
        unsigned spins = 0;
        unsigned res = 1u;
        while (ld_relaxed(g) == 0u) {
          if ((++spins & 31u) == 0u && ld_relaxed(&p.ctl->error.v) != 0u) {
            res = 2u;
            break;
          }
          if (wall_clock64() - t0 > p.spin_limit) {
            or_relaxed(&p.ctl->error.v, ERR_TIMEOUT);
            res = 2u;
            break;
          }
          __builtin_amdgcn_s_sleep(16);
        }
        __hip_atomic_store(&lds_flag[which], res, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        ok = res == 1u;
        break;
      }
      __builtin_amdgcn_s_sleep(8);
    }
  }
  ok = __builtin_amdgcn_readfirstlane(ok);
  fence_acquire();
  return ok != 0;
}

// The same wait for the first n of a row of posts: the polling wave reads all of them at once, so that nobody counts.
// (A counter takes 90 atomics a microsecond: with 256 workgroups the last one waited up to 3 us for its turn, then
// for the count to come back and for the flags it raised.)
__device__ __forceinline__ bool wait_posts(ParamsRef p, const unsigned* posts, int n, unsigned raised, unsigned* lds_flag,
                                           unsigned* lds_poller) {
  const int lane = lane_id();
  unsigned state = 0u;  // 1: all raised, 2: failed, 3: this wave polls
  if (lane == 0) {
    while (true) {
      state = __hip_atomic_load(lds_flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      if (state != 0u) break;
      if (__hip_atomic_exchange(lds_poller, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) == 0u) {
        state = 3u;
        break;
      }
      __builtin_amdgcn_s_sleep(8);
    }
  }
  state = __builtin_amdgcn_readfirstlane(state);
  if (state == 3u) {
    const CoherentBuffer words = coherent_buffer(posts, static_cast<unsigned>(n) * 4u);
    const long long t0 = wall_clock64();
    unsigned spins = 0;
    state = 1u;
    int at = 4 * lane;  // this lane's next words that may be missing
    while (true) {
      // (The load is no atomic one, which carries 8 bytes at most: without this the compiler may take words it has read.)
      asm volatile("" ::: "memory");
      if (at < n) {
        const uint4 v = ld16_agent(words, static_cast<unsigned>(at) * 4u);
        const bool missing = v.x != raised || (at + 1 < n && v.y != raised) || (at + 2 < n && v.z != raised) || (at + 3 < n && v.w != raised);
        if (!missing) at += 256;
      }
      if (__ballot(at < n) == 0ull) break;
      if ((++spins & 31u) == 0u && __builtin_amdgcn_readfirstlane(ld_relaxed(&p.ctl->error.v)) != 0u) {
        state = 2u;
        break;
      }
      if (wall_clock64() - t0 > p.spin_limit) {
        if (lane == 0) or_relaxed(&p.ctl->error.v, ERR_TIMEOUT);
        state = 2u;
        break;
      }
      __builtin_amdgcn_s_sleep(24);  // (8: row-major T=48 0.7 % slower, one token 0.2 us faster)
    }
    if (lane == 0) __hip_atomic_store(lds_flag, state, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  }
  fence_acquire();
  return state == 1u;
}

// ---------------------------------------------------------- row-major weights
// Fragments of the caller's row-major weights: a fragment wants lane l to hold row l % 16,
// 16-byte chunk l / 16 of a 64-byte row segment, which read that way makes every lane of a
// load touch a line of its own.
// So lane l loads chunk l % 4 of row l / 4 instead, four neighbouring lanes one contiguous
// 64-byte segment, and the fragment is put right in registers afterwards: lane l takes the
// four dwords of lane 4 * (l % 16) + l / 16 (ds_bpermute_b32: the LDS crossbar, no LDS memory).
__device__ __forceinline__ uint4 fragment_from_row_order(const uint4& v, int pull_from) {
  uint4 r;
  r.x = static_cast<unsigned>(__builtin_amdgcn_ds_bpermute(pull_from, static_cast<int>(v.x)));
  r.y = static_cast<unsigned>(__builtin_amdgcn_ds_bpermute(pull_from, static_cast<int>(v.y)));
  r.z = static_cast<unsigned>(__builtin_amdgcn_ds_bpermute(pull_from, static_cast<int>(v.z)));
  r.w = static_cast<unsigned>(__builtin_amdgcn_ds_bpermute(pull_from, static_cast<int>(v.w)));
  return r;
}
// row and 16-byte chunk (of the 64-byte segment of one k-step) that this lane loads of a
// 16-row weight block in the caller's row-major layout
__device__ __forceinline__ int row_order_row() { return lane_id() >> 2; }
__device__ __forceinline__ int row_order_chunk() { return lane_id() & 3; }

// -------------------------------------------------------------------- combine
// out[t, c0..c0+256) = sum over slots, in slot order, of the weighted rows
// (refFullMoe.h:35,62-65; src/hip/kernel/tasks/internal/reduceBlock.h:35-53).
template <typename DT>
__device__ void combine_task(ParamsRef p, int t, int chunk) {
  const int lane = lane_id();
  const int c = chunk * COMBINE_COLS + lane * 4;
  if (c < p.H) {
    float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
    // eight slots at a time: their validity and their rows are loaded together
    // (one memory latency per group instead of two per slot), then added in slot order
    for (int k0 = 0; k0 < p.K; k0 += 8) {
      int idx[8];
      uint4 v[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const int kk = min(k0 + k, p.K - 1);
        idx[k] = ldc(&p.topk_idx[static_cast<size_t>(t) * p.K + kk]);
        v[k] = ld16_once(p.y + (static_cast<size_t>(t) * p.K + kk) * p.H + c);
      }
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        if (k0 + k < p.K && idx[k] >= 0) {
          s.x += __uint_as_float(v[k].x);
          s.y += __uint_as_float(v[k].y);
          s.z += __uint_as_float(v[k].z);
          s.w += __uint_as_float(v[k].w);
        }
      }
    }
    const size_t off = static_cast<size_t>(t) * p.H + c;
    if (p.residual != nullptr) {  // output = input row + layer, the row added last
      if constexpr (DT::EPV == 8) {
        const unsigned long long xx = *as_global(
            reinterpret_cast<const unsigned long long*>(reinterpret_cast<const unsigned short*>(p.residual) + off));
        const uint2 x = make_uint2(static_cast<unsigned>(xx), static_cast<unsigned>(xx >> 32));
        s.x += bf16_lo(x.x);
        s.y += bf16_hi(x.x);
        s.z += bf16_lo(x.y);
        s.w += bf16_hi(x.y);
      } else {
        const uint4 x = ld16(reinterpret_cast<const float*>(p.residual) + off);
        s.x += __uint_as_float(x.x);
        s.y += __uint_as_float(x.y);
        s.z += __uint_as_float(x.z);
        s.w += __uint_as_float(x.w);
      }
    }
    if constexpr (DT::EPV == 8) {
      uint2 pk;
      pk.x = f2bf(s.x) | (f2bf(s.y) << 16);
      pk.y = f2bf(s.z) | (f2bf(s.w) << 16);
      *reinterpret_cast<uint2*>(reinterpret_cast<unsigned short*>(p.out) + off) = pk;
    } else {
      *reinterpret_cast<float4*>(reinterpret_cast<float*>(p.out) + off) = s;
    }
  }
  // the selection masks are dead once the permutation is written: clear this
  // token block's words for the next launch
  if (chunk == 0 && (t & 63) == 0) {
    for (int e = lane; e < p.E; e += 64) stc(&p.masks[static_cast<size_t>(e) * p.W + (t >> 6)], 0ull);
  }
}

// The combine items slot, slot + n_workers, ... of one worker (a function of its
// own so that the worker loop's registers are not shared with it).
template <typename DT>
__device__ __noinline__ void combine_items(ParamsRef pv, unsigned slot, unsigned nc,
                                           unsigned ncomb, unsigned worker, unsigned id0,
                                           long long t_fetch) {
  ParamsRef p = uniform_params(pv);
  const int lane = lane_id();
  for (unsigned q = slot; q < nc; q += static_cast<unsigned>(p.n_workers)) {
    const long long t_item = p.trace ? wall_clock64() : 0;
    combine_task<DT>(p, static_cast<int>(q / ncomb), static_cast<int>(q % ncomb));
    const unsigned id = id0 + q;
    if (p.trace && lane == 0 && id < p.trace_cap) {
      const long long t_end = wall_clock64();
      TraceRec* r = p.trace + id;
      st16(r, u32x4{id, 5u, worker, q / ncomb});
      st16(reinterpret_cast<char*>(r) + 16,
           u32x4{static_cast<unsigned>(t_fetch), static_cast<unsigned>(t_fetch >> 32),
                 static_cast<unsigned>(t_item), static_cast<unsigned>(t_item >> 32)});
      st16(reinterpret_cast<char*>(r) + 32,
           u32x4{static_cast<unsigned>(t_end), static_cast<unsigned>(t_end >> 32), 0u, 0u});
    }
  }
}

}  // namespace fmoe
