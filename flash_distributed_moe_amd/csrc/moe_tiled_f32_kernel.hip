// Persistent MoE kernel, tiled variant of float32 layers for gfx950: batches where an expert sees
// more rows than a streaming tile shares its weights with.
//
// Two workgroups of 4 waves per CU draw task tickets. Stages as in the bf16 tiled kernel:
//   router   8 tokens x 8 experts a wave (the streaming kernel's chains), then selections of four or two tokens a wave
//   scan, scatter
//   gate/up  (row tile, 128 h columns), down (row tile, 256 output columns): up to 96 token rows x
//            256 weight rows, k stepped by 32; a wave owns 64 weight rows x all token rows
//   combine  (token, 256 columns), as in the streaming kernel
//
// The products run on the bf16 matrix cores, sixteen times as fast as the float32 ones here. Both
// operands are split into three bf16 parts, x = hi + mid + lo: each part is the rest rounded to
// nearest, 8 significant bits each, so the three hold all 24 bits of a float exactly. Of the nine products
// of parts the six largest are accumulated in float32: hi*hi, hi*mid, mid*hi, mid*mid, hi*lo, lo*hi. What
// is left out, mid*lo and lo*mid above all, is below 2^-24 of a product (0.991 * 2^-24 for
// 1.0038986 squared), about as much as one rounding of a float32 multiplication may be off: a sum that has one
// product only can be off by 7.5e-8 where a float32 multiplication is by 5.9e-8. A sum of K products is
// rounded 6*K/32 times instead of K times, which outweighs that from a few products on (K=128: 2.5 times
// nearer). The layer's error against float64, relative 2-norm, float32
// matrix instructions (streaming kernel) / this: 30B shape T=256 1.85e-6 / 1.72e-6, T=512 1.84e-6 /
// 1.71e-6; E=40, k=5, H=1344, I=736 T=900 1.29e-6 / 1.16e-6; E=10, k=3, H=320, I=2016 T=2000 9.4e-7 / 8.2e-7.
//
// Bound by HBM up to some 40 rows an expert, above by splitting and products together: at T=1024 on the 30B shape
// the matrix cores are busy 44 % of the SIMD cycles, other vector instructions take 30 %, and 2.79 GB are moved
// of the 2.43 GB needed. us, streaming / this, 30B shape: T=256 586 / 444, T=512 800 / 466, T=1024 1077 / 585
// (77 GFLOP: 132 TFLOP/s of float32); row-major weights T=1024 1076 / 627; E=32 T=4096 2400 / 1450.
//
// A value that is no finite number, or rounds to none in bf16, has no such parts: its products come
// out as infinities or NaN. One below 2^-102 has parts below the smallest normal bf16 number, which lose
// bits or vanish (an error below 2^-126): that shows where a whole sum is small. A wave whose sums hold an infinity, a NaN
// or a value below 2^-64 that is not zero multiplies that token row again with the float32
// matrix instructions, so such inputs give what they give in the streaming kernel. (Sums of ordinary values do
// not come that near to zero. In a sum of 2^-64 and more, 2^-126 of a weight is less than a float's last bit
// as long as a thousand of the token's values are below 2^28.)
//
// Weights go straight to registers (no other wave of the workgroup reads them), 16 bytes per lane and
// load, one 32-k step ahead, and are split there; token rows are split once per workgroup, on
// their way to LDS. The k of a fragment is permuted the way the loads bring it: lane group g of a
// matrix operand holds k = 4g..4g+3 and 16+4g..16+4g+3 of a step, in both operands.
//
// Replaces, for this regime, the reference's moeKernel (src/hip/kernel/moeKernel.h:37-107).
#include <type_traits>

#include "moe_stream_device.h"
#include "moe_tiled_device.h"

namespace fmoe {

constexpr int F_JB = 6;              // 16-row token blocks of the tallest row tile
constexpr int F_TM = 16 * F_JB;      // 96 token rows
constexpr int F_TN = 256;            // weight rows of a task
constexpr int F_WAVES = T_THREADS / 64;

// LDS of a workgroup: two steps of token rows, [row block][part][lane] of 16 bytes, then
// the tile's rows; the routing tasks use it from its first byte on before that.
constexpr int f_stage_bytes(int jb) { return (jb + (jb & 1)) * 3 * 1024; }
constexpr int F_SIDE_OFF = 2 * f_stage_bytes(F_JB);
constexpr int F_LDS_BYTES = F_SIDE_OFF + F_TM * 8 > F_WAVES * ROUTER_LDS_FLOATS * 4 ? F_SIDE_OFF + F_TM * 8 : F_WAVES * ROUTER_LDS_FLOATS * 4;
static_assert(2 * (F_LDS_BYTES + 256) <= 160 * 1024, "two workgroups a CU");

// four floats -> two words of each part
__device__ __forceinline__ void split4(const uint4& v, u32x4 (&p)[3], int at) {
  const unsigned in[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    float a = __uint_as_float(in[2 * q]), b = __uint_as_float(in[2 * q + 1]);
    const unsigned hi = pack_bf16(a, b);
    a -= bf16_lo(hi);
    b -= bf16_hi(hi);
    const unsigned mid = pack_bf16(a, b);
    a -= bf16_lo(mid);
    b -= bf16_hi(mid);
    p[0][at + q] = hi;
    p[1][at + q] = mid;
    p[2][at + q] = pack_bf16(a, b);
  }
}
__device__ __forceinline__ f32x4 mma_bf16(const u32x4& a, const u32x4& b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// 16 bytes at a lane's offset plus a uniform one; AUX 2: non-temporal
template <int AUX>
__device__ __forceinline__ uint4 ld16_buffer(const CoherentBuffer& b, unsigned off, unsigned uniform_off) {
  const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(b.rsrc, static_cast<int>(off), static_cast<int>(uniform_off), AUX);
  return make_uint4(v.x, v.y, v.z, v.w);
}

// What a task multiplies. Weight block i (16 of the wave's 64 rows): this lane's 16 bytes of the
// k-step of 16 number q are at wbase + woff + wblock[i] + q * wstep.
struct FloatOperands {
  const unsigned char* wbase;  // uniform
  unsigned woff;               // this lane's 16 bytes of block 0, k-step 0
  unsigned wblock[4];          // uniform: bytes from block 0 to block i
  unsigned wstep;              // uniform
  const unsigned char* tbase;  // uniform: tokens or h
  unsigned toff[F_JB];         // this thread's 16 bytes of token load q at step 0
  int ksteps;                  // k / 32
};

// acc[i][j] = weight block i x token block j over ksteps * 32 k. Step k, from the loads of the steps
// before it: its weights are split, the token rows of step k+1 are split and go to the other LDS
// buffer, the loads of the token rows of k+2 and of the weights of k+1 go out, then the products.
// The splitting (44 vector instructions a weight block and step) is what the step pays for beside the
// products; the other wave of the SIMD multiplies meanwhile. A second step of weights in flight gained
// nothing (30B shape, us, T=512 490 against 466, T=768 536 / 522, T=1024 585 / 585), nor did splitting
// the next step's weights between the products of this one (two sets of parts do not fit the
// registers: T=768 641, T=1024 753).
template <int JB, bool ONCE>
__device__ __forceinline__ void float_gemm(const FloatOperands& op, f32x4 (&acc)[4][JB]) {
  const int tid = threadIdx.x, lane = tid & 63;
  const int r16 = lane & 15, g = lane >> 4;
  unsigned char* lds = reinterpret_cast<unsigned char*>(lds_dyn);
  // The 16-byte slot of (lane group g, row r) in a fragment: 16 g + (r ^ 4 g), so that the rows and
  // groups a wave writes together fall into different banks.
  const int rd = (16 * g + (r16 ^ (4 * g))) * 16;
  // Token load q brings 16 bytes (four k) of row 32 q + tid / 8: chunk tid % 8 of the row's 128 bytes.
  const int c = tid & 7, trow = tid >> 3;
  const int wr = (trow >> 4) * 3072 + ((c & 3) * 16 + ((trow & 15) ^ (4 * (c & 3)))) * 16 + (c >> 2) * 8;
  constexpr int NT = (JB + 1) / 2;
  const bool odd_half = (JB & 1) && tid >= 128;  // uniform in a wave: rows of the last load that do not exist

  // (through buffer descriptors: a lane offset and a uniform one, no 64-bit address per lane)
  const CoherentBuffer wbuf = coherent_buffer(op.wbase, 0xFFFFFFFFu), tbuf = coherent_buffer(op.tbase, 0xFFFFFFFFu);
  uint4 tr[NT], aw[4][2];
  auto load_t = [&](int k) {
#pragma unroll
    for (int q = 0; q < NT; ++q) tr[q] = ld16_buffer<0>(tbuf, op.toff[q], static_cast<unsigned>(k) * 128u);
  };
  auto store_t = [&](int buf) {
#pragma unroll
    for (int q = 0; q < NT; ++q) {
      u32x4 p[3];
      split4(tr[q], p, 0);
      if (q + 1 < NT || !odd_half) {
#pragma unroll
        for (int m = 0; m < 3; ++m)
          *reinterpret_cast<uint2*>(lds + buf * f_stage_bytes(JB) + q * 6144 + m * 1024 + wr) = make_uint2(p[m][0], p[m][1]);
      }
    }
  };
  auto load_w = [&](int k) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        aw[i][h] = ld16_buffer<ONCE ? 2 : 0>(wbuf, op.woff, static_cast<unsigned>(2 * k + h) * op.wstep + op.wblock[i]);
      }
  };
  const int last = op.ksteps - 1;
  load_t(0);
  load_w(0);
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < JB; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  store_t(0);
  load_t(min(1, last));
  lds_barrier();
  auto step = [&](int k, auto b_tag) {
    constexpr int B = decltype(b_tag)::value;
    u32x4 a[4][3];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      split4(aw[i][0], a[i], 0);
      split4(aw[i][1], a[i], 2);
    }
    store_t(B ^ 1);
    __builtin_amdgcn_sched_barrier(0);
    load_t(min(k + 2, last));
    load_w(min(k + 1, last));
    __builtin_amdgcn_sched_barrier(0);
    // a token block's fragments are read under the products of the one before it, and not earlier
    const unsigned char* st = lds + B * f_stage_bytes(JB) + rd;
    u32x4 b[2][3];
#pragma unroll
    for (int m = 0; m < 3; ++m) b[0][m] = *reinterpret_cast<const u32x4*>(st + m * 1024);
#pragma unroll
    for (int j = 0; j < JB; ++j) {
      if (j + 1 < JB) {
#pragma unroll
        for (int m = 0; m < 3; ++m) b[(j + 1) & 1][m] = *reinterpret_cast<const u32x4*>(st + (j + 1) * 3072 + m * 1024);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int pr = 0; pr < 6; ++pr) {
        constexpr int pa[6] = {0, 2, 1, 0, 1, 0}, pb[6] = {2, 0, 1, 1, 0, 0};
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[i][j] = mma_bf16(a[i][pa[pr]], b[j & 1][pb[pr]], acc[i][j]);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    lds_barrier();
  };
  // The first two steps stand in front of the loop: the compiler counts the loads a wait may leave in
  // flight from the orders of all ways that lead there.
  auto pair = [&](int k) {
    step(k, std::integral_constant<int, 0>{});
    step(k + 1, std::integral_constant<int, 1>{});
  };
  pair(0);  // (k >= 128)
  int k = 2;
  asm volatile("; end of the first pair" ::: "memory");
  for (; k + 1 < op.ksteps; k += 2) pair(k);
  if (k < op.ksteps) step(k, std::integral_constant<int, 0>{});
}

// The weights of an operand: the 64 rows of a wave's column block `wblk`.
template <bool down>
__device__ __forceinline__ void float_weights(ParamsRef p, int expert, int wblk, FloatOperands& op) {
  const int H = uni(p.H), I = uni(p.I), kk = down ? I : H;
  const int lane = threadIdx.x & 63, r16 = lane & 15, g = lane >> 4;
  const bool packed = uni((down ? p.ffn2_packed : p.ffn1_packed) != nullptr ? 1 : 0) != 0;
  const int nw = down ? H / 64 : I / 32;
  op.ksteps = kk >> 5;
  if (packed) {
    op.wbase = uni(reinterpret_cast<const unsigned char*>(down ? p.ffn2_packed : p.ffn1_packed)) + (static_cast<size_t>(expert) * nw + wblk) * (static_cast<size_t>(kk / 16) * 4096);
#pragma unroll
    for (int i = 0; i < 4; ++i) op.wblock[i] = static_cast<unsigned>(i * 1024);
    op.woff = static_cast<unsigned>(lane * 16);
    op.wstep = 4096u;
  } else if (down) {
    op.wbase = uni(reinterpret_cast<const unsigned char*>(p.ffn2)) + (static_cast<size_t>(expert) * H + 64 * wblk) * I * 4;
#pragma unroll
    for (int i = 0; i < 4; ++i) op.wblock[i] = static_cast<unsigned>(16 * i) * static_cast<unsigned>(I * 4);
    op.woff = static_cast<unsigned>(r16) * static_cast<unsigned>(I * 4) + g * 16;
    op.wstep = 64u;
  } else {
    op.wbase = uni(reinterpret_cast<const unsigned char*>(p.ffn1)) + (static_cast<size_t>(expert) * 2 * I + 32 * wblk) * H * 4;
#pragma unroll
    for (int i = 0; i < 4; ++i) op.wblock[i] = static_cast<unsigned>((i & 1) * 16 + (i >> 1) * I) * static_cast<unsigned>(H * 4);
    op.woff = static_cast<unsigned>(r16) * static_cast<unsigned>(H * 4) + g * 16;
    op.wstep = 64u;
  }
}

// Token rows of a tile.
struct RowSet {
  unsigned word[3];  // a bit a row
  __device__ __forceinline__ unsigned any() const { return word[0] | word[1] | word[2]; }
};
static_assert(F_TM <= 96, "rows of a RowSet");
// A sum's place in the order infinity, NaN, zero, small to large; the ordinary ones begin with 2^-64.
__device__ __forceinline__ unsigned sum_order(float x) { return (__float_as_uint(x) << 1) + 0x01000000u; }
constexpr unsigned SUM_ORDINARY = 0x01000000u + ((127u - 64u) << 24);

// One tile task. gate/up: h[row, n0 .. n0+128) (refExpertFFN1.h:51-65); wave w holds gate rows
// n0+32w.. and the matching up rows, so SiLU(gate)*up happens in registers. down:
// y[t*K+slot, n0 .. n0+256) = w * (h[row] . W2[e]^T) (refFullMoe.h:58-65, src/hip/kernel/tasks/ffn2Task.h:37-40),
// float rows with the gate weight applied, as the streaming kernel leaves them. Both are written
// through, 64 bytes of a row at a time, from the accumulators. Returns the token rows for which a sum of
// the wave is no finite number or a small one: float_exact_rows writes those again.
template <int JB, bool down>
__device__ __noinline__ RowSet float_task(ParamsRef pv, int expert_in, int row0_in, int rows_in, int shared_in, int nblk_in) {
  ParamsRef p = uniform_params(pv);
  const int expert = uni(expert_in), row0 = uni(row0_in), rows = uni(rows_in);
  const bool packed = uni((down ? p.ffn2_packed : p.ffn1_packed) != nullptr ? 1 : 0) != 0;
  // weights that no other tile reads pass through the caches without staying; row-major ones come half a
  // line at a time and have to stay
  const bool shared = uni(shared_in) != 0 || !packed;
  const int H = uni(p.H), I = uni(p.I), K = uni(p.K);
  const int tid = threadIdx.x, lane = tid & 63, wave = uni(tid >> 6);
  const int r16 = lane & 15, g = lane >> 4;
  const int nblk = uni(nblk_in);
  const int cols = down ? 64 : 32;                        // of a wave
  const int nw = (down ? H : I) / cols, w0 = nblk * F_WAVES + wave;
  const int wblk = min(w0, nw - 1);
  const int* perm = uni(p.perm) + row0;
  uint2* side = reinterpret_cast<uint2*>(reinterpret_cast<unsigned char*>(lds_dyn) + F_SIDE_OFF);  // row -> (token, slot), weight
  FloatOperands op;
  float_weights<down>(p, expert, wblk, op);
  op.tbase = down ? uni(reinterpret_cast<const unsigned char*>(p.h)) + static_cast<size_t>(row0) * I * 4
                  : uni(reinterpret_cast<const unsigned char*>(p.tokens));
  auto row_offset = [&](int row) {
    const int r = min(row, rows - 1);
    return down ? static_cast<unsigned>(r) * static_cast<unsigned>(I * 4)
                : static_cast<unsigned>(ldc(&perm[r]) / K) * static_cast<unsigned>(H * 4);
  };
#pragma unroll
  for (int q = 0; q < (JB + 1) / 2; ++q) op.toff[q] = row_offset(32 * q + (tid >> 3)) + (tid & 7) * 16;
  if (down && tid < rows)
    side[tid] = make_uint2(static_cast<unsigned>(ldc(&perm[tid])), __float_as_uint(ldc(&uni(p.row_w)[row0 + tid])));

  f32x4 acc[4][JB];
  if (shared) {
    float_gemm<JB, false>(op, acc);
  } else {
    float_gemm<JB, true>(op, acc);
  }
  RowSet again = {{0u, 0u, 0u}};
  if (w0 >= nw) return again;  // this wave's columns do not exist: it has multiplied the last ones that do
  unsigned least = 0xFFFFFFFFu;
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < JB; ++j)
#pragma unroll
      for (int v = 0; v < 4; ++v) least = min(least, sum_order(acc[i][j][v]));
  if (__any(least < SUM_ORDINARY)) {
#pragma unroll
    for (int j = 0; j < JB; ++j) {
      bool odd = false;
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int v = 0; v < 4; ++v) odd |= sum_order(acc[i][j][v]) < SUM_ORDINARY && acc[i][j][v] != 0.0f;
      const unsigned long long b = __ballot(odd && 16 * j + r16 < rows);  // a row's lanes stand 16 apart
      const unsigned both = static_cast<unsigned>(b) | static_cast<unsigned>(b >> 32);
      again.word[j >> 1] |= ((both | both >> 16) & 0xFFFFu) << (16 * (j & 1));
    }
  }

  if (!down) {
    float* h = uni(reinterpret_cast<float*>(p.h)) + static_cast<size_t>(row0) * I + 32 * w0 + 4 * g;
#pragma unroll
    for (int j = 0; j < JB; ++j) {
      const int row = 16 * j + r16;
      if (row < rows) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          unsigned hv[4];
#pragma unroll
          for (int v = 0; v < 4; ++v) hv[v] = __float_as_uint(silu_mul(acc[i][j][v], acc[2 + i][j][v]));
          st16_through(h + static_cast<size_t>(row) * I + 16 * i, make_uint4(hv[0], hv[1], hv[2], hv[3]));
        }
      }
    }
  } else {
    float* y = uni(p.y) + 64 * w0 + 4 * g;
#pragma unroll
    for (int j = 0; j < JB; ++j) {
      const int row = 16 * j + r16;
      if (row < rows) {
        const uint2 d = side[row];
        const float w = __uint_as_float(d.y);
#pragma unroll
        for (int i = 0; i < 4; ++i)
          st16_through(y + static_cast<size_t>(d.x) * H + 16 * i,
                       make_uint4(__float_as_uint(acc[i][j][0] * w), __float_as_uint(acc[i][j][1] * w),
                                  __float_as_uint(acc[i][j][2] * w), __float_as_uint(acc[i][j][3] * w)));
      }
    }
  }
  return again;
}

// The `again` rows of this wave's columns with the float32 matrix instructions, 16 at a time: operands straight
// from memory, the wave on its own, EXACT_AHEAD steps of 16 k in flight. Every task of an infinite token's
// experts does this (a NaN token has none), so the launch waits for it. us, 30B shape, packed, without / with
// one / with eight infinite tokens: T=160 440 / 520 / 527, T=256 455 / 537 / 548, T=1024 598 / 650 / 657 (whole
// blocks of the tile, no step in flight:
// T=160 434 / 630 / 665, T=1024 600 / 1223 / 1257; streaming kernel T=160 546 / 545 / 552, T=1024 1664 / 1668 /
// 1666). A function of its own: inlined in the tasks it cost every launch 1 %.
constexpr int EXACT_AHEAD = 4;
template <bool down>
__device__ __noinline__ void float_exact_rows(ParamsRef pv, int expert_in, int row0_in, int nblk_in, RowSet again) {
  ParamsRef p = uniform_params(pv);
  const int expert = uni(expert_in), row0 = uni(row0_in);
  const int H = uni(p.H), I = uni(p.I), K = uni(p.K);
  const int lane = threadIdx.x & 63, r16 = lane & 15, g = lane >> 4;
  const int w0 = uni(nblk_in) * F_WAVES + uni(static_cast<int>(threadIdx.x >> 6));
  FloatOperands op;
  float_weights<down>(p, expert, w0, op);
  const int n = 2 * op.ksteps;  // (k >= 128: at least EXACT_AHEAD)
  unsigned left[3];
#pragma unroll
  for (int q = 0; q < 3; ++q) left[q] = uni(static_cast<int>(again.word[q]));
  while ((left[0] | left[1] | left[2]) != 0u) {
    int row = 0, found = 0;  // this lane's row: the r16-th of those left, or the last of them
    while (found < 16 && (left[0] | left[1] | left[2]) != 0u) {
      const int q = left[0] != 0u ? 0 : left[1] != 0u ? 1 : 2;
      const unsigned word = q == 0 ? left[0] : q == 1 ? left[1] : left[2];
      if (r16 >= found) row = 32 * q + __builtin_ctz(word);
      ++found;
      if (q == 0) left[0] &= left[0] - 1u;
      if (q == 1) left[1] &= left[1] - 1u;
      if (q == 2) left[2] &= left[2] - 1u;
    }
    const int entry = ldc(&uni(p.perm)[row0 + row]);
    const unsigned char* b = down ? reinterpret_cast<const unsigned char*>(p.h) + static_cast<size_t>(row0 + row) * I * 4
                                  : reinterpret_cast<const unsigned char*>(p.tokens) + static_cast<size_t>(entry / K) * H * 4;
    b += g * 16;
    uint4 aw[EXACT_AHEAD][4], bt[EXACT_AHEAD];
    f32x4 sum[4];
    auto load = [&](int u, int q) {
      bt[u] = ld16(b + static_cast<size_t>(q) * 64);
#pragma unroll
      for (int i = 0; i < 4; ++i) aw[u][i] = ld16(op.wbase + op.wblock[i] + static_cast<size_t>(q) * op.wstep + op.woff);
    };
    auto multiply = [&](int u) {
#pragma unroll
      for (int i = 0; i < 4; ++i) sum[i] = mma16<F32>(aw[u][i], bt[u], sum[i]);
    };
#pragma unroll
    for (int i = 0; i < 4; ++i) sum[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int u = 0; u < EXACT_AHEAD; ++u) load(u, u);
    int q0 = 0;
#pragma unroll 1
    for (; q0 + EXACT_AHEAD <= n; q0 += EXACT_AHEAD) {
#pragma unroll
      for (int u = 0; u < EXACT_AHEAD; ++u) {
        multiply(u);
        load(u, min(q0 + u + EXACT_AHEAD, n - 1));
        __builtin_amdgcn_sched_barrier(0);
      }
    }
#pragma unroll
    for (int u = 0; u < EXACT_AHEAD - 1; ++u)
      if (q0 + u < n) multiply(u);
    fence_release();  // what the task has written here is overwritten
    if (r16 < found) {
      if (!down) {
        float* h = reinterpret_cast<float*>(p.h) + static_cast<size_t>(row0 + row) * I + 32 * w0 + 4 * g;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          unsigned hv[4];
#pragma unroll
          for (int v = 0; v < 4; ++v) hv[v] = __float_as_uint(silu_mul(sum[i][v], sum[2 + i][v]));
          st16_through(h + 16 * i, make_uint4(hv[0], hv[1], hv[2], hv[3]));
        }
      } else {
        const float w = ldc(&uni(p.row_w)[row0 + row]);
        float* y = p.y + static_cast<size_t>(entry) * H + 64 * w0 + 4 * g;
#pragma unroll
        for (int i = 0; i < 4; ++i)
          st16_through(y + 16 * i, make_uint4(__float_as_uint(sum[i][0] * w), __float_as_uint(sum[i][1] * w),
                                              __float_as_uint(sum[i][2] * w), __float_as_uint(sum[i][3] * w)));
      }
    }
  }
}

// Column block `nblk` of a row tile.
template <bool down>
__device__ __forceinline__ void float_tile(ParamsRef p, const TileDesc& t, int nblk) {
  const int expert = uni(t.expert), row0 = uni(t.row0), rows = uni(t.rows), shared = uni(t.shared);
  RowSet again;
  switch ((rows + 15) >> 4) {
    case 1: again = float_task<1, down>(p, expert, row0, rows, shared, nblk); break;
    case 2: again = float_task<2, down>(p, expert, row0, rows, shared, nblk); break;
    case 3: again = float_task<3, down>(p, expert, row0, rows, shared, nblk); break;
    case 4: again = float_task<4, down>(p, expert, row0, rows, shared, nblk); break;
    case 5: again = float_task<5, down>(p, expert, row0, rows, shared, nblk); break;
    default: again = float_task<6, down>(p, expert, row0, rows, shared, nblk); break;
  }
  if (uni(static_cast<int>(again.any())) != 0) float_exact_rows<down>(p, expert, row0, nblk, again);
}

// ---------------------------------------------------------------- worker loop
// Routing, scan and scatter tasks are handed out statically: every workgroup of the launch is
// resident (two a CU; the launcher asks). The GEMM tasks come from one queue per XCD, as in the bf16
// tiled kernel; the other workgroup of the CU covers what a task waits for at its ends.
// traced: with task records (asked at run time: T=1024 on the 30B shape 577.2 -> 580.2 us)
template <bool traced>
__global__ __launch_bounds__(T_THREADS, 2) __attribute__((disable_tail_calls)) void moe_tiled_f32_kernel(
    const Params params) {
  ParamsRef p = kernel_params();
  __shared__ WgShared sh;
  if (threadIdx.x == 0) {
    sh.ticket = 0u;
    sh.ok = 1u;
    sh.flag[0] = sh.flag[1] = sh.flag[2] = sh.flag[3] = 0u;
  }
  __syncthreads();
  Control* ctl = p.ctl;
  const int T = p.T, E = p.E;
  const int G = static_cast<int>(gridDim.x), b = static_cast<int>(blockIdx.x);
  const int wave = uni(static_cast<int>(threadIdx.x >> 6));
  const int me = wave * G + b, waves = G * F_WAVES;

  const int n_eg = (E + ROUTER_EXP - 1) / ROUTER_EXP;
  const int n_dot = (T + ROUTER_TOK - 1) / ROUTER_TOK * n_eg;
  const bool lane0 = traced && lane_id() == 0, thread0 = traced && threadIdx.x == 0;
  for (int i = me; i < n_dot; i += waves) {
    const long long t0 = trace_clock(traced);
    router_dot_task<F32>(p, i / n_eg, i % n_eg);
    trace_task(p, lane0, i, 0, i, t0, t0);
  }
  const int tok = select_tokens(E, p.K, T);
  for (int i = me; i * tok < T; i += waves) {
    const long long t0 = trace_clock(traced);
    const int n = router_select_tokens_task(p, i, static_cast<unsigned>(n_eg), reinterpret_cast<unsigned char*>(lds_dyn + wave * ROUTER_LDS_FLOATS));
    if (n == 0) break;
    unsigned old = 0;
    if (lane_id() == 0) old = add_relaxed(&ctl->router_done.v, static_cast<unsigned>(n));
    if (uni(static_cast<int>(old)) + n == T) broadcast_flag(p, FLAG_ROUTED);
    trace_task(p, lane0, n_dot + i, 6, i * tok, t0, t0);
  }
  long long t_fetch = trace_clock(traced);
  bool ok = wg_wait_flag(p, FLAG_ROUTED, &sh);
  const int n_es = (E + SCAN_EXPERTS - 1) / SCAN_EXPERTS;
  const unsigned t_scan0 = static_cast<unsigned>(n_dot + T), t_scatter0 = t_scan0 + n_es;
  if (ok && b < n_es) {
    const long long t_ready = trace_clock(traced);
    tiled_expert_scan_task(p, b);
    if (wg_arrive<false>(&ctl->scan_done.v, &sh) == static_cast<unsigned>(n_es) - 1u) tiled_scan_task<F_TM, 16>(p);
    trace_task(p, thread0, t_scan0 + b, 1, b, t_fetch, t_ready);
  }
  t_fetch = trace_clock(traced);
  if (ok) ok = wg_wait_flag(p, FLAG_SCAN, &sh);
  const int n_sc = (T + RT_TOK - 1) / RT_TOK;
  for (int i = b; ok && i < n_sc; i += G) {
    const long long t_ready = trace_clock(traced);
    tiled_scatter_task(p, i);
    if (wg_arrive<false>(&ctl->perm_done.v, &sh) == static_cast<unsigned>(n_sc) - 1u) wg_broadcast_flag(p, FLAG_PERM);
    trace_task(p, thread0, t_scatter0 + i, 2, i, t_fetch, t_ready);
  }
  if (ok) ok = wg_wait_flag(p, FLAG_PERM, &sh);

  const unsigned nm = ok ? ldc(&ctl->n_mtiles.v) : 0u;
  const unsigned nt1 = static_cast<unsigned>((p.I + 127) / 128), nt2 = static_cast<unsigned>((p.H + 255) / 256);
  const unsigned n2_total = nm * nt2;
  const unsigned t_dyn0 = t_scatter0 + n_sc;
  const int home = xcc_id();
  // While neither projection has more tasks than there are CUs, only the first workgroup of each (b and b + G/2 share
  // one) takes tasks. Whoever came first did before, and where both of a CU's had one they took 73 us instead of 59 (down) or
  // 134 instead of 113 (gate/up), for which the launch waited (E=3, k=3, H=2048, I=1024, T=300: some 8 of 96 tasks).
  // us, everybody / so: that layer 243 / 226, T=600 293 / 252; E=13, k=8 T=64 200 / 183; E=16, k=2, T=300 200 / 182; E=32, k=4, T=200 (256
  // tasks each) 234 / 196; I=512: H=1024, E=16, T=2000 172 / 152, E=3, T=64 level. With more tasks than CUs a second workgroup is needed.
  const unsigned half = static_cast<unsigned>(G) / 2u;
  const bool takes = static_cast<unsigned>(b) < half || nm * nt1 > half || n2_total > half;
  for (int hop = 0; ok && takes && hop < 8; ++hop) {
    const unsigned q = static_cast<unsigned>((home + hop) & 7);
    const unsigned lo = nm * q / 8u, hi = nm * (q + 1u) / 8u;
    const unsigned q1 = (hi - lo) * nt1, q2 = (hi - lo) * nt2;
    while (ok) {
      t_fetch = trace_clock(traced);
      if (threadIdx.x == 0) sh.ticket = add_relaxed(&ctl->xq[q].v, 1u);
      __syncthreads();
      const unsigned j = uni(static_cast<int>(sh.ticket));
      __syncthreads();
      if (j >= q1 + q2) break;
      if (j < q1) {
        const unsigned m = lo + j / nt1;
        const long long t_ready = trace_clock(traced);
        const TileDesc tile = ld_tile(&p.mtiles[m]);
        float_tile<false>(p, tile, static_cast<int>(j % nt1));
        wg_arrive<false>(&p.g1_done[m].v, &sh);
        trace_task(p, thread0, t_dyn0 + lo * nt1 + j, 3, m, t_fetch, t_ready);
      } else {
        const unsigned jj = j - q1, m = lo + jj / nt2;
        const TileDesc tile = ld_tile(&p.mtiles[m]);
        ok = wg_wait_ge(p, &p.g1_done[m].v, nt1, &sh);
        if (ok) {
          const long long t_ready = trace_clock(traced);
          float_tile<true>(p, tile, static_cast<int>(jj % nt2));
          if (wg_arrive<false>(&ctl->g2_done.v, &sh) == n2_total - 1u) wg_broadcast_flag(p, FLAG_G2);
          trace_task(p, thread0, t_dyn0 + nm * nt1 + lo * nt2 + jj, 4, m, t_fetch, t_ready);
        }
      }
    }
  }
  t_fetch = trace_clock(traced);
  if (ok && n2_total != 0u) ok = wg_wait_flag(p, FLAG_G2, &sh);
  if (ok) {
    const unsigned ncomb = static_cast<unsigned>((p.H + COMBINE_COLS - 1) / COMBINE_COLS);
    combine_items<F32>(p, static_cast<unsigned>(me), static_cast<unsigned>(T) * ncomb, ncomb, blockIdx.x,
                       t_dyn0 + nm * (nt1 + nt2), t_fetch);
  }

  // The last workgroup out returns every counter to zero for the next launch.
  fence_release();
  __syncthreads();
  if (threadIdx.x == 0) sh.ok = (add_relaxed(&ctl->exit_count.v, 1u) == static_cast<unsigned>(G) - 1u) ? 1u : 0u;
  __syncthreads();
  if (sh.ok) {
    const unsigned err = ldc(&ctl->error.v);
    if (err != 0u) {
      recover_after_error(p, err, static_cast<int>(threadIdx.x), T_THREADS);
      __syncthreads();
    }
    const unsigned nmr = min(ldc(&ctl->n_mtiles.v), static_cast<unsigned>(p.max_mtiles));
    for (unsigned i = threadIdx.x; i < nmr; i += T_THREADS) stc(&p.g1_done[i].v, 0u);
    for (int i = threadIdx.x; i < G; i += T_THREADS)
      for (int f = 0; f < 4; ++f) stc(&p.wgflags[i].f[f], 0u);
    if (threadIdx.x < 8) stc(&ctl->xq[threadIdx.x].v, 0u);
    if (threadIdx.x == 0) {
      stc(&ctl->launches.v, ldc(&ctl->launches.v) + 1u);
      stc(&ctl->router_done.v, 0u);
      stc(&ctl->scan_done.v, 0u);
      stc(&ctl->perm_done.v, 0u);
      stc(&ctl->g2_done.v, 0u);
      stc(&ctl->n_mtiles.v, 0u);
      stc(&ctl->exit_count.v, 0u);
    }
  }
}

namespace {
const auto kPlain = moe_tiled_f32_kernel<false>, kTraced = moe_tiled_f32_kernel<true>;
}  // namespace

hipError_t launch_tiled_f32_kernel(const Params& p, int grid, hipStream_t stream) {
  hipLaunchKernelGGL(p.trace ? kTraced : kPlain, dim3(grid), dim3(T_THREADS), F_LDS_BYTES, stream, p);
  return hipGetLastError();
}

hipError_t prepare_tiled_f32_kernel() {
  for (auto kernel : {kPlain, kTraced}) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, F_LDS_BYTES);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

// the lesser of the two kernels' numbers of workgroups a CU holds
hipError_t tiled_f32_kernel_occupancy(int* per_cu) {
  *per_cu = 0x7FFFFFFF;
  for (auto kernel : {kPlain, kTraced}) {
    int n = 0;
    const hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, kernel, T_THREADS, F_LDS_BYTES);
    if (e != hipSuccess) return e;
    if (n < *per_cu) *per_cu = n;
  }
  return hipSuccess;
}

}  // namespace fmoe
