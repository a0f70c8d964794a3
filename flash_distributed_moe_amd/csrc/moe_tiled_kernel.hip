// Persistent MoE kernel, tiled variant for gfx950: the shape for batches where an
// expert sees many rows (prefill) and the layer is bound by matrix throughput,
// bf16 only.
//
// One workgroup of 4 waves per CU (one per SIMD, each with the SIMD's whole
// register file) draws workgroup-wide task tickets from the same kind of counter
// as the streaming variant; tasks depend only on tasks with smaller tickets.
// Stages (ticket order):
//   router   16 tokens x all experts: logits in the oracle's summation order as
//            chains of f32 matrix instructions, then top-k / softmax
//   scan     one wave per expert: counts and running prefixes of its mask
//            words; then one short task: offsets and the row-tile table
//   scatter  32 tokens: permuted row of every (token, slot)
//   gate/up  (row tile, 128 h columns): 256 token rows x 256 weight rows, gate
//            and up rows side by side so that SiLU(gate)*up happens in registers
//   down     (row tile, 256 output columns): same tile, bf16 rows to y (ragged shapes: weighted float rows)
//   combine  1 to 8 tokens: out = sum over slots of y
// GEMM tile: up to 320 token rows x 256 weight rows, K stepped by 64; each wave
// owns 64 weight rows x all token rows of it as 4 x (2*JT) MFMA 16x16x32 blocks
// (JT = 32-row blocks of the tile), up to 320 accumulator registers. Two
// pipelines: both operands through LDS stages (row-major weights, tall tiles), or
// packed weights straight to registers and token rows through LDS. Weight rows
// are the MFMA "A" operand so that a lane ends up with runs of 4 consecutive
// output columns of one token row. A tile with fewer rows multiplies fewer token blocks, so its
// time follows its rows.
//
// Replaces, for this regime, the reference's moeKernel
// (src/hip/kernel/moeKernel.h:37-107) and its TILE_M=1 GEMV tiles
// (src/hip/kernel/tasks/internal/gemmImpl/basicGemmTileImpl.h:14-94).
#include <type_traits>
#include <utility>

#include "moe_stream_device.h"
#include "moe_tiled_device.h"

namespace fmoe {

constexpr int JT_MAX = 10;         // 32-row token blocks of the tallest row tile
constexpr int TM_MAX = 32 * JT_MAX;  // 320 token rows
constexpr int TN = 256;            // weight rows per tile
constexpr int KS = 64;             // k per LDS stage
constexpr int ROWB = KS * 2;       // bytes of a row per stage: one 128-byte line
constexpr int WAVES = T_THREADS / 64;  // one per SIMD
constexpr int NLD = 8;             // 8-row loads per wave, operand and stage
constexpr int G1_COLS = TN / 2;    // h columns per gate/up task
constexpr int CMB_TOK = 8;         // tokens per combine task at most

extern __shared__ __align__(16) unsigned char lds_raw[];

// ------------------------------------------------- direct-to-LDS load helpers
#define FMOE_G1 __attribute__((address_space(1)))
#define FMOE_L3 __attribute__((address_space(3)))

// wait until at most N of this wave's vector-memory operations are outstanding
// (they complete in order); nothing else is waited for
template <int N>
__device__ __forceinline__ void wait_vm() {
  __builtin_amdgcn_s_waitcnt((N & 15) | (7 << 4) | (15 << 8) | ((N >> 4) << 14));
}

// One wave-wide 16-byte-per-lane load from global memory straight into LDS:
// lane l's 16 bytes from base + off land at LDS byte address lds_addr + 16*l.
// Written as assembly so that the compiler does not order LDS reads of other
// stages behind it; completion is tracked by hand with wait_vm.
__device__ __forceinline__ void load_to_lds(unsigned off, const unsigned char* base, unsigned lds_addr) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
               :
               : "v"(off), "s"(base), "s"(lds_addr)
               : "memory");
}


typedef unsigned v4u_t __attribute__((ext_vector_type(4)));
// 16 bytes of LDS at a byte address. The k-loops address LDS by number: the dynamic block's
// base is looked up in memory wherever its name is used inside a function that is not inlined,
// and a scalar load in the loop makes every LDS read in flight be waited for.
__device__ __forceinline__ v4u_t lds_read16(unsigned addr) {
  return *(const FMOE_L3 v4u_t*)addr;
}

// --------------------------------------------------------------------- router
// Logits as in test/singleGPU/cpp/moe/reference/refGemm.h:21-24: one chain per
// output, k ascending, one rounding per step. The chain runs on the matrix
// core: V_MFMA_F32_16X16X4_F32 adds its four products to the accumulator one after
// the other in k order (checked bit for bit against a CPU fmaf chain), and a product
// of two bf16 values is exact in float, so every step is the oracle's acc = fmaf(x, w, acc).
// A task is 16 or 32 tokens x a slab of 128 experts; a wave carries the 16x16 chains of
// its 32 experts (16w..16w+15 and 64+16w..64+16w+15) and each block of 16 tokens.
//
// Bound by the float matrix instructions: 32 cycles each, and the SIMD's vector unit does nothing else
// meanwhile (measured: four of them take 128 cycles, with one vector instruction between them 141, with four 159,
// with eight 203). So the loop has none: lane l multiplies row l % 16 of both operands at k = 4*g + l/16, and
// DS_READ_U16_D16_HI brings that bf16 into the upper half of a register whose lower half stays zero: the
// float itself. 33.8 cycles an instruction, whatever the number of CUs at work. (A byte permute an operand
// behind 16-byte reads: 50; 32x32x2 instructions on such operands: 96 for the 64 they take.) With the
// selection of four tokens a wave, a task at H=2048 with all CUs: 32 tokens 63 -> 43 us, 16 tokens 38 -> 25.6 us.
//
// All waves load: 64 k of the token rows and the 128 expert rows per stage, four stages deep, with coalesced
// direct-to-LDS loads. Stage rows are 144 bytes (128 of data, 16 of padding), so the reads of 16 rows at one k
// fall into different banks. Token rows are padded to whole wave-wide loads, so a load has one base.
// Then selection as in refTopk.h:36-58 / refMoeGate.h:27-30.
constexpr int RT16_TOK = 16;  // tokens of the small router task; the large one has twice as many
constexpr int RT_ROW_BYTES = 144;
constexpr int RT_STAGES = 4;
constexpr int RT_NL = 6;                                  // loads per wave and stage
constexpr int RT_STAGE_BYTES = WAVES * RT_NL * 1024;      // 24 KiB
constexpr int rt_token_loads(int nb) { return (nb * RT16_TOK * 9 + 63) / 64; }
static_assert(rt_token_loads(2) + 128 * 9 / 64 <= WAVES * RT_NL, "router stage too small");
constexpr int ROUTER_LDS_BYTES = RT_STAGES * RT_STAGE_BYTES + 2 * RT16_TOK * MAX_EXPERTS * 4;
static_assert(WAVES * SELECT_ROWS_BYTES <= RT_STAGES * RT_STAGE_BYTES, "selection scratch exceeds the stages");

// Sixteen groups of 4 k to a stage. A group's operands (one register a block of token or expert rows) pass
// through a ring of four: the group three ahead is asked for in front of a group's instructions. Whole runs of groups
// are one assembly block each, which ends when all of its reads have returned: no register the compiler knows of is
// ever in flight. FMOE_RD: the operands of ring place q, at byte `off` of the rows' stage; FMOE_MM: its instructions.
#define FMOE_RD2(q, off)                                                                                       \
  "ds_read_u16_d16_hi %[x" #q "0], %[xa] offset:" #off "\n\tds_read_u16_d16_hi %[w" #q "0], %[wa] offset:" #off \
  "\n\tds_read_u16_d16_hi %[w" #q "1], %[wa] offset:9216+" #off "\n\tds_read_u16_d16_hi %[x" #q               \
  "1], %[xa] offset:2304+" #off "\n\t"
#define FMOE_RD1(q, off)                                                                                       \
  "ds_read_u16_d16_hi %[x" #q "0], %[xa] offset:" #off "\n\tds_read_u16_d16_hi %[w" #q "0], %[wa] offset:" #off \
  "\n\tds_read_u16_d16_hi %[w" #q "1], %[wa] offset:9216+" #off "\n\t"
#define FMOE_MM1(q)                                                                                            \
  "v_mfma_f32_16x16x4_f32 %[c00], %[x" #q "0], %[w" #q "0], %[c00]\n\tv_mfma_f32_16x16x4_f32 %[c01], %[x" #q   \
  "0], %[w" #q "1], %[c01]\n\t"
#define FMOE_MM2(q)                                                                                            \
  FMOE_MM1(q)                                                                                                  \
  "v_mfma_f32_16x16x4_f32 %[c10], %[x" #q "1], %[w" #q "0], %[c10]\n\tv_mfma_f32_16x16x4_f32 %[c11], %[x" #q   \
  "1], %[w" #q "1], %[c11]\n\t"
#define FMOE_WAIT(n) "s_waitcnt lgkmcnt(" #n ")\n\t"
// ask for the group at `off` into ring place r, multiply the one in place q, wait for the next (all but the `n` reads
// of the two groups behind it)
#define FMOE_STEP2(q, r, off) FMOE_RD2(r, off) FMOE_MM2(q) FMOE_WAIT(8)
#define FMOE_STEP1(q, r, off) FMOE_RD1(r, off) FMOE_MM1(q) FMOE_WAIT(6)
#define FMOE_STEPS(S)                                                                                                 \
  S(0, 3, 24) S(1, 0, 32) S(2, 1, 40) S(3, 2, 48) S(0, 3, 56) S(1, 0, 64) S(2, 1, 72) S(3, 2, 80) S(0, 3, 88) S(1, 0, 96) \
      S(2, 1, 104) S(3, 2, 112) S(0, 3, 120)
#define FMOE_X1 [x00] "+&v"(o.x[0][0]), [x10] "+&v"(o.x[1][0]), [x20] "+&v"(o.x[2][0]), [x30] "+&v"(o.x[3][0])
#define FMOE_X2 FMOE_X1, [x01] "+&v"(o.x[0][1]), [x11] "+&v"(o.x[1][1]), [x21] "+&v"(o.x[2][1]), [x31] "+&v"(o.x[3][1])
#define FMOE_W                                                                                              \
  [w00] "+&v"(o.w[0][0]), [w10] "+&v"(o.w[1][0]), [w20] "+&v"(o.w[2][0]), [w30] "+&v"(o.w[3][0]), [w01] "+&v"(o.w[0][1]), \
      [w11] "+&v"(o.w[1][1]), [w21] "+&v"(o.w[2][1]), [w31] "+&v"(o.w[3][1])
#define FMOE_C1 [c00] "+&v"(acc[0][0]), [c01] "+&v"(acc[0][1])
#define FMOE_C2 FMOE_C1, [c10] "+&v"(acc[1][0]), [c11] "+&v"(acc[1][1])
#define FMOE_ADDR [xa] "v"(xa), [wa] "v"(wa)

template <int NB>
struct RouterRing {
  unsigned x[4][NB], w[4][2];  // (lower halves zero, always)
};
// the first three groups of a stage into their places
template <int NB>
__device__ __forceinline__ void router_first(RouterRing<NB>& o, unsigned xa, unsigned wa) {
  if constexpr (NB == 2)
    asm volatile(FMOE_RD2(0, 0) FMOE_RD2(1, 8) FMOE_RD2(2, 16) FMOE_WAIT(0) : FMOE_X2, FMOE_W : FMOE_ADDR : "memory");
  else
    asm volatile(FMOE_RD1(0, 0) FMOE_RD1(1, 8) FMOE_RD1(2, 16) FMOE_WAIT(0) : FMOE_X1, FMOE_W : FMOE_ADDR : "memory");
}
// groups 0..12 of a stage, and the reads of its last three
template <int NB>
__device__ __forceinline__ void router_stage(RouterRing<NB>& o, f32x4 (&acc)[NB][2], unsigned xa, unsigned wa) {
  if constexpr (NB == 2)
    asm volatile(FMOE_STEPS(FMOE_STEP2) FMOE_WAIT(0) : FMOE_X2, FMOE_W, FMOE_C2 : FMOE_ADDR : "memory");
  else
    asm volatile(FMOE_STEPS(FMOE_STEP1) FMOE_WAIT(0) : FMOE_X1, FMOE_W, FMOE_C1 : FMOE_ADDR : "memory");
}
// groups 13..15, and the first three of the next stage
template <int NB>
__device__ __forceinline__ void router_stage_end(RouterRing<NB>& o, f32x4 (&acc)[NB][2], unsigned xa, unsigned wa) {
  if constexpr (NB == 2)
    asm volatile(FMOE_RD2(0, 0) FMOE_MM2(1) FMOE_RD2(1, 8) FMOE_MM2(2) FMOE_RD2(2, 16) FMOE_MM2(3) FMOE_WAIT(0)
                 : FMOE_X2, FMOE_W, FMOE_C2
                 : FMOE_ADDR
                 : "memory");
  else
    asm volatile(FMOE_RD1(0, 0) FMOE_MM1(1) FMOE_RD1(1, 8) FMOE_MM1(2) FMOE_RD1(2, 16) FMOE_MM1(3) FMOE_WAIT(0)
                 : FMOE_X1, FMOE_W, FMOE_C1
                 : FMOE_ADDR
                 : "memory");
}
// the wait states between the last matrix instruction, which the compiler does not see, and the first read of a sum
template <int NB>
__device__ __forceinline__ void router_settle(f32x4 (&acc)[NB][2]) {
  if constexpr (NB == 2)
    asm volatile("s_nop 15\n\ts_nop 15" : FMOE_C2);
  else
    asm volatile("s_nop 15\n\ts_nop 15" : FMOE_C1);
}

template <int NB>  // blocks of 16 tokens
__device__ __noinline__ void tiled_router_task(ParamsRef pv, int blk) {
  constexpr int NTOK = NB * RT16_TOK;
  constexpr int W_OFF = rt_token_loads(NB) * 1024;  // expert rows in a stage
  ParamsRef p = uniform_params(pv);
  const int T = uni(p.T), E = uni(p.E), H = uni(p.H);
  const unsigned char* tokens = uni(reinterpret_cast<const unsigned char*>(p.tokens));
  const unsigned char* gate = uni(reinterpret_cast<const unsigned char*>(p.gate));
  const float* bias = uni(p.bias);
  unsigned* keys = reinterpret_cast<unsigned*>(lds_raw + RT_STAGES * RT_STAGE_BYTES);  // [NTOK][MAX_EXPERTS]
  const unsigned lds_addr = uni(static_cast<unsigned>(
      reinterpret_cast<size_t>((FMOE_L3 unsigned char*)lds_raw)));
  const int tid = threadIdx.x;
  const int wave = uni(tid >> 6), lane = tid & 63;
  const int t0 = uni(blk) * NTOK;
  const int nsteps = H >> 6;
  const int r16 = lane & 15, kq = lane >> 4;  // row and k of the group
  const unsigned xoff = lds_addr + r16 * RT_ROW_BYTES + 2 * kq;
  const unsigned woff = xoff + W_OFF + wave * 16 * RT_ROW_BYTES;
  RouterRing<NB> o;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    o.w[q][0] = o.w[q][1] = 0u;
#pragma unroll
    for (int n = 0; n < NB; ++n) o.x[q][n] = 0u;
  }
  for (int e0 = 0; e0 < E; e0 += 128) {
    // slot g of the token or the expert rows (16 bytes): position g % 9 of row g / 9 (position 8 is padding); slots
    // past the last row repeat it
    unsigned off[RT_NL];
    const unsigned char* base[RT_NL];
#pragma unroll
    for (int i = 0; i < RT_NL; ++i) {
      const int ld = wave * RT_NL + i;
      const bool tok = ld < rt_token_loads(NB);
      const int g = (tok ? ld : ld - rt_token_loads(NB)) * 64 + lane;
      const int row = tok ? min(min(g / 9, NTOK - 1), T - 1 - t0) : min(min(g / 9, 127), E - 1 - e0);
      off[i] = static_cast<unsigned>(row) * static_cast<unsigned>(H * 2) + static_cast<unsigned>(min(g % 9, 7) * 16);
      base[i] = uni(tok ? tokens + static_cast<size_t>(t0) * H * 2 : gate + static_cast<size_t>(e0) * H * 2);
    }
    auto issue = [&](int step) {  // past the last step: the last one again, into a stage nobody reads
      const size_t koff = static_cast<size_t>(min(step, nsteps - 1)) * 128;
      const unsigned st = lds_addr + (step & (RT_STAGES - 1)) * RT_STAGE_BYTES + wave * (RT_NL * 1024);
#pragma unroll
      for (int i = 0; i < RT_NL; ++i) load_to_lds(off[i], base[i] + koff, st + i * 1024);
    };
    f32x4 acc[NB][2];
#pragma unroll
    for (int n = 0; n < NB; ++n) acc[n][0] = acc[n][1] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int st = 0; st < RT_STAGES; ++st) issue(st);
    wait_vm<(RT_STAGES - 1) * RT_NL>();
    __builtin_amdgcn_s_barrier();  // stage 0 is in
    asm volatile("" ::: "memory");
    router_first<NB>(o, xoff, woff);
    for (int st = 0; st < nsteps; ++st) {
      const unsigned at = static_cast<unsigned>(st & (RT_STAGES - 1)) * RT_STAGE_BYTES;
      const unsigned next = static_cast<unsigned>((st + 1) & (RT_STAGES - 1)) * RT_STAGE_BYTES;
      router_stage<NB>(o, acc, xoff + at, woff + at);  // (this wave no longer reads stage st)
      wait_vm<(RT_STAGES - 2) * RT_NL>();              // its loads of stage st+1 are in
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      issue(st + RT_STAGES);
      // after the last step this reads a stage that is being refilled; the values are never used
      router_stage_end<NB>(o, acc, xoff + next, woff + next);
    }
    router_settle<NB>(acc);
    wait_vm<0>();                  // nothing may land in a stage after this slab
    __builtin_amdgcn_s_barrier();  // the stages may be refilled for the next slab
    asm volatile("" ::: "memory");
    // acc[n][j][v] of lane l: token 16*n + 4*(l/16) + v, expert e0 + 64*j + 16*wave + l%16
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int e = e0 + 64 * j + 16 * wave + r16;
      const float bv = (bias != nullptr && e < E) ? as_global(bias)[e] : 0.0f;
#pragma unroll
      for (int n = 0; n < NB; ++n)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const float x = bias != nullptr ? __fadd_rn(acc[n][j][v], bv) : acc[n][j][v];
          if (e < MAX_EXPERTS) keys[(16 * n + 4 * kq + v) * MAX_EXPERTS + e] = ordered_bits(x, e < E);
        }
    }
  }
  __syncthreads();
  // selection: four tokens of every block of 16 to a wave, in the memory of the stages
#pragma unroll 1
  for (int n = 0; n < NB; ++n) {
    const int tl = 16 * n + 4 * wave + kq;
    const int t = t0 + tl < T ? t0 + tl : -1;
    auto select = [&](auto epl) {
      constexpr int EPL = decltype(epl)::value;
      unsigned val[EPL];
#pragma unroll
      for (int j = 0; j < EPL; j += 4) {
        const uint4 v = *reinterpret_cast<const uint4*>(keys + tl * MAX_EXPERTS + EPL * r16 + j);
        val[j] = v.x;
        val[j + 1] = v.y;
        val[j + 2] = v.z;
        val[j + 3] = v.w;
      }
      router_select_rows<EPL, 16>(p, t, val, lds_raw + wave * SELECT_ROWS_BYTES);
    };
    if (E <= 128) {
      select(std::integral_constant<int, 8>{});
    } else {
      select(std::integral_constant<int, 16>{});
    }
  }
}


// ------------------------------------------------------------ the short router
// The same chains where a batch has too few 16-token tasks for the CUs: 16 tokens x 32 experts a
// workgroup, as the streaming kernel's router_dot16_task does it for 16 experts. Waves 0 and 1 only
// multiply, one 16x16 chain each; waves 2 and 3 load 32 bytes of a row, widen them to float and leave
// them in LDS in the order the instruction wants them (see router_dot16_task), two stages of 256 k, the
// loads of four stages in flight. k past H counts as zero: a sum is never -0, so adding +0 leaves it.
// Bound by the chains (512 dependent instructions of 32 cycles at H=2048). The logits go to memory
// and a wave picks the winners of four tokens once theirs are in.
constexpr int DOT32_AHEAD = 4;
constexpr int DOT32_STAGE_BYTES = 3 * DOT16_OP_BYTES;  // experts 0..15, 16..31, tokens
constexpr int DOT32_LDS_BYTES = 2 * DOT32_STAGE_BYTES;

__device__ __noinline__ void router_dot32_task(ParamsRef pv, int tg_in, int eg_in) {
  ParamsRef p = uniform_params(pv);
  const int H = uni(p.H), E = uni(p.E), T = uni(p.T), tg = uni(tg_in), eg = uni(eg_in);
  const int lane = lane_id();
  const int wave = uni(static_cast<int>(threadIdx.x >> 6));
  const int nc = (H + DOT16_KC - 1) / DOT16_KC;
  const unsigned lds0 = uni(static_cast<unsigned>(reinterpret_cast<size_t>((FMOE_L3 unsigned char*)lds_raw)));
  if (wave < 2) {
    f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
    const unsigned wmine = lds0 + wave * DOT16_OP_BYTES + lane * 16, xmine = lds0 + 2 * DOT16_OP_BYTES + lane * 16;
    v4u_t wc, xc, wn, xn;
    lds_barrier();  // stage 0 is written
    wc = lds_read16(wmine);
    xc = lds_read16(xmine);
    for (int c = 0; c < nc; ++c) {
      const unsigned st = (c & 1) * DOT32_STAGE_BYTES, st_next = ((c + 1) & 1) * DOT32_STAGE_BYTES;
#pragma unroll
      for (int g = 0; g < DOT16_GROUPS; ++g) {
        if (g + 1 < DOT16_GROUPS) {
          wn = lds_read16(wmine + st + (g + 1) * 1024);
          xn = lds_read16(xmine + st + (g + 1) * 1024);
        } else {
          // every read of this stage has returned: it may be refilled, and the next one is
          // complete once the others have arrived too
          lds_barrier();
          if (c + 1 < nc) {
            wn = lds_read16(wmine + st_next);
            xn = lds_read16(xmine + st_next);
          }
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < 4; ++i)
          acc = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(wc[i]), __uint_as_float(xc[i]), acc, 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        wc = wn;
        xc = xn;
      }
    }
    // acc[v] of lane l: expert 32*eg + 16*wave + 4*(l/16) + v, token 16*tg + l%16
    const int t = tg * 16 + (lane & 15);
    const int e0 = eg * 32 + wave * 16 + 4 * (lane >> 4);
    if (eg * 32 + wave * 16 < E) {
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
      if (lane < 16 && t < T) add_relaxed(&p.tok_arrive[t], 1u);
    }
  } else {
    // unit n of this lane: operand n / 2, (row, 16-k group) as in router_dot16_task: four lanes
    // cover 128 contiguous bytes of a row
    const int hl = (wave - 2) * 64 + lane;
    const unsigned short* src[6];
    unsigned dst[6];
    int gk[2];
#pragma unroll
    for (int n = 0; n < 6; ++n) {
      const int idx = hl + 128 * (n & 1);
      const int row = (idx & 63) >> 2, g = (idx >> 6) * 4 + (idx & 3);
      gk[n & 1] = g * 16;
      const unsigned short* base =
          n < 4 ? reinterpret_cast<const unsigned short*>(p.gate) + static_cast<size_t>(min(eg * 32 + 16 * (n >> 1) + row, E - 1)) * H
                : reinterpret_cast<const unsigned short*>(p.tokens) + static_cast<size_t>(min(tg * 16 + row, T - 1)) * H;
      src[n] = base;
      dst[n] = lds0 + (n >> 1) * DOT16_OP_BYTES + g * 1024 + row * 16;
    }
    struct Regs {
      uint4 a[6], b[6];
    };
    auto load = [&](Regs& r, int c) {  // past the last k: the row's first ones again, counted as zero
#pragma unroll
      for (int n = 0; n < 6; ++n) {
        const int k = c * DOT16_KC + gk[n & 1];
        const unsigned short* at = src[n] + (k < H ? k : 0);
        r.a[n] = ld16(at);
        r.b[n] = ld16(at + 8);
      }
    };
    auto widen = [&](const Regs& r, int c) {
#pragma unroll
      for (int n = 0; n < 6; ++n) {
        const unsigned keep = c * DOT16_KC + gk[n & 1] < H ? 0xFFFFFFFFu : 0u;
        const unsigned hi = keep & 0xFFFF0000u;
        const uint4 a = make_uint4(r.a[n].x & keep, r.a[n].y & keep, r.a[n].z & keep, r.a[n].w & keep);
        const uint4 b = make_uint4(r.b[n].x & keep, r.b[n].y & keep, r.b[n].z & keep, r.b[n].w & keep);
        const unsigned d = dst[n] + (c & 1) * DOT32_STAGE_BYTES;
        auto put = [&](unsigned off, unsigned v0, unsigned v1, unsigned v2, unsigned v3) {
          *(FMOE_L3 v4u_t*)(d + off) = v4u_t{v0, v1, v2, v3};
        };
        put(0, a.x << 16, a.z << 16, b.x << 16, b.z << 16);
        put(256, a.x & hi, a.z & hi, b.x & hi, b.z & hi);
        put(512, a.y << 16, a.w << 16, b.y << 16, b.w << 16);
        put(768, a.y & hi, a.w & hi, b.y & hi, b.w & hi);
      }
    };
    Regs r[DOT32_AHEAD];
#pragma unroll
    for (int i = 0; i < DOT32_AHEAD; ++i) load(r[i], i);
    for (int c0 = 0; c0 < nc; c0 += DOT32_AHEAD) {
#pragma unroll
      for (int i = 0; i < DOT32_AHEAD; ++i) {
        if (c0 + i < nc) {
          widen(r[i], c0 + i);
          load(r[i], c0 + i + DOT32_AHEAD);
          lds_barrier();  // the stage is written; the multiplying waves are done with the one before
        }
      }
    }
    lds_barrier();  // the multiplying waves have read everything: the LDS is free again
  }
}

// ------------------------------------------------------- the short scan and scatter
// Where the mask words of the batch fit LDS, the workgroups that write a share of the permutation
// (256 entries each) build the tables they need for it themselves; the first of them also writes
// the row-tile table and what the host may read back.
constexpr int SHORT_PRE_OFF = (SHORT_MASK_WORDS + MAX_EXPERTS) * 8;  // (rows of the mask table have an odd pitch)
constexpr int SHORT_CNT_OFF = SHORT_PRE_OFF + (SHORT_MASK_WORDS + MAX_EXPERTS) * 2;
constexpr int SHORT_OFF_OFF = SHORT_CNT_OFF + MAX_EXPERTS * 4;
constexpr int SHORT_LDS_BYTES = SHORT_OFF_OFF + MAX_EXPERTS * 4;

template <bool RAGGED>
__device__ __noinline__ void short_scatter_task(ParamsRef pv, int blk_in) {
  ParamsRef p = uniform_params(pv);
  const RouteTables r = route_tables(p);
  const int blk = uni(blk_in), tid = threadIdx.x, lane = tid & 63;
  const int wact = (r.T + 63) >> 6, nw = r.E * wact, pitch = wact | 1;
  unsigned long long* lmask = reinterpret_cast<unsigned long long*>(lds_raw);
  unsigned short* lpre = reinterpret_cast<unsigned short*>(lds_raw + SHORT_PRE_OFF);  // rows of the expert before the word
  int* lcnt = reinterpret_cast<int*>(lds_raw + SHORT_CNT_OFF);
  int* loff = reinterpret_cast<int*>(lds_raw + SHORT_OFF_OFF);
  const int i = blk * T_THREADS + tid;
  const int e = i < r.T * r.K ? ldc(&r.topk_idx[i]) : -1;
  float weight = 0.0f;
  if (RAGGED && i < r.T * r.K) weight = ldc(&r.topk_w[i]);
  for (int w0 = tid; w0 < nw; w0 += 4 * T_THREADS) {
    unsigned long long m[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int w = min(w0 + q * T_THREADS, nw - 1);
      m[q] = ldc(&r.masks[static_cast<size_t>(w / wact) * r.W + w % wact]);
    }
#pragma unroll
    for (int q = 0; q < 4; ++q)
      if (w0 + q * T_THREADS < nw) {
        const int w = w0 + q * T_THREADS;
        lmask[w / wact * pitch + w % wact] = m[q];
      }
  }
  __syncthreads();
  if (tid < r.E) {
    int c = 0;
#pragma unroll 4
    for (int w = 0; w < wact; ++w) {
      lpre[tid * pitch + w] = static_cast<unsigned short>(c);
      c += __popcll(lmask[tid * pitch + w]);
    }
    lcnt[tid] = c;
  }
  __syncthreads();
  if (tid < 64) {
    const int epl = (r.E + 63) >> 6;
    int base = 0, tile_base = 0;
    for (int j = 0; j < epl; ++j) {
      const int x = lane + 64 * j;
      const int c = x < r.E ? lcnt[x] : 0;
      const int incl = wave_inclusive_scan(c);
      const int off = base + incl - c;
      if (x < r.E) loff[x] = off;
      if (blk == 0) tile_base = scan_tiles<TM_MAX, 32>(r, x, c, off, tile_base);
      base += __shfl(incl, 63, 64);
    }
    if (blk == 0) scan_totals(p, r, lane, base, tile_base);
  }
  __syncthreads();
  if (blk == 0 && tid < r.E) stc(&r.expert_count[tid], lcnt[tid]);
  if (e >= 0) {
    const int t = i / r.K, wd = t >> 6;
    const int w = e * pitch + wd;
    const int pos = loff[e] + lpre[w] + __popcll(lmask[w] & ((1ull << (t & 63)) - 1ull));
    stc(&r.perm[pos], i);
    if (RAGGED) stc(&r.row_w[pos], weight);
  }
}

// -------------------------------------------------------------- the GEMM tile
// Operands go HBM/L2 -> LDS directly (global_load_lds_dwordx4: lane l's 16 bytes
// land at LDS base + 16*l, from any global address), in stages of 64 k: one
// 128-byte line of every operand row, so every request uses whole cache lines
// whatever the row pitch. Two or three stages; no register staging, no LDS write
// instructions, almost no vector-ALU work in the loop.
//
// One wave per SIMD, each with 64 weight rows x all token rows of the tile:
// acc[4][2*JT] blocks of 16x16. The first 16 token blocks' accumulators fill the
// 256 accumulator registers a[0:255]; a tile of 257..320 rows (JT 9, 10) keeps
// the last blocks' in v[...]. Per 32 k a wave reads 4 weight and 2*JT token
// fragments (16 bytes per lane each) for 8*JT matrix instructions.
//
// Why 16x16x32 and not 32x32x16: at the board's power cap the smaller instruction
// delivers more. Back to back on all CUs with normally distributed operands in
// registers: 32x32x16 1717 TFLOP/s at 1.74 GHz, 16x16x32 1919 TFLOP/s at 1.99 GHz
// (2478 and 2407 on 8 CUs, where the clock stays at 2.4 GHz). Per multiply-add it
// reads twice the operand registers but moves half the accumulators. What it gains is therefore
// there in a row of launches that keep the board at its cap (T=8192 on the 30B shape 769 -> 746 us),
// hardly in one launch behind a pause (792 -> 786), and it costs a little where a few tall tiles
// have the chip to themselves (E=64, k=2, T=700, four hot experts, row-major 128 -> 133 us).
//
// LDS stage layout: rows of 128 bytes, unpadded, weight rows 0..255 then token
// rows. Row R keeps its eight 16-byte chunks permuted: chunk C sits at position
// C ^ ((R >> 1) & 7), so the 16 rows a quarter-wave reads together at one k fall
// into 16 different 16-byte bank groups. One wave-wide load fills 8 rows; lane
// l brings the chunk that belongs at position l & 7 of row l >> 3.
//
// The matrix instructions are written as assembly with the accumulator pinned
// to its register file: 256 accumulators fill a[0:255] exactly, and the
// compiler's own choice moved parts of them in and out of v[...] (it also
// chose the vector-register form of the instruction, which cannot reach a[...]).
// The first instruction of every accumulator takes the constant 0 as its
// addend, so nothing zeroes them.
constexpr int JB_MAX = 2 * JT_MAX;  // 16-row token blocks of the tallest tile
constexpr int JB_ACC = 16;          // of these, the ones whose accumulators are in a[...]

template <bool INIT, bool IN_V>
__device__ __forceinline__ void mma(const v4u_t& a, const v4u_t& b, f32x4& c) {
  if (IN_V) {
    if (INIT) {
      asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, 0" : "=v"(c) : "v"(a), "v"(b));
    } else {
      asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+v"(c) : "v"(a), "v"(b));
    }
  } else {
    if (INIT) {
      asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, 0" : "=a"(c) : "v"(a), "v"(b));
    } else {
      asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
    }
  }
}

// The compiler does not see matrix instructions in the assembly above: keep the wait states between the
// last of them and the first read of an accumulator, and the reads behind them (it may place the reads of what an
// assembly does not name anywhere).
template <int JT>
__device__ __forceinline__ void settle(f32x4 (&acc)[4][JB_MAX]) {
  asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 2 * JT; ++j) {
      if (j < JB_ACC) asm volatile("" : "+a"(acc[i][j])); else asm volatile("" : "+v"(acc[i][j]));
    }
}

constexpr int stage_bytes_of(int jt) { return (TN + 32 * jt) * ROWB; }
// Stages of the LDS-staged pipeline: three where they fit. The tiles of a batch of some 40 to
// 160 rows an expert are bound by how much of the weights is in flight, taller ones are not.
constexpr int nst_of(int jt) { return jt <= 5 ? 3 : 2; }
constexpr int TILE_LDS_BYTES = 3 * stage_bytes_of(5);               // 159744
static_assert(TILE_LDS_BYTES >= 2 * stage_bytes_of(JT_MAX), "stages");
// behind the stages: the tile's destination rows for the down epilogue, and (ragged shapes) their gate weights
constexpr int SIDE_OFF = TILE_LDS_BYTES;
constexpr int SIDE_BYTES = TM_MAX * 8;
// and behind those one 16-byte line of words a GEMM task leaves for the worker loop: the ticket it
// drew for the workgroup's next task. They live in
// the dynamic block because a file-scope LDS variable written from a function that is not
// inlined landed on top of the dynamic block's first bytes.
constexpr int NOTE_OFF = SIDE_OFF + SIDE_BYTES;
constexpr int NOTE_BYTES = 16;
__device__ __forceinline__ unsigned* task_notes() { return reinterpret_cast<unsigned*>(lds_raw + NOTE_OFF); }

struct TileOperands {
  const unsigned char* wbase;  // uniform: the weight matrix (or this wave's packed slice) the offsets are relative to
  const unsigned char* tbase;  // uniform: tokens, or h
  unsigned wstride;            // uniform: bytes from one stage's weights to the next
  bool wpacked;                // uniform: the weights come from the packed layout (see packed_run_offset)
  unsigned wlast, tlast;       // uniform: byte offsets of the last stage's weights and token rows
  unsigned woff[NLD];          // this lane's 16 bytes of weight load q at stage 0
  unsigned toff[10];           // the same for the token rows
};

// Stage row (within its operand) that this lane's part of load q belongs to when a wave
// issues `per_wave` loads per stage, and the byte offset inside the row's 128-byte line of
// the chunk it brings.
__device__ __forceinline__ int stage_row(int per_wave, int q) {
  return ((threadIdx.x >> 6) * per_wave + q) * 8 + ((threadIdx.x & 63) >> 3);
}
__device__ __forceinline__ unsigned stage_chunk_bytes(int row) {
  return static_cast<unsigned>(((threadIdx.x & 7) ^ ((row >> 1) & 7)) << 4);
}

// f(integral_constant<int, 0>) ... f(integral_constant<int, N - 1>)
template <typename F, int... I>
__device__ __forceinline__ void static_for_(F&& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
  static_for_(f, std::make_integer_sequence<int, N>{});
}

// A stage is NSL = 4*JT slots, two sub-steps (32 k each) of 2*JT: slot n multiplies token
// block n % (2*JT) of its sub-step with the wave's four weight blocks, four instructions of
// 16 cycles. The token fragments pass through a ring of registers: a slot's fragment is
// replaced, as soon as its instructions have been issued, by the one RING slots later, so
// every LDS read has RING * 64 cycles to return. RING divides the slots of a stage.
constexpr int ring_of(int jt) { return jt == 2 ? 4 : jt == 3 ? 6 : jt == 5 ? 5 : jt == 7 ? 7 : jt == 9 ? 6 : 8; }

// acc[i][j] = weight block i (16 of this wave's 64 weight rows) x token block j (16 rows),
// j < 2*JT, over nstages * 64 k (nstages >= 2). Token rows from 32*JT on are neither loaded
// nor multiplied.
//
// Hand-over between stages BAR slots after the last fragment of stage s has been asked for:
// this wave's reads of stage s have returned and its loads of stage s+1 have landed, then
// the workgroup barrier; from there on the next stage's first fragments are read and the
// loads of stage s+NST go out into the buffer just left, LPS per slot, the rest under the next
// stage's first slots. (With the 32x32 form of this loop, on all 256 CUs: all 16 loads behind
// the barrier at once, barrier in front of the sub-step: 51 us per 256x256x2048 tile; spread
// out: 48 us.)
//
// Bookkeeping rides along: at the first hand-over (every memory operation this wave issued
// before it, the previous task's stores included, has completed there anyway) thread 0
// signals the previous task's completion on `pend` (if any) and draws the workgroup's next
// ticket from `queue` into `next`, so neither trip to memory is waited for between tasks.
//
// HALF: k is an odd number of 32-k steps. The last stage then covers the last 64 k, the first 32
// of which the stage before it has multiplied already, and only its second sub-step runs (`wlast`,
// `tlast`: the byte offsets of the last stage's operands, which no stage's exceed). A template
// parameter and not a branch: where two ways part or meet the compiler may copy accumulators, and
// it does not know that a matrix instruction in assembly has yet to write them.
template <int JT, bool HALF, typename AfterFirstLoads>
__device__ __forceinline__ void tile_gemm(const TileOperands& op, int nstages, f32x4 (&acc)[4][JB_MAX],
                                          unsigned* pend, unsigned* queue, unsigned& next,
                                          AfterFirstLoads after_first_loads) {
  const int lane = threadIdx.x & 63, wave = uni(threadIdx.x >> 6);
  const int r16 = lane & 15, kg = lane >> 4;
  const unsigned lds_addr = uni(static_cast<unsigned>(
      reinterpret_cast<size_t>((FMOE_L3 unsigned char*)lds_raw)));
  constexpr int STG = stage_bytes_of(JT), NST = nst_of(JT);
  constexpr int JB = 2 * JT, NSL = 2 * JB, RING = ring_of(JT);
  constexpr int BAR = 2;                                     // slots between the last read of a stage and the hand-over
  constexpr int HO = NSL - RING + BAR;                       // the slot the hand-over stands in front of
  constexpr int AFTER = NSL - HO;                            // slots behind it
  constexpr int NL = NLD + JT;                               // loads per wave and stage
  constexpr int LPS = (NL + AFTER + JB - 1) / (AFTER + JB);  // loads per slot
  constexpr int APS = (4 + AFTER - 1) / AFTER;               // weight fragments of the next stage read per slot behind the hand-over
  static_assert(NSL % RING == 0 && RING > BAR && JB >= 4 && RING <= JB && HO >= JB, "slot schedule");
  static_assert(NST * STG <= TILE_LDS_BYTES, "stages exceed the tile's LDS");

  unsigned fo[2];  // per-lane token fragment offsets of the two 32-k sub-steps
#pragma unroll
  for (int u = 0; u < 2; ++u) fo[u] = lds_addr + r16 * ROWB + (((4 * u + kg) ^ ((r16 >> 1) & 7)) << 4);
  // weight fragments: from row-major stage rows as the token fragments, or, when the wave's
  // weight rows keep the packed order (eight runs [k-step 0..1][block 0..3] of [chunk][row]),
  // 16 bytes per lane of the run of k-step u, block i
  unsigned ao[2];
#pragma unroll
  for (int u = 0; u < 2; ++u) ao[u] = wave * (64 * ROWB) + (op.wpacked ? lds_addr + u * 4096 + lane * 16 : fo[u]);
  const int ablock = uni(op.wpacked ? 1024 : 16 * ROWB);  // bytes from one weight block to the next

  auto issue_one = [&](int s, int buf, int q) {  // q: 0..7 weights, 8..8+JT-1 tokens; buf: the stage buffer's byte offset
    const unsigned st = uni(static_cast<int>(lds_addr) + buf);
    if (q < NLD) {
      const size_t at = HALF ? min(static_cast<unsigned>(s) * op.wstride, op.wlast) : static_cast<size_t>(s) * op.wstride;
      load_to_lds(op.woff[q], op.wbase + at, st + (wave * 64 + q * 8) * ROWB);
    } else if (q < NL) {
      const int qq = q - NLD;
      const size_t at = HALF ? min(static_cast<unsigned>(s * ROWB), op.tlast) : static_cast<size_t>(s) * ROWB;
      load_to_lds(op.toff[qq], op.tbase + at, st + TN * ROWB + ((wave * JT + qq) * 8) * ROWB);
    }
  };
  auto read_a = [&](int buf, int u, int i) { return lds_read16(ao[u] + static_cast<unsigned>(buf + i * ablock)); };
  auto read_b = [&](int buf, int n) {  // the fragment of slot n
    return lds_read16(fo[n / JB] + static_cast<unsigned>(buf + TN * ROWB + (n % JB) * (16 * ROWB)));
  };

  auto bookkeeping = [&]() {
    if (threadIdx.x == 0) {
      if (pend != nullptr) (void)add_relaxed(pend, 1u);
      next = add_relaxed(queue, 1u);
    }
  };

  v4u_t af[2][4], ring[RING];
#pragma unroll
  for (int st = 0; st < NST; ++st) {
    if (st < 2 || nstages > st) {
#pragma unroll
      for (int q = 0; q < NL; ++q) issue_one(st, st * STG, q);
    }
  }
  // Loads to registers that the task still needs go out here, behind the loads to LDS: a
  // load to registers that is still on its way when a younger load to LDS is issued may not
  // deliver its data (seen with 16-byte loads; the register kept its old content). Every
  // later load to LDS follows a wait for all outstanding loads to registers.
  after_first_loads();
  // stage 0 has landed, then everybody's. (The wait is for everything this wave has asked
  // for, the later stages and the loads to registers included: the two kinds of load are not
  // counted in order with each other, so a count that leaves stage 1 in flight would not say
  // that stage 0 is in.)
  wait_vm<0>();
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
#pragma unroll
  for (int i = 0; i < 4; ++i) af[0][i] = read_a(0, 0, i);
#pragma unroll
  for (int n = 0; n < RING; ++n) ring[n] = read_b(0, n);

  // One stage. R: stages after it, NST meaning NST or more. cur, nxt, prv: byte offsets of the
  // buffers of this stage, the next one and the last one (with two buffers the latter are one).
  int cur = 0, nxt = STG, prv = (NST - 1) * STG;
  auto stage = [&](int s, auto first_tag, auto rem_tag) {
    constexpr bool FIRST = decltype(first_tag)::value;
    constexpr int R = decltype(rem_tag)::value;
    constexpr bool EARLY = !FIRST && R >= NST - 1;  // the tail of stage s+NST-1's loads is still to go out
    constexpr bool LATE = R >= NST;                 // stage s+NST exists
    constexpr bool NEXT = R >= 1;                   // stage s+1 exists
    // loads of the stages behind the next one, which may still be in flight at the hand-over
    constexpr int YOUNGER = NST == 3 && R >= 2 ? NL : 0;
#pragma unroll
    for (int n = 0; n < NSL; ++n) {
      const int u = n / JB, j = n % JB;
      if (n == HO && NEXT) {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        wait_vm<YOUNGER>();
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if (FIRST) bookkeeping();
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if (FIRST && u == 0) {
          if (j < JB_ACC) mma<true, false>(af[u][i], ring[n % RING], acc[i][j]); else mma<true, true>(af[u][i], ring[n % RING], acc[i][j]);
        } else {
          if (j < JB_ACC) mma<false, false>(af[u][i], ring[n % RING], acc[i][j]); else mma<false, true>(af[u][i], ring[n % RING], acc[i][j]);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
      if (n + RING < NSL) ring[n % RING] = read_b(cur, n + RING);
      if (n < 4) af[1][n] = read_a(cur, 1, n);
      if (NEXT && n >= HO) {
        if (n == HO) {
#pragma unroll
          for (int m = 0; m < BAR; ++m) ring[(NSL - RING + m) % RING] = read_b(nxt, m);
        }
        ring[n % RING] = read_b(nxt, n - (NSL - RING));
#pragma unroll
        for (int i = (n - HO) * APS; i < (n - HO + 1) * APS; ++i)
          if (i < 4) af[0][i] = read_a(nxt, 0, i);
      }
#pragma unroll
      for (int l = 0; l < LPS; ++l) {
        if (EARLY && n < HO) issue_one(s + NST - 1, prv, (AFTER + n) * LPS + l);
        if (LATE && n >= HO) issue_one(s + NST, cur, (n - HO) * LPS + l);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    prv = cur;
    cur = nxt;
    nxt = uni(nxt == (NST - 1) * STG ? 0 : nxt + STG);
  };
  using Yes = std::true_type;
  using No = std::false_type;
  using Full = std::integral_constant<int, NST>;
  if (nstages > NST) {
    stage(0, Yes{}, Full{});
  } else if (NST == 3 && nstages == 3) {
    stage(0, Yes{}, std::integral_constant<int, 2>{});
  } else {
    stage(0, Yes{}, std::integral_constant<int, 1>{});
  }
  int s = 1;
  for (; s + NST < nstages; ++s) stage(s, No{}, Full{});
  static_for<NST - 1>([&](auto i) {
    constexpr int r = NST - 1 - decltype(i)::value;  // stages after the next one to run
    if (s + r < nstages) {
      stage(s, No{}, std::integral_constant<int, r>{});
      ++s;
    }
  });
  if constexpr (HALF) {
#pragma unroll
    for (int i = 0; i < 4; ++i) af[1][i] = read_a(cur, 1, i);
#pragma unroll
    for (int j = 0; j < JB; ++j) {
      ring[j % RING] = read_b(cur, JB + j);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if (j < JB_ACC) mma<false, false>(af[1][i], ring[j % RING], acc[i][j]); else mma<false, true>(af[1][i], ring[j % RING], acc[i][j]);
      }
    }
  } else {
    stage(s, No{}, std::integral_constant<int, 0>{});
  }
  settle<JT>(acc);
}

// The same product when the weights come from the packed layout, on a deeper pipeline that
// keeps its depth in registers instead of LDS.
//
// A wave's 64 weight rows are its own: no other wave reads them. So they do not go through
// LDS at all: every fragment (16 rows x 32 k, 16 bytes per lane) is one global load straight
// into the registers the matrix instruction reads, one whole 1 KiB run of the packed layout
// per instruction. D register sets: the fragments of stage s+D are requested into the
// registers of stage s as soon as its sub-step is through. The token rows, which all four
// waves read, still meet in LDS, but they travel global -> registers -> LDS (ds_write_b128)
// instead of straight to LDS: a wave requests its JT loads of 8 rows of stage s+D+1 during
// stage s, into the registers whose previous content (stage s+1) it has just written to LDS.
// Three LDS buffers of 4 KiB per 32-row block, written one stage before they are read: the
// buffer a wave writes during stage s was last read in stage s-2, and the workgroup barrier
// of stage s-1 lies between, so a hand-over waits for nothing but this wave's writes of the
// next stage (long done) and the slowest wave.
//
// Loads straight to LDS are not used here on purpose: a load to registers that was still
// outstanding when a younger load-to-LDS was issued did not deliver its data (the register
// kept its old content; measured, deterministic), and the two kinds are not counted in order
// with each other either. With one kind of load only, completion is in order and how many
// younger loads may stay in flight at each wait is a constant of the schedule: every wave
// issues the same loads in the same order. direct_wait() counts them from the list of what
// a stage issues (which also covers the last stages, where loads of stages that do not exist
// are left out):
//   sub-step 0: weights (s+D-1, sub-step 1), then the token rows of stage s+D+1;
//   sub-step 1: weights (s+D, sub-step 0).
// The loads in front of the loop are issued in the same order, as if by stages -D ... -1.
constexpr int DIRECT_GROUPS = 3;
constexpr int DIRECT_JT_MAX = 8;     // taller tiles do not leave the registers for it
// Register sets for a product of nstages stages, 0: not this pipeline. Short tiles have few
// accumulators and are bound by the weights' way from memory: four sets, where the stages are
// enough to pay for filling and draining them (us, four / two sets: 30B shape T=512, 32 stages,
// 302 / 303; 235B shape T=600, 64 stages, 983 / 985; but H=I=512 T=900, 8 stages, 71.4 / 70.4;
// H=I=1024, 16 stages, 141.5 / 139.1; H=I=1536, 24 stages, 242.7 / 240.7). Two are enough for tall
// ones, whose stages last 2000 cycles, and serve every other number of stages; against the LDS
// pipeline (us, two sets / LDS): H=2048, I=256, 4 stages, T=448 162 / 166 and T=768 166 / 170; I=640,
// 10 stages, T=768 276 / 275; I=1408, 22 stages, T=768 499 / 499.
constexpr int direct_depth(int jt, int nstages) {
  if (jt <= 2 && nstages % 4 == 0 && nstages >= 32) return 4;
  return jt <= DIRECT_JT_MAX && nstages % 2 == 0 && nstages >= 4 ? 2 : 0;
}
// Loads that group g (in issue order) of a stage with r stages after it puts out, with d sets.
constexpr int direct_group(int jt, int d, int r, int g) {
  switch (g) {
    case 0: return r >= d - 1 ? 4 : 0;
    case 1: return r >= d + 1 ? jt : 0;
    default: return r >= d ? 4 : 0;
  }
}
// Loads issued after group g0 of the stage `back` stages before the present one (which has
// r stages after it) and before group g1 of the present stage: those may still be in flight
// when everything up to and including that group has to have landed.
constexpr int direct_in_flight(int jt, int d, int r, int back, int g0, int g1) {
  int n = 0;
  for (int b = back; b >= 0; --b) {
    const int lo = b == back ? g0 + 1 : 0;
    const int hi = b == 0 ? g1 : DIRECT_GROUPS;
    for (int g = lo; g < hi; ++g) n += direct_group(jt, d, r + b, g);
  }
  return n;
}
// wait in front of sub-step w of a stage with r stages after it: its weight fragments and,
// for sub-step 0, the token rows of the next stage, which that sub-step writes to LDS
constexpr int direct_wait(int jt, int d, int r, int w) {
  return w == 0 ? direct_in_flight(jt, d, r, d, 2, 0) : direct_in_flight(jt, d, r, d - 1, 0, 1);
}
static_assert(direct_wait(2, 4, 5, 0) < 64 && direct_wait(8, 2, 3, 0) < 64, "vmcnt holds 6 bits");

// 16 bytes per lane from base + off + OFF into the registers of `dst`; completion is tracked
// by hand (wait_vm), so the compiler must not believe it knows when the value is there: the
// operand is read-write, which keeps the value in one place from the load to its last use.
template <int OFF>
__device__ __forceinline__ void load_fragment(v4u_t& dst, unsigned off, const unsigned char* base) {
  asm volatile("global_load_dwordx4 %0, %1, %2 offset:%3" : "+v"(dst) : "v"(off), "s"(base), "n"(OFF) : "memory");
}
// 16 bytes per lane from registers to LDS (byte address `lds_off` + OFF)
template <int OFF>
__device__ __forceinline__ void store_fragment(unsigned lds_off, const v4u_t& src) {
  asm volatile("ds_write_b128 %0, %1 offset:%2" : : "v"(lds_off), "v"(src), "n"(OFF) : "memory");
}
template <int N>
__device__ __forceinline__ void wait_lds() {
  asm volatile("s_waitcnt lgkmcnt(%0)" : : "n"(N) : "memory");
}
template <int JT, int D>
__device__ __forceinline__ void tile_gemm_direct(const TileOperands& op, int nstages, f32x4 (&acc)[4][JB_MAX],
                                                 unsigned* pend, unsigned* queue, unsigned& next) {
  static_assert(JT <= DIRECT_JT_MAX, "tile too tall for the register-staged pipeline");
  constexpr int JB = 2 * JT, NSL = 2 * JB, RING = ring_of(JT);
  constexpr int HO = NSL - RING;                  // the slot the hand-over stands in front of
  constexpr int STG = 32 * JT * ROWB;             // token rows of one stage
  // LDS operations a wave issues between its last write of the next stage (slot JT - 1) and the hand-over
  constexpr int LDS_YOUNGER = HO - (JT - 1) < 15 ? HO - (JT - 1) : 15;
  static_assert(3 * STG <= TILE_LDS_BYTES, "token stages exceed the tile's LDS");
  static_assert(NSL % RING == 0 && HO >= JT && JB >= 4, "slot schedule");
  const int lane = threadIdx.x & 63, wave = uni(threadIdx.x >> 6);
  const int r16 = lane & 15, kg = lane >> 4;
  const unsigned lds_addr = uni(static_cast<unsigned>(
      reinterpret_cast<size_t>((FMOE_L3 unsigned char*)lds_raw)));

  unsigned fo[2];  // per-lane token fragment offsets of the two 32-k sub-steps
#pragma unroll
  for (int u = 0; u < 2; ++u) fo[u] = lds_addr + r16 * ROWB + (((4 * u + kg) ^ ((r16 >> 1) & 7)) << 4);
  // weight fragment (sub-step u, block i) of stage s in the wave's packed slice: the run at
  // 8192*s + 4096*u + 1024*i, 16 bytes per lane
  const unsigned aoff = static_cast<unsigned>(lane) * 16u;
  // where this lane's 16 bytes of the wave's token load q belong in a stage buffer: the
  // eight rows of load q are one run of 1 KiB, lane l at 16*l
  const unsigned wr_off = lds_addr + static_cast<unsigned>((wave * JT) * 1024 + lane * 16);

  v4u_t as[D][2][4];   // weight fragments: [stage % D][sub-step][block]
  v4u_t bs[D][JT];     // token rows on their way to LDS: [stage % D][load]
  v4u_t ring[RING];
#pragma unroll
  for (int p = 0; p < D; ++p) {
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int i = 0; i < 4; ++i) as[p][u][i] = v4u_t{0u, 0u, 0u, 0u};
#pragma unroll
    for (int q = 0; q < JT; ++q) bs[p][q] = v4u_t{0u, 0u, 0u, 0u};
  }
#pragma unroll
  for (int n = 0; n < RING; ++n) ring[n] = v4u_t{0u, 0u, 0u, 0u};

  auto issue_a = [&](int s, int u, auto i_tag, v4u_t& dst) {
    load_fragment<decltype(i_tag)::value * 1024>(dst, aoff, op.wbase + static_cast<size_t>(s) * 8192 + u * 4096);
  };
  auto issue_b = [&](int s, int q, v4u_t& dst) {  // q-th token load of this wave for stage s
    load_fragment<0>(dst, op.toff[q], op.tbase + static_cast<size_t>(s) * ROWB);
  };
  // the fragment of token block j; `base`: this lane's address in the stage buffer and sub-step
  auto read_b = [&](unsigned base, int j) { return lds_read16(base + static_cast<unsigned>(j * (16 * ROWB))); };

  // ---- in front of the loop. First what stage 0 needs at once: its token rows (through the
  // ring's registers, idle until then), its weight fragments, and the token rows of stage 1
  // (which stage 0 writes to LDS); then what the stages -D+1 ... -1 would have issued.
  static_assert(JT <= RING, "stage 0's token rows pass through the ring's registers");
#pragma unroll
  for (int q = 0; q < JT; ++q) issue_b(0, q, ring[q]);
  static_for<4>([&](auto i) { issue_a(0, 0, i, as[0][0][i]); });
#pragma unroll
  for (int q = 0; q < JT; ++q) issue_b(1, q, bs[1][q]);
  static_for<4>([&](auto i) { issue_a(0, 1, i, as[0][1][i]); });
  // All of this has landed, and so have the stores of the previous task's epilogue (loads and
  // stores are not taken to complete in order with each other, so only a wait for all of them
  // covers the stores): behind the workgroup barrier below thread 0 may signal that task's
  // completion. The later stages' loads go out behind the wait; in front of it, with a wait that
  // left them in flight, they gained nothing (us, full wait / partial: T=600 305 / 305, T=8192
  // 760 / 759, 235B shape T=1024 1018 / 1019).
  wait_vm<0>();
#pragma unroll
  for (int b = 1; b < D; ++b) {
    if (b > 1) static_for<4>([&](auto i) { issue_a(b - 1, 1, i, as[b - 1][1][i]); });
#pragma unroll
    for (int q = 0; q < JT; ++q) issue_b(b + 1, q, bs[(b + 1) % D][q]);
    static_for<4>([&](auto i) { issue_a(b, 0, i, as[b][0][i]); });
  }
  static_for<JT>([&](auto q) { store_fragment<q * 1024>(wr_off, ring[q]); });
  wait_lds<0>();
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  if (threadIdx.x == 0) {
    if (pend != nullptr) (void)add_relaxed(pend, 1u);
    next = add_relaxed(queue, 1u);
  }
#pragma unroll
  for (int n = 0; n < RING; ++n) ring[n] = read_b(fo[0], n);

  // One stage. P: its register set, stage % D. R: stages after it, D+1 meaning D+1 or more. cur, nxt: byte offsets of its and the next stage's buffer;
  // rd: where this lane reads sub-step 0 of the present stage.
  static_assert(RING <= JB, "fragments of the next stage read in advance are sub-step 0's");
  int cur = 0, nxt = STG;
  unsigned rd = fo[0];
  auto stage = [&](auto par_tag, auto rem_tag, auto first_tag, int s) {
    constexpr int P = decltype(par_tag)::value;
    constexpr int R = decltype(rem_tag)::value;
    constexpr bool FIRST = decltype(first_tag)::value;
    constexpr bool A0 = R >= D, A1 = R >= D - 1, NEXT = R >= 1, BN = R >= D + 1;
    constexpr int P1 = (P + D - 1) % D;  // the set of the last stage, and of stage s+D-1
    constexpr int PB = (P + 1) % D;      // the set of the next stage's token rows
    // (pinned, so that the reads and writes below are these registers plus constants)
    unsigned wr = wr_off + static_cast<unsigned>(nxt), rd1 = fo[1] + static_cast<unsigned>(cur),
             rdn = fo[0] + static_cast<unsigned>(nxt);
    asm volatile("" : "+v"(wr), "+v"(rd1), "+v"(rdn));
    static_for<NSL>([&](auto n_tag) {
      constexpr int n = decltype(n_tag)::value, u = n / JB, j = n % JB;
      if (n == 0) wait_vm<direct_wait(JT, D, R, 0)>();
      if (n == JB) wait_vm<direct_wait(JT, D, R, 1)>();
      if (n == HO && NEXT) {
        wait_lds<LDS_YOUNGER>();
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) mma<FIRST && u == 0, false>(as[P][u][i], ring[n % RING], acc[i][j]);
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (u == 0) {
        if constexpr (j < 2 && A1) {
          issue_a(s + D - 1, 1, std::integral_constant<int, 2 * j>{}, as[P1][1][2 * j]);
          issue_a(s + D - 1, 1, std::integral_constant<int, 2 * j + 1>{}, as[P1][1][2 * j + 1]);
        }
        if constexpr (j < JT && NEXT) store_fragment<j * 1024>(wr, bs[PB][j]);  // token rows of stage s+1
        if constexpr (j >= JT && BN) issue_b(s + D + 1, j - JT, bs[PB][j - JT]);
      } else if constexpr (j < 4 && A0) {
        // (one a slot; before, two in each of the first two slots: us, T=600 304.1 -> 303.5, behind other
        // launchers' memory 317.2 -> 316.3, T=900 307.8 -> 306.9, 235B shape T=1024 1017 -> 1016)
        issue_a(s + D, 0, std::integral_constant<int, j>{}, as[P][0][j]);
      }
      if constexpr (n + RING < JB) {
        ring[n % RING] = read_b(rd, n + RING);
      } else if constexpr (n + RING < NSL) {
        ring[n % RING] = read_b(rd1, n + RING - JB);
      } else if constexpr (NEXT) {
        ring[n % RING] = read_b(rdn, n + RING - NSL);
      }
      __builtin_amdgcn_sched_barrier(0);
    });
    rd = rdn;
    cur = nxt;
    nxt = uni(nxt == 2 * STG ? 0 : nxt + STG);
  };
  using Yes = std::true_type;
  using No = std::false_type;
  // nstages is a multiple of D and at least 2*D; the last 2*D - 1 stages stand behind the loop.
  // (One way through the code on purpose: where two ways meet or part the compiler may move
  // registers about, and a value that is still on its way from memory must never be copied.)
  stage(std::integral_constant<int, 0>{}, std::integral_constant<int, D + 1>{}, Yes{}, 0);
  int s = 1;
  for (; s + 2 * D - 1 < nstages; s += D)
    static_for<D>([&](auto i) {
      stage(std::integral_constant<int, (1 + decltype(i)::value) % D>{}, std::integral_constant<int, D + 1>{}, No{},
            s + decltype(i)::value);
    });
  static_for<2 * D - 1>([&](auto i) {
    constexpr int k = decltype(i)::value, r = 2 * D - 2 - k;
    stage(std::integral_constant<int, (1 + k) % D>{}, std::integral_constant<int, r < D + 1 ? r : D + 1>{}, No{}, s + k);
  });
  settle<JT>(acc);
  wait_vm<0>();
}

// Weights in the packed layout (the streaming variant's: per wave task and 32-k step four
// runs of 1 KiB, one per 16-row block, each [16-byte chunk 0..3][row 0..15]). This wave's 64
// stage rows are exactly one packed task: gate/up task (expert, 32 h columns) = gate blocks
// 0,1 and up blocks 2,3; down task (expert, 64 output columns) = blocks 0..3. A stage of 64 k
// is two 32-k steps, i.e. eight runs, and load q of the wave copies run (k-step q / 4, block
// q % 4) as it is: eight whole lines read by consecutive lanes. (Permuting the chunks into the
// row-major stage layout on the way in made every 16 lanes touch 8 lines: prefill 798 -> 867 us.)
// So with packed weights the wave's weight rows keep the packed order in LDS, and only the
// fragment reads differ: see tile_gemm.
static_assert(G1_NB == 2 && G2_NB == 4, "the tiled variant reads the packed layout as 32+32-row and 64-row tasks");
__device__ __forceinline__ unsigned packed_run_offset(int q) {
  return static_cast<unsigned>((q >> 2) * 4096 + (q & 3) * 1024 + (threadIdx.x & 63) * 16);
}

// ------------------------------------------------------------------ epilogues
// A lane ends with four consecutive columns of each 16-column block of its token row: 8 bytes of bf16, and
// the four lanes of a token 32 bytes a block. Two neighbouring blocks change places between lanes 16
// apart (V_PERMLANE16_SWAP: odd rows of 16 lanes of the first register against even rows of the second), and
// every lane has 8 consecutive columns of the 32, the four lanes of a token 64 contiguous bytes: a store
// instruction writes half lines of 16 rows, straight from the accumulators. No LDS, so no barrier and no trip
// through it stands between a task's last matrix instruction and its stores, and the waves of a
// workgroup leave the task one by one.
__device__ __forceinline__ void swap_rows16(unsigned& a, unsigned& b) {
  const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
  a = r[0];
  b = r[1];
}
// the 16 bytes of this lane out of its packed values of two blocks, and the column (of the 32) they start at
__device__ __forceinline__ uint4 pair_columns(uint2 a, uint2 b) {
  swap_rows16(a.x, b.x);
  swap_rows16(a.y, b.y);
  return make_uint4(a.x, a.y, b.x, b.y);
}
__device__ __forceinline__ unsigned pair_column(int kg) { return static_cast<unsigned>((kg & 1) * 16 + (kg >> 1) * 8); }
// Tiles of more than 256 rows go through LDS instead, where rows become whole again: they come in numbers, from experts
// that draw far more tokens than others, and there whole rows are ahead. us, 30B shape, half lines at all heights / as here /
// whole rows at all heights: four hot experts T=16384 1393 / 1382 / 1394, T=8192 725 / 723 / 768, T=2048 row-major 340 / 338 /
// 358; 235B shape T=4096 1382 / 1389 / 1409. It is not for the bytes: FETCH_SIZE of T=8192 is 1.168, 1.231 and 1.206 M KiB, of T=16384
// 1.816, 1.861 and 1.820 (WRITE_SIZE of half lines 1.7 % more): presumably an expert's tiles that leave in two ways drift
// apart and share fewer weights in the L2.
constexpr int EPI_LD = TN * 2 + 16;  // bytes per row of the down slab
static_assert(128 * EPI_LD <= TILE_LDS_BYTES && TM_MAX * (G1_COLS * 2 + 16) <= TILE_LDS_BYTES, "epilogue slab exceeds the stage buffers");
// eight rows' reads first, then their stores: a store's assembly orders memory operations around it, and one LDS round
// trip a store would add up to microseconds
template <int N, typename Read, typename Store>
__device__ __forceinline__ void for_rows(Read read, Store store) {
#pragma unroll
  for (int i0 = 0; i0 < N; i0 += 8) {
    uint4 v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (i0 + u < N) v[u] = read(i0 + u);
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (i0 + u < N) store(i0 + u, v[u]);
  }
}
// st16_through at a uniform base and a lane's offset
__device__ __forceinline__ void st16_through_at(unsigned char* base, unsigned off, const uint4& v) {
  const v4u_t d = {v.x, v.y, v.z, v.w};
  asm volatile("global_store_dwordx4 %0, %1, %2 sc1\n\ts_nop 1" : : "v"(off), "v"(d), "s"(base) : "memory");
}

// One GEMM tile task, gate/up or down, for a row tile of up to 32*JT rows.
//
// gate/up: h[row, n0 .. n0+128) (test/singleGPU/cpp/moe/reference/refExpertFFN1.h:51-65).
// h is [T*K, I] row-major, rows in permuted order. Wave w holds gate rows n0+32w.. and the
// matching up rows, so SiLU(gate)*up happens in registers.
//
// down: y[t*K+slot, n0 .. n0+256) = h[row] . W2[e]^T (refFullMoe.h:58-65,
// src/hip/kernel/tasks/ffn2Task.h:37-40), bf16. The rows' destinations are fetched when the task starts
// and parked in LDS behind the stages, so the epilogue waits for no memory. The slot's gate weight is applied
// by the combine task, which has instruction slots to spare; here every instruction of the
// epilogue is one the matrix cores wait for.
//
// Tiles of up to 256 rows store 64-byte pieces of their rows straight from the accumulators, each wave its own columns; taller
// ones go through LDS: gate/up as 256-byte row segments, down as 512-byte ones, 128 rows at a time. Only these end
// with a barrier. Without one a wave may still read the destinations and the next ticket (sdst, task_notes) while others
// are in the next task: both are written behind that task's k-loop, whose first barrier every wave reaches with its reads done.
//
// RAGGED: H is no multiple of 256 or I none of 128. The last task of a row tile may stand out over the
// last column: a wave whose columns do not exist repeats the last ones that do, and its results are not
// stored. These layers keep what the streaming variant computes for them, bit for bit: the division in
// SwiGLU is a division, and y holds float rows that carry their gate weight, stored from the accumulators
// (16 bytes a lane, 64 of a row). With bf16 rows as below they would be faster, but held in fewer bits than
// their small batches: relative error against float64 2.87e-3 instead of 2.35e-3 (us, streaming variant / float
// rows / bf16 rows, E=40, k=5, H=1344, I=736: T=260 127 / 101 / 98, T=2000 361 / 166 / 150, T=8000 1118 / 453 /
// 375; E=100, k=6, H=3904, I=1952: T=1200 1622 / 1028 / 997, T=4000 3746 / 1497 / 1384).
//
// HALF (down): I is an odd number of 32-k steps (see tile_gemm).
template <int JT, bool down, bool RAGGED = false, bool HALF = false>
__device__ __forceinline__ void tile_task(ParamsRef p, int expert, int row0, int rows, int nblk, unsigned* pend,
                                          unsigned* queue) {
  const int H = uni(p.H), I = uni(p.I), K = uni(p.K);
  const int wave = uni(threadIdx.x >> 6), lane = threadIdx.x & 63;
  // packed weights and enough stages: the deeper pipeline
  const int hp = RAGGED ? tiled_h_pitch(I) : I;
  const int depth = HALF ? 0 : uni((down ? p.ffn2_packed : p.ffn1_packed) != nullptr ? direct_depth(JT, (down ? I : H) / KS) : 0);
  const int* perm = uni(p.perm) + row0;
  const int n0 = uni(nblk) * (down ? TN : G1_COLS);
  const int wcol = down ? n0 / 64 + wave : n0 / 32 + wave;  // the wave's column block, and the last that exists
  const int wblk = RAGGED ? min(wcol, (down ? H / 64 : I / 32) - 1) : wcol;
  TileOperands op;
  int side_dst[2] = {-1, -1};
  float side_w[2] = {0.0f, 0.0f};
  int nstages;
  if (down) {
    nstages = (I + KS - 1) / KS;
    op.tlast = static_cast<unsigned>(I - KS) * 2u;
    const bool packed = uni(p.ffn2_packed != nullptr ? 1 : 0) != 0;
    op.wlast = packed ? static_cast<unsigned>(I / 32 - 2) * 4096u : op.tlast;
    if (packed) {
      const size_t task = static_cast<size_t>(expert) * (H / 64) + wblk;
      op.wbase = uni(reinterpret_cast<const unsigned char*>(p.ffn2_packed)) + task * (static_cast<size_t>(I / 32) * 4096);
      op.wstride = 8192u;
      op.wpacked = true;
    } else {
      op.wpacked = false;
      op.wbase = uni(reinterpret_cast<const unsigned char*>(p.ffn2)) + (static_cast<size_t>(expert) * H + 64 * wblk) * I * 2;
      op.wstride = static_cast<unsigned>(ROWB);
    }
    op.tbase = uni(reinterpret_cast<const unsigned char*>(p.h)) + static_cast<size_t>(row0) * hp * 2;
#pragma unroll
    for (int q = 0; q < NLD; ++q) {
      const int row = stage_row(NLD, q);
      op.woff[q] = packed ? packed_run_offset(q)
                          : static_cast<unsigned>(row & 63) * static_cast<unsigned>(I * 2) + stage_chunk_bytes(row);
    }
#pragma unroll
    for (int q = 0; q < JT; ++q) {
      const int row = stage_row(JT, q);
      op.toff[q] = static_cast<unsigned>(min(row, rows - 1)) * static_cast<unsigned>(hp * 2) + stage_chunk_bytes(row);
    }
  } else {
    nstages = H / KS;
    op.wlast = op.tlast = 0u;  // (not looked at)
    const bool packed = uni(p.ffn1_packed != nullptr ? 1 : 0) != 0;
    if (packed) {
      const size_t task = static_cast<size_t>(expert) * (I / 32) + wblk;
      op.wbase = uni(reinterpret_cast<const unsigned char*>(p.ffn1_packed)) + task * (static_cast<size_t>(H / 32) * 4096);
      op.wstride = 8192u;
      op.wpacked = true;
    } else {
      op.wpacked = false;
      op.wbase = uni(reinterpret_cast<const unsigned char*>(p.ffn1)) + static_cast<size_t>(expert) * 2 * I * H * 2;
      op.wstride = static_cast<unsigned>(ROWB);
    }
    op.tbase = uni(reinterpret_cast<const unsigned char*>(p.tokens));
#pragma unroll
    for (int q = 0; q < NLD; ++q) {
      const int row = stage_row(NLD, q);
      // weight stage rows 64w..64w+31: gate rows n0+32w.., 64w+32..64w+63: up rows I+n0+32w..
      const int wl = row & 63;
      const int wrow = (wl < 32 ? 0 : I - 32) + 32 * wblk + wl;
      op.woff[q] = packed ? packed_run_offset(q)
                          : static_cast<unsigned>(wrow) * static_cast<unsigned>(H * 2) + stage_chunk_bytes(row);
    }
#pragma unroll
    for (int q = 0; q < JT; ++q) {
      const int row = stage_row(JT, q);
      const int tok = ldc(&perm[min(row, rows - 1)]) / K;
      op.toff[q] = static_cast<unsigned>(tok) * static_cast<unsigned>(H * 2) + stage_chunk_bytes(row);
    }
  }
  f32x4 acc[4][JB_MAX];
  unsigned next = 0u;
  // down: where the tile's rows go (token, slot), fetched while the k-loop runs
  auto load_side = [&]() {
    if (down) {
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const int r = static_cast<int>(threadIdx.x) + k * T_THREADS;
        side_dst[k] = r < rows ? ldc(&perm[r]) : -1;
        if (RAGGED && r < rows) side_w[k] = ldc(&uni(p.row_w)[row0 + r]);
      }
    }
  };
  if (depth != 0) {
    load_side();
    if constexpr (JT <= 2) {
      if (depth == 4) tile_gemm_direct<JT, 4>(op, nstages, acc, pend, queue, next);
      else tile_gemm_direct<JT, 2>(op, nstages, acc, pend, queue, next);
    } else if constexpr (JT <= DIRECT_JT_MAX) {
      tile_gemm_direct<JT, 2>(op, nstages, acc, pend, queue, next);
    }
  } else {
    tile_gemm<JT, HALF>(op, nstages, acc, pend, queue, next, load_side);
  }
  // What the workgroup shares from here on goes to LDS in front of the one barrier behind the k-loop: the
  // next ticket, and (down) where the rows go. It also says that nobody reads the stages any more.
  int* sdst = reinterpret_cast<int*>(lds_raw + SIDE_OFF);
  if (threadIdx.x == 0) task_notes()[0] = next;
  if (down) {
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const int r = static_cast<int>(threadIdx.x) + k * T_THREADS;
      if (r < TM_MAX) sdst[r] = side_dst[k];
      if (RAGGED && r < TM_MAX) reinterpret_cast<float*>(sdst + TM_MAX)[r] = side_w[k];
    }
  }
  __syncthreads();
  if (RAGGED && wcol != wblk) return;  // these columns do not exist

  const int r16 = lane & 15, kg = lane >> 4;
  // token blocks below this one have all of their rows (a tile has more than 32 * (JT - 1); JT = 2: or fewer)
  constexpr int FULL = JT == 2 ? 0 : 2 * (JT - 1);
  const unsigned colb = pair_column(kg) * 2u;
  if constexpr (!RAGGED && JT > 8) {
    unsigned char* slab = lds_raw;
    if (!down) {
      constexpr int LD = G1_COLS * 2 + 16;  // slab row pitch in bytes
#pragma unroll
      for (int j = 0; j < 2 * JT; ++j)
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          float hv[4];
#pragma unroll
          for (int v = 0; v < 4; ++v) hv[v] = silu_mul_fast(acc[i][j][v], acc[2 + i][j][v]);
          *reinterpret_cast<uint2*>(slab + (j * 16 + r16) * LD + (wave * 32 + i * 16 + kg * 4) * 2) =
              make_uint2(pack_bf16(hv[0], hv[1]), pack_bf16(hv[2], hv[3]));
        }
      __syncthreads();
      // 16 lanes store one row's 256 bytes
      unsigned char* h = uni(reinterpret_cast<unsigned char*>(p.h)) + (static_cast<size_t>(row0) * hp + 32 * (wcol - wave)) * 2;
      for_rows<8 * JT / WAVES>([&](int it) { return *reinterpret_cast<const uint4*>(slab + ((it * WAVES + wave) * 4 + kg) * LD + r16 * 16); },
                               [&](int it, const uint4& v) {
                                 const int row = (it * WAVES + wave) * 4 + kg;
                                 if (row < rows) st16_through(h + static_cast<size_t>(row) * hp * 2 + r16 * 16, v);
                               });
      __syncthreads();  // the slab is stage memory again
    } else {
      unsigned char* y = uni(reinterpret_cast<unsigned char*>(p.y)) + 128 * (wcol - wave);
#pragma unroll
      for (int part = 0; part < (JT + 3) / 4; ++part) {
#pragma unroll
        for (int jj = 0; jj < 8; ++jj) {
          const int j = part * 8 + jj;
          if (j < 2 * JT) {
#pragma unroll
            for (int i = 0; i < 4; ++i)
              *reinterpret_cast<uint2*>(slab + (jj * 16 + r16) * EPI_LD + (wave * 64 + i * 16 + kg * 4) * 2) =
                  make_uint2(pack_bf16(acc[i][j][0], acc[i][j][1]), pack_bf16(acc[i][j][2], acc[i][j][3]));
          }
        }
        __syncthreads();
        // 32 lanes store one row's 512 bytes at the row's (token, slot)
        for_rows<128 / (2 * WAVES)>(
            [&](int it) { return *reinterpret_cast<const uint4*>(slab + ((it * WAVES + wave) * 2 + (lane >> 5)) * EPI_LD + (lane & 31) * 16); },
            [&](int it, const uint4& v) {
              const int row = part * 128 + (it * WAVES + wave) * 2 + (lane >> 5);
              const int dst = row < 32 * JT ? sdst[row] : -1;
              if (dst >= 0) st16_through(y + static_cast<size_t>(dst) * H * 2 + (lane & 31) * 16, v);
            });
        __syncthreads();
      }
    }
  } else if (!down) {
    unsigned char* h = uni(reinterpret_cast<unsigned char*>(p.h)) + (static_cast<size_t>(row0) * hp + 32 * wcol) * 2;
    const unsigned off = static_cast<unsigned>(r16) * static_cast<unsigned>(hp * 2) + colb;
#pragma unroll
    for (int j = 0; j < 2 * JT; ++j) {
      uint2 pk[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) {  // gate blocks 0, 1 with their up blocks 2, 3
        float hv[4];
#pragma unroll
        for (int v = 0; v < 4; ++v)
          hv[v] = RAGGED ? silu_mul(acc[i][j][v], acc[2 + i][j][v]) : silu_mul_fast(acc[i][j][v], acc[2 + i][j][v]);
        pk[i] = make_uint2(pack_bf16(hv[0], hv[1]), pack_bf16(hv[2], hv[3]));
      }
      const uint4 v = pair_columns(pk[0], pk[1]);
      if (j < FULL || 16 * j + r16 < rows) st16_through_at(h + static_cast<size_t>(j) * (32 * hp), off, v);
    }
  } else if constexpr (RAGGED) {
    float* yf = uni(p.y) + 64 * wcol + 4 * kg;
#pragma unroll
    for (int j = 0; j < 2 * JT; ++j) {
      const int dst = sdst[16 * j + r16];
      const float w = reinterpret_cast<const float*>(sdst + TM_MAX)[16 * j + r16];
      if (dst >= 0) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          st16_through(yf + static_cast<size_t>(dst) * H + 16 * i,
                       make_uint4(__float_as_uint(acc[i][j][0] * w), __float_as_uint(acc[i][j][1] * w),
                                  __float_as_uint(acc[i][j][2] * w), __float_as_uint(acc[i][j][3] * w)));
      }
    }
  } else {
    unsigned char* y = uni(reinterpret_cast<unsigned char*>(p.y)) + 128 * wcol + colb;
    int dst[2 * JT];
#pragma unroll
    for (int j = 0; j < 2 * JT; ++j) dst[j] = sdst[16 * j + r16];
#pragma unroll
    for (int j = 0; j < 2 * JT; ++j) {
      uint2 pk[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) pk[i] = make_uint2(pack_bf16(acc[i][j][0], acc[i][j][1]), pack_bf16(acc[i][j][2], acc[i][j][3]));
      const uint4 lo = pair_columns(pk[0], pk[1]), hi = pair_columns(pk[2], pk[3]);
      if (j < FULL || dst[j] >= 0) {
        unsigned char* row = y + static_cast<size_t>(dst[j]) * H * 2;
        st16_through(row, lo);
        st16_through(row + 64, hi);
      }
    }
  }
}

// one straight-line instantiation per number of live token blocks
__device__ __noinline__ void tiled_gemm_task(ParamsRef pv, const TileDesc& tile_in, int nblk, int down_in,
                                             unsigned* pend_in, unsigned* queue_in) {
  ParamsRef p = uniform_params(pv);
  unsigned* pend = uni(pend_in);
  unsigned* queue = uni(queue_in);
  const int expert = uni(tile_in.expert), row0 = uni(tile_in.row0), rows = uni(tile_in.rows);
  const bool down = uni(down_in) != 0;
  const int jt = (rows + 31) >> 5;
  if (jt > 9) {
    if (down) tile_task<10, true>(p, expert, row0, rows, nblk, pend, queue); else tile_task<10, false>(p, expert, row0, rows, nblk, pend, queue);
  } else if (jt > 8) {
    if (down) tile_task<9, true>(p, expert, row0, rows, nblk, pend, queue); else tile_task<9, false>(p, expert, row0, rows, nblk, pend, queue);
  } else if (jt > 7) {
    if (down) tile_task<8, true>(p, expert, row0, rows, nblk, pend, queue); else tile_task<8, false>(p, expert, row0, rows, nblk, pend, queue);
  } else if (jt > 6) {
    if (down) tile_task<7, true>(p, expert, row0, rows, nblk, pend, queue); else tile_task<7, false>(p, expert, row0, rows, nblk, pend, queue);
  } else if (jt > 5) {
    if (down) tile_task<6, true>(p, expert, row0, rows, nblk, pend, queue); else tile_task<6, false>(p, expert, row0, rows, nblk, pend, queue);
  } else if (jt > 4) {
    if (down) tile_task<5, true>(p, expert, row0, rows, nblk, pend, queue); else tile_task<5, false>(p, expert, row0, rows, nblk, pend, queue);
  } else if (jt > 3) {
    if (down) tile_task<4, true>(p, expert, row0, rows, nblk, pend, queue); else tile_task<4, false>(p, expert, row0, rows, nblk, pend, queue);
  } else if (jt > 2) {
    if (down) tile_task<3, true>(p, expert, row0, rows, nblk, pend, queue); else tile_task<3, false>(p, expert, row0, rows, nblk, pend, queue);
  } else {
    if (down) tile_task<2, true>(p, expert, row0, rows, nblk, pend, queue); else tile_task<2, false>(p, expert, row0, rows, nblk, pend, queue);
  }
}

// the tasks of ragged layers, and their down tasks where I is an odd number of 32-k steps
template <bool down, bool HALF>
__device__ __forceinline__ void ragged_tile(ParamsRef pv, const TileDesc& tile_in, int nblk, unsigned* pend_in,
                                            unsigned* queue_in) {
  ParamsRef p = uniform_params(pv);
  unsigned* pend = uni(pend_in);
  unsigned* queue = uni(queue_in);
  const int expert = uni(tile_in.expert), row0 = uni(tile_in.row0), rows = uni(tile_in.rows);
  switch ((rows + 31) >> 5) {
    case 1:
    case 2: tile_task<2, down, true, HALF>(p, expert, row0, rows, nblk, pend, queue); break;
    case 3: tile_task<3, down, true, HALF>(p, expert, row0, rows, nblk, pend, queue); break;
    case 4: tile_task<4, down, true, HALF>(p, expert, row0, rows, nblk, pend, queue); break;
    case 5: tile_task<5, down, true, HALF>(p, expert, row0, rows, nblk, pend, queue); break;
    case 6: tile_task<6, down, true, HALF>(p, expert, row0, rows, nblk, pend, queue); break;
    case 7: tile_task<7, down, true, HALF>(p, expert, row0, rows, nblk, pend, queue); break;
    case 8: tile_task<8, down, true, HALF>(p, expert, row0, rows, nblk, pend, queue); break;
    case 9: tile_task<9, down, true, HALF>(p, expert, row0, rows, nblk, pend, queue); break;
    default: tile_task<10, down, true, HALF>(p, expert, row0, rows, nblk, pend, queue); break;
  }
}
__device__ __noinline__ void tiled_ragged_gate_up_task(ParamsRef p, const TileDesc& tile, int nblk, unsigned* pend,
                                                       unsigned* queue) {
  ragged_tile<false, false>(p, tile, nblk, pend, queue);
}
__device__ __noinline__ void tiled_ragged_down_task(ParamsRef p, const TileDesc& tile, int nblk, unsigned* pend,
                                                    unsigned* queue) {
  ragged_tile<true, false>(p, tile, nblk, pend, queue);
}
__device__ __noinline__ void tiled_odd_down_task(ParamsRef p, const TileDesc& tile, int nblk, unsigned* pend,
                                                 unsigned* queue) {
  ragged_tile<true, true>(p, tile, nblk, pend, queue);
}

constexpr int TILED_LDS_BYTES = NOTE_OFF + NOTE_BYTES;
static_assert(TILED_LDS_BYTES >= DOT32_LDS_BYTES && TILED_LDS_BYTES >= SHORT_LDS_BYTES && TILED_LDS_BYTES >= ROUTER_LDS_BYTES && TILED_LDS_BYTES + 256 <= 160 * 1024, "LDS of a workgroup");

// combine: out[t] = sum over slots, in slot order, of w[t,slot] * y[t*K+slot]
// (refFullMoe.h:35,62-65): y holds each slot's down-projection row rounded to bf16; weight
// and sum are float, one fused multiply-add per slot, then one rounding to bf16.
//
// One item = 8 columns of one token; a unit = the rows of up to 8 slots of one item (16
// bytes each). A thread walks through its units with the loads of the next CMB_D - 1 units
// in flight while it sums the present one: with one wave per SIMD nothing else covers the
// summing, and a thread that loads everything and then sums everything leaves the memory
// pipeline idle half of the time (4.4 TB/s; measured with four items loaded at once).
constexpr int CMB_D = 3;  // units of a thread: one being summed, the others in flight
constexpr int CMB_RUN = 8;  // units of one straight-line run (30B shape: one task)
// Every thread of the task walks through the same number of units with unconditional loads
// (a thread without an item of its own repeats the task's last one and stores nothing; slots
// past K repeat slot K-1 and are not summed), so control flow is uniform and every wave has
// the same loads in flight. The loads are issued from assembly and waited for by count
// (left to itself the compiler waited for all but one unit's loads before every sum).
// Stores are not counted: they may complete out of order with the loads, and leaving them
// out of the count only makes a wait longer, never shorter.
__device__ __forceinline__ void load_once(v4u_t& dst, unsigned off, const unsigned char* base) {
  asm volatile("global_load_dwordx4 %0, %1, %2 nt" : "=v"(dst) : "v"(off), "s"(base) : "memory");
}
template <bool RESIDUAL>
__device__ __forceinline__ void combine_units(const unsigned short* y, const unsigned short* residual,
                                              unsigned short* out, const float* wts, const unsigned char* flag,
                                              int t0, int nitems, int cpr, int H, int K) {
  constexpr int LPU = RESIDUAL ? 9 : 8;  // loads per unit
  const int tid = threadIdx.x;
  const int nchunks = uni((K + 7) >> 3);  // units per item
  const int nunits = uni(((nitems + T_THREADS - 1) / T_THREADS) * nchunks);
  v4u_t v[CMB_D][8];
  v4u_t rv[CMB_D];
  // the task's rows of y and of the residual (uniform); a lane's offsets inside them fit 32 bits
  const unsigned char* ybase = uni(reinterpret_cast<const unsigned char*>(y + static_cast<size_t>(t0) * K * H));
  const unsigned char* rbase = uni(reinterpret_cast<const unsigned char*>(residual + static_cast<size_t>(t0) * H));
  auto where = [&](int unit, int& tl, int& col, int& k0, bool& live) {
    const int item = unit / nchunks;  // uniform
    k0 = (unit - item * nchunks) << 3;
    const int it = tid + item * T_THREADS;
    live = it < nitems;
    const int itc = min(it, nitems - 1);
    tl = itc / cpr;
    col = (itc - tl * cpr) << 3;
  };
  auto issue = [&](int unit, v4u_t (&dst)[8], v4u_t& rdst) {
    int tl, col, k0;
    bool live;
    where(unit, tl, col, k0, live);
    const unsigned yoff = static_cast<unsigned>((tl * K * H + col) * 2);
#pragma unroll
    for (int k = 0; k < 8; ++k) load_once(dst[k], yoff, ybase + static_cast<size_t>(min(k0 + k, K - 1)) * H * 2);
    if (RESIDUAL) load_once(rdst, static_cast<unsigned>((tl * H + col) * 2), rbase);
  };
  float s[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) s[i] = 0.0f;
  auto consume = [&](int unit, const v4u_t (&src)[8], const v4u_t& rsrc) {
    int tl, col, k0;
    bool live;
    where(unit, tl, col, k0, live);
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const int kk = min(k0 + k, K - 1);
      // a slot without an expert holds rows nobody wrote: they are not looked at
      const bool use = k0 + k < K && flag[tl * K + kk] != 0;
      const float w = wts[tl * K + kk];
      float f[8];
      unpack<BF16>(make_uint4(src[k].x, src[k].y, src[k].z, src[k].w), f);
#pragma unroll
      for (int i = 0; i < 8; ++i) s[i] = use ? __fmaf_rn(f[i], w, s[i]) : s[i];
    }
    if (k0 + 8 >= K) {  // the item's last unit (uniform)
      if (RESIDUAL) {  // output = input row + layer, the row added last
        float f[8];
        unpack<BF16>(make_uint4(rsrc.x, rsrc.y, rsrc.z, rsrc.w), f);
#pragma unroll
        for (int i = 0; i < 8; ++i) s[i] += f[i];
      }
      if (live)
        st16(out + static_cast<size_t>(t0 + tl) * H + col,
             u32x4{pack_bf16(s[0], s[1]), pack_bf16(s[2], s[3]), pack_bf16(s[4], s[5]), pack_bf16(s[6], s[7])});
#pragma unroll
      for (int i = 0; i < 8; ++i) s[i] = 0.0f;
    }
  };
  // Units go in straight-line runs of CMB_RUN, 4, 2 and 1 (no loop-carried registers: a value that is
  // still on its way from memory must never be copied).
  auto run = [&](auto n_tag, int u0) {
    constexpr int N = decltype(n_tag)::value;
#pragma unroll
    for (int d = 0; d + 1 < CMB_D && d < N; ++d) issue(u0 + d, v[d], rv[d]);
#pragma unroll
    for (int d = 0; d < N; ++d) {
      if (d + CMB_D - 1 < N) {
        issue(u0 + d + CMB_D - 1, v[(d + CMB_D - 1) % CMB_D], rv[(d + CMB_D - 1) % CMB_D]);
        wait_vm<(CMB_D - 1) * LPU>();
      } else if (d + 2 < N && CMB_D > 3) {
        wait_vm<2 * LPU>();
      } else if (d + 1 < N) {
        wait_vm<LPU>();
      } else {
        wait_vm<0>();
      }
      __builtin_amdgcn_sched_barrier(0);
      consume(u0 + d, v[d % CMB_D], rv[d % CMB_D]);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  int u0 = 0;
  for (; u0 + CMB_RUN <= nunits; u0 += CMB_RUN) run(std::integral_constant<int, CMB_RUN>{}, u0);
  if (u0 + 4 <= nunits) {
    run(std::integral_constant<int, 4>{}, u0);
    u0 += 4;
  }
  if (u0 + 2 <= nunits) {
    run(std::integral_constant<int, 2>{}, u0);
    u0 += 2;
  }
  if (u0 < nunits) run(std::integral_constant<int, 1>{}, u0);
}

__device__ __noinline__ void tiled_combine_task(ParamsRef pv, int blk, int tok_in) {
  ParamsRef p = uniform_params(pv);
  const int H = uni(p.H), K = uni(p.K), T = uni(p.T), E = uni(p.E), W = uni(p.W);
  unsigned short* out = uni(reinterpret_cast<unsigned short*>(p.out));
  const unsigned short* y = uni(reinterpret_cast<const unsigned short*>(p.y));
  const unsigned short* residual = uni(reinterpret_cast<const unsigned short*>(p.residual));
  const int* topk_idx = uni(p.topk_idx);
  const float* topk_w = uni(p.topk_w);
  unsigned long long* masks = uni(p.masks);
  const int tid = threadIdx.x;
  const int tok = uni(tok_in);
  const int t0 = uni(blk) * tok;
  const int ntok = uni(min(tok, T - t0));
  // which (token, slot) pairs of this task hold an expert, and their gate weights: one load each
  float* wts = reinterpret_cast<float*>(lds_raw);                      // [CMB_TOK * MAX_TOPK]
  unsigned char* flag = lds_raw + CMB_TOK * MAX_TOPK * sizeof(float);  // [CMB_TOK * MAX_TOPK]
  if (tid < ntok * K) {
    flag[tid] = ldc(&topk_idx[static_cast<size_t>(t0) * K + tid]) >= 0 ? 1 : 0;
    wts[tid] = ldc(&topk_w[static_cast<size_t>(t0) * K + tid]);
  }
  __syncthreads();
  const int cpr = H >> 3;  // items per token
  if (residual != nullptr) {
    combine_units<true>(y, residual, out, wts, flag, t0, ntok * cpr, cpr, H, K);
  } else {
    combine_units<false>(y, residual, out, wts, flag, t0, ntok * cpr, cpr, H, K);
  }
  for (int tl = 0; tl < ntok; ++tl) {
    const int t = t0 + tl;
    if ((t & 63) == 0) {
      for (int e = tid; e < E; e += T_THREADS) stc(&masks[static_cast<size_t>(e) * W + (t >> 6)], 0ull);
    }
  }
  __syncthreads();  // flag[] and wts[] are reused by the next task
}
// ---------------------------------------------------------------- worker loop
// Ticket layout. The prologue (router, scan, scatter) uses one global counter.
// The GEMM tasks are split into eight queues, one per XCD: queue x owns a
// contiguous eighth of the row-tile table (which is sorted by expert), first all
// its gate/up tasks (tile-major), then all its down tasks. A workgroup serves
// the queue of the XCD it runs on, so tasks that share a token tile or a weight
// tile run on CUs behind the same L2 at about the same time, and a tile's h
// rows are consumed where they were produced. A workgroup whose queue is empty
// steals from the next queue. Dependencies stay inside one queue and point to
// smaller tickets, so whoever holds them is already running. Combine tasks
// come from a last global counter once every queue is empty.
// The launch parameters are read in place and the task calls keep the local
// calling convention, as in the streaming variant (see its worker loop).
// RAGGED: see tile_task. ODD: I is an odd number of 32-k steps, which only ragged layers have (kernels of
// their own: as a branch of this one the odd steps cost every task of the others half a microsecond). TRACED:
// with task records (kernels of their own: asking at run time costs the others, 30B shape, us, with / without
// the question: T=600 283.5 / 278.8, T=2048 row-major 367.3 / 359.5, T=8192 766.9 / 762.5).
template <bool RAGGED, bool ODD, bool TRACED>
__global__ __launch_bounds__(T_THREADS) __attribute__((disable_tail_calls)) void moe_tiled_kernel(
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
  const unsigned T = static_cast<unsigned>(p.T);
  const unsigned n_sc = (T + RT_TOK - 1u) / RT_TOK;  // scatter tasks
  // router tasks: 16 tokens each while one round of them covers the batch, 32 beyond that
  // (a task of 32 takes longer than one of 16, but less than two of them)
  const bool rt2 = (T + RT16_TOK - 1u) / RT16_TOK > gridDim.x;
  const unsigned rt_tok = rt2 ? 2u * RT16_TOK : 1u * RT16_TOK;
  const unsigned n_rt = (T + rt_tok - 1u) / rt_tok;
  const unsigned n_es = (static_cast<unsigned>(p.E) + SCAN_EXPERTS - 1u) / SCAN_EXPERTS;
  const unsigned t_escan0 = n_rt;
  const unsigned t_scan = n_rt + n_es;
  const unsigned t_scatter0 = t_scan + 1u;
  unsigned t_dyn0 = t_scatter0 + n_sc;
  const unsigned nt1 = static_cast<unsigned>((p.I + G1_COLS - 1) / G1_COLS);
  const unsigned nt2 = static_cast<unsigned>((p.H + TN - 1) / TN);
  // as few tokens to a combine task as one round of tasks allows (8 tokens always, us, 30B shape: T=600
  // 306.5 -> 302.3, where 75 workgroups had a task and the others none; 235B shape T=700 1027 -> 1021; two
  // rounds of half as many tokens: T=600 303.9)
  int cmb_tok = 1;
  while (cmb_tok < CMB_TOK && T > gridDim.x * cmb_tok) cmb_tok *= 2;
  const unsigned ncmb = (T + cmb_tok - 1u) / cmb_tok;
  const unsigned n_groups = gridDim.x;
  const int home = xcc_id();
  bool first = true, ok = true;

  constexpr bool traced = TRACED;
  auto trace = [&](unsigned id, unsigned kind, unsigned aux, long long t_fetch, long long t_ready) {
    trace_task(p, traced && threadIdx.x == 0, id, kind, aux, t_fetch, t_ready);
  };

  // ---- prologue, few tokens: handed out statically (every workgroup of the launch is resident)
  if (p.dot16) {
    const int G = static_cast<int>(n_groups), b = static_cast<int>(blockIdx.x), wave = uni(static_cast<int>(threadIdx.x >> 6));
    const int Ti = static_cast<int>(T), n_eg = (p.E + 31) >> 5, n_dot = ((Ti + 15) >> 4) * n_eg;
    // (records: router tasks, one for the selections of each wave, scatter tasks)
    unsigned t_perm0 = n_rt;
    if (p.dot16 == 1) {
      for (int i = b; i < n_dot; i += G) {
        const long long t0 = trace_clock(traced);
        router_dot32_task(p, i / n_eg, i % n_eg);
        trace(i, 0, i, t0, t0);
      }
      const int sel_groups = min(n_dot, G);
      const int i0 = b + sel_groups * wave, tok = select_tokens(p.E, p.K, Ti);
      // (the launcher takes this start while there are as many waves as selections, at least)
      if (b < sel_groups && i0 * tok < Ti) {
        const long long t0 = trace_clock(traced);
        const int n = router_select_tokens_task(p, i0, static_cast<unsigned>((p.E + 15) >> 4), lds_raw + wave * SELECT_ROWS_BYTES);
        unsigned old = 0;
        if (lane_id() == 0) old = add_relaxed(&ctl->router_done.v, static_cast<unsigned>(n));
        // (n = 0: a wait that failed has raised an error bit, which every later wait sees)
        if (uni(static_cast<int>(old)) + n == Ti) broadcast_flag(p, FLAG_ROUTED);
        trace_task(p, traced && lane_id() == 0, n_dot + i0, 6, i0 * tok, t0, t0);
      }
      t_perm0 = n_dot + WAVES * sel_groups;
    } else {
      for (int i = b; i < static_cast<int>(n_rt); i += G) {
        const long long t0 = trace_clock(traced);
        if (rt2) {
          tiled_router_task<2>(p, i);
        } else {
          tiled_router_task<1>(p, i);
        }
        if (wg_arrive<false>(&ctl->router_done.v, &sh) == n_rt - 1u) wg_broadcast_flag(p, FLAG_ROUTED);
        trace(i, 0, i, t0, t0);
      }
    }
    const int n_perm = (Ti * p.K + T_THREADS - 1) / T_THREADS;
    t_dyn0 = t_perm0 + n_perm;
    const long long t_fetch = trace_clock(traced);
    if (b < n_perm) ok = wg_wait_flag(p, FLAG_ROUTED, &sh);
    for (int i = b; ok && i < n_perm; i += G) {
      const long long t_ready = trace_clock(traced);
      short_scatter_task<RAGGED>(p, i);
      if (wg_arrive<false>(&ctl->perm_done.v, &sh) == static_cast<unsigned>(n_perm) - 1u) wg_broadcast_flag(p, FLAG_PERM);
      trace(t_perm0 + i, 2, i, i == b ? t_fetch : t_ready, t_ready);
    }
  }
  // ---- prologue otherwise: router, scan, scatter from the global counter
  while (ok && !p.dot16) {
    const long long t_fetch = trace_clock(traced);
    if (threadIdx.x == 0) sh.ticket = first ? blockIdx.x : n_groups + add_relaxed(&ctl->ticket.v, 1u);
    first = false;
    __syncthreads();
    const unsigned tk = sh.ticket;
    __syncthreads();
    if (tk >= t_dyn0) break;
    long long t_ready = 0;
    if (tk < n_rt) {
      if (traced) t_ready = wall_clock64();
      if (rt2) {
        tiled_router_task<2>(p, static_cast<int>(tk));
      } else {
        tiled_router_task<1>(p, static_cast<int>(tk));
      }
      wg_arrive<false>(&ctl->router_done.v, &sh);
      trace(tk, 0, tk, t_fetch, t_ready);
    } else if (tk < t_scan) {
      ok = wg_wait_ge(p, &ctl->router_done.v, n_rt, &sh);
      if (ok) {
        if (traced) t_ready = wall_clock64();
        tiled_expert_scan_task(p, static_cast<int>(tk - t_escan0));
        wg_arrive<false>(&ctl->scan_done.v, &sh);
        trace(tk, 6, tk - t_escan0, t_fetch, t_ready);
      }
    } else if (tk == t_scan) {
      ok = wg_wait_ge(p, &ctl->scan_done.v, n_es, &sh);
      if (ok) {
        if (traced) t_ready = wall_clock64();
        tiled_scan_task<TM_MAX, 32>(p);
        trace(tk, 1, 0, t_fetch, t_ready);
      }
    } else {
      ok = wg_wait_flag(p, FLAG_SCAN, &sh);
      if (ok) {
        if (traced) t_ready = wall_clock64();
        tiled_scatter_task(p, static_cast<int>(tk - t_scatter0));
        if (wg_arrive<false>(&ctl->perm_done.v, &sh) == n_sc - 1u) wg_broadcast_flag(p, FLAG_PERM);
        trace(tk, 2, tk - t_scatter0, t_fetch, t_ready);
      }
    }
  }

  // ---- GEMM tasks from the per-XCD queues
  unsigned nm = 0, n2_total = 0;
  if (ok && !p.dot16) ok = wg_wait_flag(p, FLAG_SCAN, &sh);
  if (ok) ok = wg_wait_flag(p, FLAG_PERM, &sh);
  if (ok) {
    nm = ldc(&ctl->n_mtiles.v);
    n2_total = nm * nt2;
  }
  for (int hop = 0; ok && hop < 8; ++hop) {
    const unsigned q = static_cast<unsigned>((home + hop) & 7);
    const unsigned lo = nm * q / 8u, hi = nm * (q + 1u) / 8u;
    const unsigned tiles = hi - lo;
    const unsigned q1 = tiles * nt1, q2 = tiles * nt2;
    // The first ticket of a queue is drawn on its own; every task then draws its successor
    // while it runs, and its own completion is signalled under the next task (`pend`), so a
    // workgroup goes from one task's last store to the next task's first load without a trip
    // to memory. A completion that is still pending is signalled at once (after waiting for
    // the stores) when the next task has to wait for a dependency or there is no next task:
    // nobody may wait on a counter that a waiting workgroup holds back.
    if (threadIdx.x == 0) sh.ticket = add_relaxed(&ctl->xq[q].v, 1u);
    __syncthreads();
    unsigned j = sh.ticket;
    __syncthreads();
    unsigned* pend = nullptr;
    auto flush = [&]() {
      if (pend != nullptr) {
        fence_release();
        __syncthreads();
        if (threadIdx.x == 0) (void)add_relaxed(pend, 1u);
        pend = nullptr;
      }
    };
    while (ok) {
      const long long t_fetch = trace_clock(traced);
      if (j >= q1 + q2) break;
      long long t_ready = 0;
      if (j < q1) {
        const unsigned m = lo + j / nt1;
        if (traced) t_ready = wall_clock64();
        const TileDesc tile = ld_tile(&p.mtiles[m]);
        if constexpr (RAGGED) {
          tiled_ragged_gate_up_task(p, tile, static_cast<int>(j % nt1), pend, &ctl->xq[q].v);
        } else {
          tiled_gemm_task(p, tile, static_cast<int>(j % nt1), 0, pend, &ctl->xq[q].v);
        }
        pend = &p.g1_done[m].v;
        trace(t_dyn0 + lo * nt1 + j, 3, m, t_fetch, t_ready);
        j = task_notes()[0];
      } else {
        const unsigned jj = j - q1;
        const unsigned m = lo + jj / nt2;
        const TileDesc tile = ld_tile(&p.mtiles[m]);  // in flight while thread 0 looks at the counter
        if (pend != nullptr) {
          if (threadIdx.x == 0) sh.ok = ld_relaxed(&p.g1_done[m].v) >= nt1 ? 1u : 0u;
          __syncthreads();
          const bool ready = sh.ok != 0u;
          __syncthreads();
          if (!ready) flush();
        }
        ok = wg_wait_ge(p, &p.g1_done[m].v, nt1, &sh);
        if (ok) {
          if (traced) t_ready = wall_clock64();
          if constexpr (ODD) {
            tiled_odd_down_task(p, tile, static_cast<int>(jj % nt2), pend, &ctl->xq[q].v);
          } else if constexpr (RAGGED) {
            tiled_ragged_down_task(p, tile, static_cast<int>(jj % nt2), pend, &ctl->xq[q].v);
          } else {
            tiled_gemm_task(p, tile, static_cast<int>(jj % nt2), 1, pend, &ctl->xq[q].v);
          }
          pend = &ctl->g2_done.v;
          trace(t_dyn0 + nm * nt1 + lo * nt2 + jj, 4, m, t_fetch, t_ready);
          j = task_notes()[0];
        }
      }
    }
    flush();
  }

  // ---- combine tasks from the last global counter; float rows of y as the streaming variant sums them
  if (ok && n2_total != 0u) ok = wg_wait_ge(p, &ctl->g2_done.v, n2_total, &sh);
  if constexpr (RAGGED) {
    if (ok) {
      const unsigned ncomb = (static_cast<unsigned>(p.H) + COMBINE_COLS - 1u) / COMBINE_COLS;
      const unsigned slot = static_cast<unsigned>(uni(static_cast<int>(threadIdx.x >> 6))) * n_groups + blockIdx.x;
      combine_items<BF16>(p, slot, T * ncomb, ncomb, blockIdx.x, t_dyn0 + nm * (nt1 + nt2), trace_clock(traced));
    }
  }
  while (!RAGGED && ok) {
    const long long t_fetch = trace_clock(traced);
    if (threadIdx.x == 0) sh.ticket = add_relaxed(&ctl->cticket.v, 1u);
    __syncthreads();
    const unsigned c = sh.ticket;
    __syncthreads();
    if (c >= ncmb) break;
    const long long t_ready = trace_clock(traced);
    tiled_combine_task(p, static_cast<int>(c), cmb_tok);
    trace(t_dyn0 + nm * (nt1 + nt2) + c, 5, c, t_fetch, t_ready);
  }

  // The last workgroup out returns every counter to zero for the next launch.
  fence_release();  // flags this wave has raised for others have landed before anybody clears them
  __syncthreads();
  if (threadIdx.x == 0) sh.ok = (add_relaxed(&ctl->exit_count.v, 1u) == n_groups - 1u) ? 1u : 0u;
  __syncthreads();
  if (sh.ok) {
    const unsigned err = ldc(&ctl->error.v);
    if (err != 0u) {
      recover_after_error(p, err, static_cast<int>(threadIdx.x), T_THREADS);
      __syncthreads();
    }
    const unsigned nmr = min(ldc(&ctl->n_mtiles.v), static_cast<unsigned>(p.max_mtiles));
    for (unsigned i = threadIdx.x; i < nmr; i += T_THREADS) stc(&p.g1_done[i].v, 0u);
    for (unsigned g = threadIdx.x; g < n_groups; g += T_THREADS) {
      stc(&p.wgflags[g].f[FLAG_SCAN], 0u);
      stc(&p.wgflags[g].f[FLAG_PERM], 0u);
      stc(&p.wgflags[g].f[FLAG_G2], 0u);
      stc(&p.wgflags[g].f[FLAG_ROUTED], 0u);
    }
    if (threadIdx.x < 8) stc(&ctl->xq[threadIdx.x].v, 0u);
    if (threadIdx.x == 0) {
      stc(&ctl->launches.v, ldc(&ctl->launches.v) + 1u);
      stc(&ctl->router_done.v, 0u);
      stc(&ctl->perm_done.v, 0u);
      stc(&ctl->g2_done.v, 0u);
      stc(&ctl->n_mtiles.v, 0u);
      stc(&ctl->exit_count.v, 0u);
      stc(&ctl->cticket.v, 0u);
      stc(&ctl->scan_done.v, 0u);
      stc(&ctl->ticket.v, 0u);
    }
  }
}

// Largest token count of the tiled variant: the launcher's capacity at top-1.
int tiled_max_tokens() { return 1 << 21; }
// y of the tiled variant: one bf16 row of H per (token, slot); ragged shapes keep the streaming variant's float rows
size_t tiled_y_bytes(size_t rows, size_t hidden) { return rows * hidden * 2; }

namespace {
using TiledKernel = void (*)(const Params);
// [ragged, ragged with an odd I or neither][with task records]
const TiledKernel kTiledKernels[3][2] = {{moe_tiled_kernel<false, false, false>, moe_tiled_kernel<false, false, true>},
                                         {moe_tiled_kernel<true, false, false>, moe_tiled_kernel<true, false, true>},
                                         {moe_tiled_kernel<true, true, false>, moe_tiled_kernel<true, true, true>}};
}  // namespace

hipError_t launch_tiled_kernel(const Params& p, int grid, hipStream_t stream) {
  const int shape = !tiled_ragged(p.H, p.I) ? 0 : p.I % KS == 0 ? 1 : 2;
  hipLaunchKernelGGL(kTiledKernels[shape][p.trace != nullptr], dim3(grid), dim3(T_THREADS), TILED_LDS_BYTES, stream, p);
  return hipGetLastError();
}

hipError_t prepare_tiled_kernel() {
  for (const auto& kernels : kTiledKernels)
    for (TiledKernel kernel : kernels) {
      const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                               hipFuncAttributeMaxDynamicSharedMemorySize, TILED_LDS_BYTES);
      if (e != hipSuccess) return e;
    }
  return hipSuccess;
}

// the least of the kernels' numbers of workgroups a CU holds
hipError_t tiled_kernel_occupancy(int* per_cu) {
  *per_cu = 0x7FFFFFFF;
  for (const auto& kernels : kTiledKernels)
    for (TiledKernel kernel : kernels) {
      int n = 0;
      const hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, kernel, T_THREADS, TILED_LDS_BYTES);
      if (e != hipSuccess) return e;
      if (n < *per_cu) *per_cu = n;
    }
  return hipSuccess;
}

}  // namespace fmoe
