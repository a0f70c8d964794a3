// Persistent MoE kernel, split-k variant for gfx950: batches of up to 24 rows an expert (bf16,
// tiles of one or two 16-row blocks) or fewer than 10 (float32, one block). A wave of the streaming
// variant carries a task of 64 weight rows over the whole of k alone: with few experts in use
// most waves have no task at all and the others need 256 KiB each through one wave's window of
// loads (one token on the 30B shape: 192 tasks on 2048 waves), and with many the launch ends in
// a tail of whole tasks. Here the eight waves of a workgroup share a task's k (gate/up: eight
// parts; down: two tasks side by side in four parts, or one in eight where that leaves a CU idle),
// so tasks are an eighth as long, and meet in LDS: every wave leaves its partial sums there, one
// barrier, and one or two waves add the parts in k order and store. The window of loads does not
// drain between tasks: a slot is asked for again, for the step SPLIT_U later of the wave's sequence
// of tasks, as soon as its matrix instructions have read it. Tasks are handed out statically
// (equal shares of equal tasks), the routing tables are built by every workgroup for itself in
// LDS from the top-k entries, and there is one grid-wide dependency between gate/up and down,
// under which the first window of down weights is on its way. T=64 on the 30B shape, us from the
// launch's first workgroup (before workgroups posted their arrivals): routed 21, tables 24, gate/up done 119 to 141, h everywhere 144, down
// done 204, out 208.
//
// Bound by HBM from some 16 tokens on, below by the chain of waits (logit chains 14 us, selection,
// gate/up, down, combine). Against the streaming kernel, us, 30B shape, weights packed in place:
// T=1 59.5 -> 42 (routed 16, tables 19, gate/up 28, h everywhere 32, down 34; since every workgroup routes small
// batches for itself and posts its arrivals, 44.4 -> 40.2 in a row of passes), T=8 120 -> 103, T=16 164 -> 150, T=64 225 -> 217 (1.19 GB: 5.5 TB/s), T=128 243 -> 223,
// T=200 266 -> 234, T=256 275 -> 241; row-major T=32 249 -> 226, T=128 290 -> 261; 235B T=1 102 -> 87,
// T=64 759 -> 762, T=256 876 -> 836. Four hot experts: T=16 146 -> 120, T=128 317 -> 240 (a tile of more
// rows than an early task carries starts over there; here it is several tiles).
// float32, weights packed in place, streaming kernel -> here: E=8, H=256, I=128, k=2 T=16 44.8 -> 26.4; 30B
// shape T=1 105.9 -> 67.8, T=4 133.8 -> 127.7, T=16 302 -> 286, T=64 397 -> 397, T=128 420 -> 408 (with four hot
// experts 837 -> 449), T=159 543 -> 433; E=40, k=5, H=1344, I=736 T=1 91.6 -> 49.9, T=79 135 -> 113.
//
// Where the batch reaches most experts, the first workgroups (as many as whole experts fill; those
// with a routing task behind it) ask for the first window of (expert b / nt1, columns b % nt1)
// before the routing is known and keep it if the expert turns out to be in use.
//
// Replaces, for this regime, the reference's moeKernel
// (src/hip/kernel/moeKernel.h:37-107), its task executors
// (src/hip/kernel/tasks/*.h) and its queue (src/hip/taskSystem/*.h).
#include "moe_stream_device.h"

namespace fmoe {

// k-steps of a wave's window, by 16-row blocks of the tile (eight and six do not fit the registers
// beside the epilogue: with eight for one block the window's last loads were spilled, T = 64 306 us)
constexpr int split_u(int rb) { return rb == 1 ? 6 : 4; }
constexpr int SPLIT_MAX_TILES = MAX_EXPERTS + SPLIT_MAX_SLOTS / 16;
// LDS: the tables, then two sets of partial sums ([wave][weight block][row block][lane][4]); the
// routing tasks use it from its first byte on before that
constexpr int SPLIT_TILE_OFF = 0;
constexpr int SPLIT_MASK_OFF = SPLIT_TILE_OFF + SPLIT_MAX_TILES * 8;
constexpr int SPLIT_W_OFF = SPLIT_MASK_OFF + SCAN_LDS_WORDS * 8;
constexpr int SPLIT_PERM_OFF = SPLIT_W_OFF + SPLIT_MAX_SLOTS * 4;
constexpr int SPLIT_TOK_OFF = SPLIT_PERM_OFF + SPLIT_MAX_SLOTS * 2;
constexpr int SPLIT_OFF_OFF = SPLIT_TOK_OFF + SPLIT_MAX_SLOTS * 2;
constexpr int SPLIT_SPEC_OFF = SPLIT_OFF_OFF + MAX_EXPERTS * 4;
constexpr int SPLIT_NOTE_OFF = SPLIT_SPEC_OFF + MAX_EXPERTS * 4;
constexpr int SPLIT_PART_OFF = SPLIT_NOTE_OFF + 64;
static_assert(SPLIT_PART_OFF % 16 == 0, "partial sums are read 16 bytes at a time");
constexpr int split_part_bytes(int rb) { return 8 * 4 * rb * 64 * 16; }
constexpr int split_lds_bytes(int rb) {
  const int n = SPLIT_PART_OFF + 2 * split_part_bytes(rb);
  return n > 8 * ROUTER_LDS_FLOATS * 4 ? n : 8 * ROUTER_LDS_FLOATS * 4;
}
static_assert(split_lds_bytes(2) + 64 <= 160 * 1024, "LDS of a workgroup");
// small batches' winners, and what the waves need to find them, where the partial sums go later
constexpr int SPLIT_SELF_OFF = SPLIT_PART_OFF;
constexpr int SPLIT_SELECT_OFF = SPLIT_SELF_OFF + SPLIT_SELF_TOKENS * MAX_TOPK * 8;
static_assert(SPLIT_SELECT_OFF + 8 * SELECT_ROWS_BYTES <= split_lds_bytes(1), "winners exceed the partial sums");

// Which steps of a task's k a wave takes. `runs` false (batches that leave most experts unused: a CU has
// a task at most): one of `parts` equal stretches. Otherwise every parts-th run of four steps (256 bytes of a
// row; of two or one where the steps do not divide into such runs), from one of up to four places
// that moves with the task's column block and once around: the eight waves then read a stretch of
// 32 KiB (packed) or 2 KiB of each row, and the CUs do not all read at the same offset of their rows, which for
// pitches of 4 KiB and more are the same channels. us, equal stretches / as here, packed: bf16 30B shape T=64
// 209.9 / 207.0, 235B T=64 742 / 733, T=200 797 / 788, float32 30B T=128 412 / 408; row-major: bf16 30B
// T=64 241.6 / 238.4, T=200 273.6 / 268.5, 235B T=64 888 / 860, T=200 1009 / 970, float32 30B T=64 499 / 474,
// T=128 521 / 498. Where the steps do not divide into runs of two, row-major weights gain too (bf16 E=60, k=4,
// H=2304, I=1408 T=100 262 / 251, T=200 289 / 276, E=128, k=8, H=2048, I=800 T=100 262 / 258), packed ones do not (E=60 T=100
// 210.1 / 210.4, T=200 222.8 / 223.7; float32 E=128, k=8, H=2880, I=1440 T=64 964 / 978, E=64, k=6, H=2240, I=1376 T=100
// 402 / 408): they go along, because both forms of the weights give the same bits. Down projections with rows of
// whole 8 KiB keep the stretches as well (row-major, runs / stretches there, bf16 E=16, k=4, H=1024, I=4096 T=24 106.6 /
// 100.4, I=8192 T=24 187.1 / 167.1, E=32, k=4, H=2048, I=4096 T=24 298.6 / 293.1; float32 E=16, k=4, H=1024, I=4096 T=24 199.9 /
// 174.5, but H=2048, E=32 T=48 621 / 633; packed level: bf16 H=1024, I=4096 86.4 / 86.4, I=8192 145.2 / 144.9). Without the moving start, bf16 row-major 235B T=64 933, float32 30B T=128 576; runs of two with
// it 900 and 537, of eight 880 and 501; starts next to each other instead of far apart, float32 row-major
// H=4096, I=512 T=100 389 instead of 373.
struct SplitSteps {
  int first, count;       // first step, number of steps
  int jump;               // from the last step of a run to the wave's next
  int shift, mask;        // steps of a run: 1 << shift, less one
  int starts, apart;      // places where it may start, less one: 0, 1 or 3; runs from one to the next
  __device__ __forceinline__ int start(int column) const { return ((column & starts) * apart) << shift; }
  __device__ __forceinline__ int at(int start) const { return first + (start >> shift) * (jump + mask); }
  __device__ __forceinline__ int span() const { return (count >> shift) * (jump + mask); }
};
__device__ __forceinline__ SplitSteps split_steps(int steps, int part, int log_parts, bool runs) {
  SplitSteps s;
  const int parts = 1 << log_parts;
  s.shift = 0;
  if (runs) {
    s.shift = max(0, min(2, __builtin_ctz(steps) - log_parts));
    const int n = steps >> (s.shift + log_parts);  // runs that every wave has
    s.starts = n >= 4 ? 3 : n >= 2 ? 1 : 0;
    s.apart = n >= 4 ? n >> 2 : 1;
    s.first = part << s.shift;
    s.count = (((steps >> s.shift) - part + parts - 1) >> log_parts) << s.shift;
    s.jump = ((parts - 1) << s.shift) + 1;
    s.mask = (1 << s.shift) - 1;
  } else {
    s.first = (steps * part) >> log_parts;
    s.count = ((steps * (part + 1)) >> log_parts) - s.first;
    s.jump = 1;
    s.apart = 1;
    s.mask = 0;
    s.starts = 0;
  }
  return s;
}

// A tile as the tables hold it: at most 16 * RB rows of one expert.
struct SplitTile {
  int expert, row0, rows;
};
__device__ __forceinline__ SplitTile split_tile(const uint2* tiles, int i) {
  const uint2 v = tiles[i];
  SplitTile t;
  t.expert = __builtin_amdgcn_readfirstlane(static_cast<int>(v.x));
  const int rr = __builtin_amdgcn_readfirstlane(static_cast<int>(v.y));
  t.row0 = rr & 0xFFFF;
  t.rows = rr >> 16;
  return t;
}

// The window: U k-steps of four 16-row weight blocks and RB blocks of token rows. PACKED weights
// are one run of 4 KiB a step; row-major ones four row-order loads (see fragment_from_row_order).
template <typename DT, bool PACKED, bool DOWN, int RB>
struct SplitStream {
  static constexpr int NP = PACKED ? 1 : 4;
  static constexpr int U = split_u(RB);
  uint4 a[U][4], b[U][RB];
  const unsigned char* ap[NP];   // where the next step's weights are
  const unsigned char* bp[RB];   // ... and its token rows (gate/up)
  unsigned boff[RB];             // ... or h rows, as offsets (down)
  int astep, bstep;              // bytes to the next step (0 behind the last task) ...
  int ajump, bjump, mask;        // ... from the last step of a run on; steps of a run - 1
  int aspan, bspan;              // from the task's first step to behind its last
  int left;                      // steps left of the task
  int turn;                      // ... when the pointers go back to its first step (0: they do not any more)
  CoherentBuffer cb;

  // Packed weights pass through the caches without staying, also where an expert has several tiles
  // that read them (unlike the streaming kernel's sweep): with ordinary loads they push the token
  // rows, h and y out of the L2s. us, non-temporal / ordinary, 30B shape: T=64 217 / 237, T=256 240 / 261,
  // with four hot experts T=64 207 / 220, T=256 269 / 272; 235B shape with four hot experts T=200 895 / 933.
  __device__ __forceinline__ void load_a(int u) {
#pragma unroll
    for (int i = 0; i < 4; ++i) a[u][i] = PACKED ? ld16_once(ap[0] + i * 1024) : ld16(ap[i]);
#pragma unroll
    for (int q = 0; q < NP; ++q) ap[q] += ((left - 1) & mask) == 0 ? ajump : astep;
  }
  __device__ __forceinline__ void load_b(int u) {
    const int step = ((left - 1) & mask) == 0 ? bjump : bstep;
#pragma unroll
    for (int r = 0; r < RB; ++r) {
      if (DOWN) {
        b[u][r] = ld16_agent(cb, boff[r]);
        boff[r] += static_cast<unsigned>(step);
      } else {
        b[u][r] = ld16(bp[r]);
        bp[r] += step;
      }
    }
  }
  // Behind the last task the loads go on (their number must not depend on a branch, or the
  // compiler waits for all of them at every step), all lanes at one address that exists.
  __device__ __forceinline__ void park(const void* somewhere) {
#pragma unroll
    for (int q = 0; q < NP; ++q) ap[q] = reinterpret_cast<const unsigned char*>(somewhere);
#pragma unroll
    for (int r = 0; r < RB; ++r) {
      bp[r] = reinterpret_cast<const unsigned char*>(somewhere);
      boff[r] = 0u;
    }
    astep = bstep = ajump = bjump = mask = 0;
    left = 0x7FFFFFFF;
    turn = 0;
  }
  // A step's loads (of A: weights, of B: token rows) are out: on to the next one, or to the next task.
  template <bool A, bool B, typename NextTask>
  __device__ __forceinline__ void advance(NextTask next_task) {
    if (--left != turn) return;
    if (left == 0) {
      next_task();
      return;
    }
    turn = 0;
#pragma unroll
    for (int q = 0; q < NP; ++q)
      if (A) ap[q] -= aspan;
#pragma unroll
    for (int r = 0; r < RB; ++r) {
      if (B && DOWN) boff[r] -= static_cast<unsigned>(bspan);
      if (B && !DOWN) bp[r] -= bspan;
    }
  }
  __device__ __forceinline__ void mma(int u, int pull_from, f32x4 (&acc)[4][RB]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint4 w = PACKED ? a[u][i] : fragment_from_row_order(a[u][i], pull_from);
#pragma unroll
      for (int r = 0; r < RB; ++r) acc[i][r] = mma16<DT>(w, b[u][r], acc[i][r]);
    }
  }
  // this wave's partial sums of a task go to LDS, and the accumulators back to zero
  __device__ __forceinline__ void leave(f32x4* part, int wave, f32x4 (&acc)[4][RB]) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int r = 0; r < RB; ++r) {
        part[((wave * 4 + i) * RB + r) * 64 + lane_id()] = acc[i][r];
        acc[i][r] = f32x4{0.f, 0.f, 0.f, 0.f};
      }
  }
};

template <typename DT, bool PACKED, int RB>
__global__ __launch_bounds__(512) __attribute__((disable_tail_calls)) void moe_split_kernel(const Params params) {
  ParamsRef p = kernel_params();
  __shared__ unsigned lds_flag[4];
  __shared__ unsigned lds_poller[4];
  if (threadIdx.x < 4) {
    lds_flag[threadIdx.x] = 0u;
    lds_poller[threadIdx.x] = 0u;
  }
  __syncthreads();
  const int tid = threadIdx.x, lane = lane_id();
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r16 = lane & 15, g = lane >> 4;
  const int G = static_cast<int>(gridDim.x), b = static_cast<int>(blockIdx.x);
  Control* ctl = p.ctl;
  const int T = p.T, E = p.E, H = p.H, K = p.K, I = p.I, W = p.W;
  unsigned char* lds = reinterpret_cast<unsigned char*>(lds_dyn);
  constexpr int U = split_u(RB), TILE_ROWS = 16 * RB;
  constexpr int ESZ = 16 / DT::EPV;
  unsigned short* lperm = reinterpret_cast<unsigned short*>(lds + SPLIT_PERM_OFF);  // permuted row -> token*K + slot
  unsigned short* ltok = reinterpret_cast<unsigned short*>(lds + SPLIT_TOK_OFF);    // permuted row -> token
  float* lw = reinterpret_cast<float*>(lds + SPLIT_W_OFF);      // permuted row -> gate weight
  unsigned long long* lmask = reinterpret_cast<unsigned long long*>(lds + SPLIT_MASK_OFF);
  int* loff = reinterpret_cast<int*>(lds + SPLIT_OFF_OFF);      // expert -> first permuted row
  uint2* tiles = reinterpret_cast<uint2*>(lds + SPLIT_TILE_OFF);
  int* spec_tile = reinterpret_cast<int*>(lds + SPLIT_SPEC_OFF);  // expert -> its early tile, or -1
  int* note = reinterpret_cast<int*>(lds + SPLIT_NOTE_OFF);

  // logit chains: bf16 16 tokens x 16 experts a workgroup, float32 8 x 8 a wave
  constexpr int DOT = DT::EPV == 8 ? 16 : ROUTER_EXP;
  const int n_eg = (E + DOT - 1) / DOT;
  const int n_dot = ((T + DOT - 1) / DOT) * n_eg;
  const int n_rt = DT::EPV == 8 ? n_dot : min(n_dot, G >> 1);  // workgroups with routing tasks
  const int nt1 = I / (16 * G1_NB), nt2 = H / (16 * G2_NB);
  const int ks1 = H / (4 * DT::EPV), ks2 = I / (4 * DT::EPV);  // steps of 64 bytes a row
  const int pull_from = (((lane & 15) << 2) | (lane >> 4)) << 2;
  const unsigned raised = post_number(ldc(&ctl->launches.posted));  // (the last workgroup out moves it on)

  // ---- routing: logit chains on the first workgroups, then (batches that split_self leaves out) selections there,
  // four or two tokens a wave. Smaller batches have every workgroup pick all winners for itself, below: that saves the
  // entries' way to memory and back and a wait in between (us, without / with: one token 41.8 / 40.2, T=11 123.2 /
  // 120.9, E=8, H=256 float32 T=16 24.4 / 23.1; but T=40 199.1 / 200.3, T=64 205.7 / 207.6, H=512, E=64 float32 T=64 44.1 /
  // 45.5).
  const bool self = split_self(E, K, T);
  const int tok = select_tokens(E, K, T);
  if (b < n_rt) {
    if constexpr (DT::EPV == 8) {
      router_dot16_task(p, b / n_eg, b % n_eg, self ? b : -1, raised);
    } else {
      for (int q = b + n_rt * wave; q < n_dot; q += 8 * n_rt) router_dot_task<DT>(p, q / n_eg, q % n_eg, self ? q : -1, raised);
    }
    for (int i = b + n_rt * wave; !self && i * tok < T; i += 8 * n_rt) {
      if (router_select_tokens_task(p, i, static_cast<unsigned>(n_eg), lds + wave * (ROUTER_LDS_FLOATS * 4)) == 0) break;
      raise_post(p, POST_ROUTE, i, raised);
    }
  }

  // ---- gate/up weights before the routing is known
  const int n_spec_experts = p.split_spec ? min(G / nt1, E) : 0;
  const int n_spec = n_spec_experts * nt1;  // workgroups b < n_spec
  const SplitSteps sk1 = split_steps(ks1, wave, 3, p.split_spec != 0);
  const int steps1 = sk1.count;
  f32x4 acc[4][RB];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int r = 0; r < RB; ++r) acc[i][r] = f32x4{0.f, 0.f, 0.f, 0.f};
  bool ok;
  int ntiles = 0;
  int cnt = 0;  // tasks this workgroup has finished: its parity names the set of partial sums
  {
    SplitStream<DT, PACKED, false, RB> st;
    st.cb = coherent_buffer(p.h, 0u);
    auto weights = [&](int expert, int nblk) {
      const int start = sk1.start(nblk), k0 = sk1.at(start);
      if constexpr (PACKED) {
        const size_t task = static_cast<size_t>(expert) * nt1 + nblk;
        st.ap[0] = reinterpret_cast<const unsigned char*>(p.ffn1_packed) + (task * ks1 + k0) * 4096 + lane * 16;
        st.astep = 4096;
        st.ajump = 4096 * sk1.jump;
        st.aspan = 4096 * sk1.span();
      } else {
        const unsigned char* w13 = reinterpret_cast<const unsigned char*>(p.ffn1) +
                                   static_cast<size_t>(expert) * 2 * I * H * ESZ + k0 * 64 + row_order_chunk() * 16;
        const int n0 = nblk * (16 * G1_NB) + row_order_row();
#pragma unroll
        for (int q = 0; q < G1_NB; ++q) {
          st.ap[q] = w13 + static_cast<size_t>(n0 + 16 * q) * H * ESZ;
          st.ap[G1_NB + q] = w13 + static_cast<size_t>(I + n0 + 16 * q) * H * ESZ;
        }
        st.astep = 64;
        st.ajump = 64 * sk1.jump;
        st.aspan = 64 * sk1.span();
      }
      st.left = steps1;
      st.turn = start;
      st.mask = sk1.mask;
    };
    if (b < n_spec) {
      weights(b / nt1, b % nt1);
    } else {
      st.park(p.gate);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      st.load_a(u);
      // (a task shorter than the window: the slots behind it are filled again below)
      st.template advance<true, false>([&] { st.park(p.gate); });
      __builtin_amdgcn_sched_barrier(0);
    }

    // ---- tables, by every workgroup for itself
    ok = wait_posts(p, post_row(p, POST_ROUTE, b % POST_COPIES), self ? n_dot : (T + tok - 1) / tok, raised,
                    &lds_flag[FLAG_ROUTED], &lds_poller[FLAG_ROUTED]);
    const int wact = (T + 63) >> 6;
    const int n = T * K;
    lds_barrier();  // the routing tasks' use of the LDS is over
    int* self_idx = reinterpret_cast<int*>(lds + SPLIT_SELF_OFF);                        // [T][K]
    float* self_w = reinterpret_cast<float*>(self_idx + SPLIT_SELF_TOKENS * MAX_TOPK);
    if (self) {
      for (int e = tid; e < E; e += 512) lmask[e] = 0ull;
      lds_barrier();
      for (int i = wave; ok && i * tok < T; i += 8) {
        const int t0 = i * tok, nt = min(tok, T - t0), row = lane * tok >> 6, t = row < nt ? t0 + row : -1;
        auto emit = [&](int tq, int s, int e, float w) {
          self_idx[tq * K + s] = e;
          self_w[tq * K + s] = w;
          if (e >= 0) atomicOr(&lmask[e], 1ull << tq);
          if (b == G - 1) {  // (what the host may read back)
            stc(&p.topk_idx[tq * K + s], e);
            stc(&p.topk_w[tq * K + s], w);
          }
        };
        unsigned char* scratch = lds + SPLIT_SELECT_OFF + wave * SELECT_ROWS_BYTES;
        if (E <= 128) {
          unsigned val[8];
          load_row_keys<8, 16>(p, t0, nt, val);
          router_select_rows<8, 16>(K, t, val, scratch, emit);
        } else if (tok == 4) {
          unsigned val[16];
          load_row_keys<16, 16>(p, t0, nt, val);
          router_select_rows<16, 16>(K, t, val, scratch, emit);
        } else {
          unsigned val[8];
          load_row_keys<8, 32>(p, t0, nt, val);
          router_select_rows<8, 32>(K, t, val, scratch, emit);
        }
      }
      lds_barrier();
    }
    int ee[SPLIT_MAX_SLOTS / 512];
    float ww[SPLIT_MAX_SLOTS / 512];
    if (ok) {
#pragma unroll
      for (int q = 0; q < SPLIT_MAX_SLOTS / 512; ++q) {
        const int i = tid + 512 * q;
        ee[q] = i >= n ? -1 : self ? self_idx[i] : ldc(&p.topk_idx[i]);
        ww[q] = i >= n ? 0.0f : self ? self_w[i] : ldc(&p.topk_w[i]);
      }
      for (int i = tid; !self && i < E * wact; i += 512) lmask[i] = ldc(&p.masks[static_cast<size_t>(i / wact) * W + i % wact]);
    }
    lds_barrier();
    if (ok && wave == 0) {
      int base = 0, rest = 0, spec = 0;
      const int epl = (E + 63) >> 6;
      for (int pass = 0; pass < 2; ++pass) {  // the early tiles stand behind all others
        if (pass == 1) base = 0;
        for (int j = 0; j < epl; ++j) {
          const int e = lane + 64 * j;
          int c = 0;
          if (e < E)
            for (int w = 0; w < wact; ++w) c += __popcll(lmask[e * wact + w]);
          const int off = base + wave_inclusive_scan(c) - c;
          base = __shfl(off + c, 63, 64);
          const int nt = (c + TILE_ROWS - 1) / TILE_ROWS;
          const bool early = e < n_spec_experts && c > 0;
          const int mine = pass == 0 ? nt - (early ? 1 : 0) : (early ? 1 : 0);
          const int incl = wave_inclusive_scan(mine);
          if (pass == 0) {
            if (e < E) loff[e] = off;
            for (int i = 0; i < mine; ++i) {
              const int r = (i + (early ? 1 : 0)) * TILE_ROWS;
              tiles[rest + incl - mine + i] =
                  make_uint2(static_cast<unsigned>(e), static_cast<unsigned>((off + r) | (min(TILE_ROWS, c - r) << 16)));
            }
            rest += __shfl(incl, 63, 64);
          } else {
            if (e < E) spec_tile[e] = early ? rest + spec + incl - 1 : -1;
            if (early)
              tiles[rest + spec + incl - 1] =
                  make_uint2(static_cast<unsigned>(e), static_cast<unsigned>(off | (min(TILE_ROWS, c) << 16)));
            spec += __shfl(incl, 63, 64);
          }
        }
      }
      if (lane == 0) {
        note[0] = rest;
        note[1] = rest + spec;
        note[2] = base;
      }
    }
    lds_barrier();
    int n_rest = 0;
    if (ok) {
      n_rest = __builtin_amdgcn_readfirstlane(note[0]);
      ntiles = __builtin_amdgcn_readfirstlane(note[1]);
#pragma unroll
      for (int q = 0; q < SPLIT_MAX_SLOTS / 512; ++q) {
        const int i = tid + 512 * q;
        if (ee[q] >= 0) {
          const int t = i / K, wd = t >> 6;
          int pos = loff[ee[q]] + __popcll(lmask[ee[q] * wact + wd] & ((1ull << (t & 63)) - 1ull));
          for (int w = 0; w < wd; ++w) pos += __popcll(lmask[ee[q] * wact + w]);
          lperm[pos] = static_cast<unsigned short>(i);
          ltok[pos] = static_cast<unsigned short>(t);
          lw[pos] = ww[q];
          if (b == G - 1) stc(&p.perm[pos], i);
        }
      }
      if (b == G - 1) {  // the tables the host may read back
        const int total = note[2];
        for (int e = tid; e < E; e += 512) {
          const int off = loff[e];
          stc(&p.expert_offset[e], off);
          stc(&p.expert_count[e], (e + 1 < E ? loff[e + 1] : total) - off);
        }
        if (tid == 0) stc(&p.expert_offset[E], total);
      }
    }
    lds_barrier();

    // ---- gate/up: the early task, then an equal share of the rest (workgroups without an early
    // task first)
    const int my_spec = ok && b < n_spec ? __builtin_amdgcn_readfirstlane(spec_tile[b / nt1]) : -1;
    const int rank = b >= n_spec ? b - n_spec : b + G - n_spec;
    const int n_tasks = n_rest * nt1;
    int ntask = (my_spec >= 0 ? 1 : 0) + (rank < n_tasks ? (n_tasks - rank + G - 1) / G : 0);
    int lq = rank;  // next task of the rest to load, and (cq) to finish
    int cq = rank;
    bool cspec = my_spec >= 0;
    auto rows_of = [&](const SplitTile& t, int nblk) {
      const int k0 = sk1.at(sk1.start(nblk));
#pragma unroll
      for (int r = 0; r < RB; ++r)
        st.bp[r] = reinterpret_cast<const unsigned char*>(p.tokens) +
                   static_cast<size_t>(ltok[t.row0 + min(16 * r + r16, t.rows - 1)]) * H * ESZ + k0 * 64 + g * 16;
      st.bstep = 64;
      st.bjump = 64 * sk1.jump;
      st.bspan = 64 * sk1.span();
    };
    auto next_task = [&]() {
      if (lq < n_tasks) {
        const SplitTile t = split_tile(tiles, lq / nt1);
        weights(t.expert, lq % nt1);
        rows_of(t, lq % nt1);
        lq += G;
      } else {
        st.park(p.gate);
      }
    };
    auto finish = [&]() {  // the task's eight parts: add up, SiLU(gate) * up, store
      const int q = cspec ? b : cq;
      const SplitTile t = split_tile(tiles, cspec ? my_spec : q / nt1);
      const int n0 = (q % nt1) * (16 * G1_NB);
      if (!cspec) cq += G;
      cspec = false;
      f32x4* part = reinterpret_cast<f32x4*>(lds + SPLIT_PART_OFF + (cnt & 1) * split_part_bytes(RB));
      st.leave(part, wave, acc);
      lds_barrier();
      const int turn = (wave - 2 * RB * cnt) & 7;  // the adding waves take turns
      const int i = turn & 1, r = turn >> 1;
      ++cnt;
      if (r < RB) {
        f32x4 s = part[(i * RB + r) * 64 + lane], v = part[((i + 2) * RB + r) * 64 + lane];
#pragma unroll 1  // (more reads in flight cost the window its registers)
        for (int w = 1; w < 8; ++w) {
          s += part[((w * 4 + i) * RB + r) * 64 + lane];
          v += part[((w * 4 + i + 2) * RB + r) * 64 + lane];
        }
        const int row = 16 * r + r16;
        if (row < t.rows) {
          unsigned hv[4];
#pragma unroll
          for (int k = 0; k < 4; ++k) {  // (one after the other, for the same reason)
            const float x = silu_mul(s[k], v[k]);
            hv[k] = DT::EPV == 8 ? f2bf(x) : __float_as_uint(x);
            __builtin_amdgcn_sched_barrier(0);
          }
          const size_t at = static_cast<size_t>(t.row0 + row) * I + n0 + 16 * i + 4 * g;
          if constexpr (DT::EPV == 8) {
            const unsigned lo = hv[0] | (hv[1] << 16), hi = hv[2] | (hv[3] << 16);
            stc(reinterpret_cast<unsigned long long*>(reinterpret_cast<unsigned short*>(p.h) + at),
                static_cast<unsigned long long>(lo) | (static_cast<unsigned long long>(hi) << 32));
          } else {
            st16_through(reinterpret_cast<float*>(p.h) + at, make_uint4(hv[0], hv[1], hv[2], hv[3]));
          }
        }
      }
    };
    if (ntask > 0) {
      if (my_spec >= 0 && steps1 >= U) {
        // the window is this task's: its token rows join it
        rows_of(split_tile(tiles, my_spec), b % nt1);
        st.left = steps1;
        st.turn = sk1.start(b % nt1);
        st.mask = sk1.mask;
#pragma unroll
        for (int u = 0; u < U; ++u) {
          st.load_b(u);
          st.template advance<false, true>(next_task);
        }
      } else {
        if (my_spec >= 0) {
          weights(b / nt1, b % nt1);
          rows_of(split_tile(tiles, my_spec), b % nt1);
        } else {
          next_task();
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
          st.load_a(u);
          st.load_b(u);
          st.template advance<true, true>(next_task);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      int cleft = steps1;
      auto round = [&]() {  // true: the last task is finished
#pragma unroll
        for (int u = 0; u < U; ++u) {
          st.mma(u, pull_from, acc);
          __builtin_amdgcn_sched_barrier(0);
          st.load_a(u);
          st.load_b(u);
          __builtin_amdgcn_sched_barrier(0);
          st.template advance<true, true>(next_task);
          if (--cleft == 0) {
            finish();
            if (--ntask == 0) return true;
            cleft = steps1;
          }
        }
        return false;
      };
      if (!round()) {
        asm volatile("; end of the first round" ::: "memory");  // as in stream_mma
        while (!round()) {
        }
      }
    }
  }

  // ---- every h row is final once all workgroups have been here
  const int parts = p.split_down;            // waves that share a down task: 4 or 8
  const int sub = wave & (parts - 1), grp = parts == 8 ? 0 : wave >> 2;
  const int per_tile = parts == 8 ? nt2 : nt2 >> 1;  // workgroup tasks of one tile
  if (ok) {
    fence_release();
    lds_barrier();
    if (wave == 0) raise_post(p, POST_GATE_UP, b, raised);
    const SplitSteps sk2 = split_steps(ks2, sub, parts == 8 ? 3 : 2, p.split_spec != 0 && I * ESZ % 8192 != 0);
    const int steps2 = sk2.count;
    const int n_tasks = ntiles * per_tile;
    int ntask = b < n_tasks ? (n_tasks - b + G - 1) / G : 0;
    if (ntask > 0) {
      SplitStream<DT, PACKED, true, RB> st;
      st.cb = coherent_buffer(p.h, static_cast<unsigned>(T * K * I * ESZ));
      int lq = b, cq = b;
      auto next_task = [&]() {
        if (lq < n_tasks) {
          const SplitTile t = split_tile(tiles, lq / per_tile);
          const int nblk = parts == 8 ? lq % per_tile : (lq % per_tile) * 2 + grp;
          const int start = sk2.start(nblk), d0 = sk2.at(start);
          if constexpr (PACKED) {
            const size_t task = static_cast<size_t>(t.expert) * nt2 + nblk;
            st.ap[0] = reinterpret_cast<const unsigned char*>(p.ffn2_packed) + (task * ks2 + d0) * 4096 + lane * 16;
            st.astep = 4096;
            st.ajump = 4096 * sk2.jump;
            st.aspan = 4096 * sk2.span();
          } else {
            const unsigned char* w2 = reinterpret_cast<const unsigned char*>(p.ffn2) +
                                      static_cast<size_t>(t.expert) * H * I * ESZ + d0 * 64 + row_order_chunk() * 16;
            const int n0 = nblk * (16 * G2_NB) + row_order_row();
#pragma unroll
            for (int q = 0; q < st.NP; ++q) st.ap[q] = w2 + static_cast<size_t>(n0 + 16 * q) * I * ESZ;
            st.astep = 64;
            st.ajump = 64 * sk2.jump;
            st.aspan = 64 * sk2.span();
          }
#pragma unroll
          for (int r = 0; r < RB; ++r)
            st.boff[r] = static_cast<unsigned>((t.row0 + min(16 * r + r16, t.rows - 1)) * I * ESZ + d0 * 64 + g * 16);
          st.bstep = 64;
          st.bjump = 64 * sk2.jump;
          st.bspan = 64 * sk2.span();
          st.left = steps2;
          st.turn = start;
          st.mask = sk2.mask;
          lq += G;
        } else {
          st.park(p.gate);
        }
      };
      // The weights of the first window go out before the wait, the h rows behind it: both walk
      // through the same steps.
      next_task();
      const int lq0 = lq, turn0 = st.turn;
      unsigned boff0[RB];
#pragma unroll
      for (int r = 0; r < RB; ++r) boff0[r] = st.boff[r];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        st.load_a(u);
        st.template advance<true, false>(next_task);
        __builtin_amdgcn_sched_barrier(0);
      }
      ok = wait_posts(p, post_row(p, POST_GATE_UP, b % POST_COPIES), G, raised, &lds_flag[FLAG_PERM], &lds_poller[FLAG_PERM]);
      if (ok) {
        const unsigned char* keep[st.NP];
#pragma unroll
        for (int q = 0; q < st.NP; ++q) keep[q] = st.ap[q];
        const int keep_step = st.astep, keep_jump = st.ajump;
        lq = lq0;
#pragma unroll
        for (int r = 0; r < RB; ++r) st.boff[r] = boff0[r];
        st.bstep = 64;
        st.bjump = 64 * sk2.jump;
        st.bspan = 64 * sk2.span();
        st.left = steps2;
        st.turn = turn0;
        st.mask = sk2.mask;
#pragma unroll
        for (int u = 0; u < U; ++u) {
          st.load_b(u);
          st.template advance<false, true>(next_task);
          __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int q = 0; q < st.NP; ++q) st.ap[q] = keep[q];
        st.astep = keep_step;
        st.ajump = keep_jump;
        auto finish = [&]() {
          const SplitTile t = split_tile(tiles, cq / per_tile);
          const int n0 = (parts == 8 ? cq % per_tile : (cq % per_tile) * 2 + grp) * (16 * G2_NB);
          cq += G;
          f32x4* part = reinterpret_cast<f32x4*>(lds + SPLIT_PART_OFF + (cnt & 1) * split_part_bytes(RB));
          st.leave(part, wave, acc);
          lds_barrier();
          // (four blocks for eight waves: one half of them, then the other)
          const int first = parts > 4 * RB ? (sub + 4 * (cnt & 1)) & 7 : sub;
          ++cnt;
          for (int blk = first; blk < 4 * RB; blk += parts) {
            const int i = blk & 3, r = blk >> 2;
            f32x4 s = part[((grp * 16 + i) * RB + r) * 64 + lane];
#pragma unroll 1
            for (int w = 1; w < parts; ++w) s += part[(((grp * 4 + w) * 4 + i) * RB + r) * 64 + lane];
            const int row = 16 * r + r16;
            if (row < t.rows) {
              const float wt = lw[t.row0 + row];
              st16_through(p.y + static_cast<size_t>(lperm[t.row0 + row]) * H + n0 + 16 * i + 4 * g,
                           make_uint4(__float_as_uint(s[0] * wt), __float_as_uint(s[1] * wt),
                                      __float_as_uint(s[2] * wt), __float_as_uint(s[3] * wt)));
            }
          }
        };
        int cleft = steps2;
        auto round = [&]() {
#pragma unroll
          for (int u = 0; u < U; ++u) {
            st.mma(u, pull_from, acc);
            __builtin_amdgcn_sched_barrier(0);
            st.load_a(u);
            st.load_b(u);
            __builtin_amdgcn_sched_barrier(0);
            st.template advance<true, true>(next_task);
            if (--cleft == 0) {
              finish();
              if (--ntask == 0) return true;
              cleft = steps2;
            }
          }
          return false;
        };
        if (!round()) {
          asm volatile("; end of the first round" ::: "memory");
          while (!round()) {
          }
        }
      }
    }
  }

  // ---- combine, by the waves that have an item
  if (ok) {
    fence_release();
    lds_barrier();
    if (wave == 0) raise_post(p, POST_DOWN, b, raised);
    const unsigned ncomb = static_cast<unsigned>((H + COMBINE_COLS - 1) / COMBINE_COLS);
    const unsigned nc = static_cast<unsigned>(T) * ncomb;
    const unsigned slot = static_cast<unsigned>(wave * G + b);
    if (slot < nc && wait_posts(p, post_row(p, POST_DOWN, b % POST_COPIES), G, raised, &lds_flag[FLAG_G2], &lds_poller[FLAG_G2]))
      combine_items<DT>(p, slot, nc, ncomb, static_cast<unsigned>(b * 8 + wave), 0u, 0);
  }

  // ---- the last workgroup out counts the launch
  __syncthreads();
  if (wave == 0) {
    fence_release();  // flags this wave has raised for others have landed before anybody clears them
    unsigned last = 0;
    if (lane == 0) last = add_relaxed(&ctl->exit_count.v, 1u) == static_cast<unsigned>(G) - 1u ? 1u : 0u;
    if (__builtin_amdgcn_readfirstlane(last) != 0u) {
      const unsigned err = ldc(&ctl->error.v);
      if (err != 0u) recover_after_error(p, err, lane, 64);
      const unsigned posted = posted_by(raised);
      if (posted == 0u)
        for (int q = lane; q < POST_PHASES * POST_COPIES * POST_PITCH; q += 64) stc(&p.posts[q], 0u);
      if (lane == 0) {
        stc(&ctl->launches.v, ldc(&ctl->launches.v) + 1u);
        stc(&ctl->launches.posted, posted);
        stc(&ctl->exit_count.v, 0u);
      }
    }
  }
}

namespace {
// The kernels, and the dynamic LDS each is launched with.
struct SplitUse {
  const void* kernel;
  int lds;
};
const SplitUse kSplitUses[] = {{reinterpret_cast<const void*>(moe_split_kernel<BF16, true, 1>), split_lds_bytes(1)},
                               {reinterpret_cast<const void*>(moe_split_kernel<BF16, false, 1>), split_lds_bytes(1)},
                               {reinterpret_cast<const void*>(moe_split_kernel<BF16, true, 2>), split_lds_bytes(2)},
                               {reinterpret_cast<const void*>(moe_split_kernel<BF16, false, 2>), split_lds_bytes(2)},
                               {reinterpret_cast<const void*>(moe_split_kernel<F32, true, 1>), split_lds_bytes(1)},
                               {reinterpret_cast<const void*>(moe_split_kernel<F32, false, 1>), split_lds_bytes(1)}};
}  // namespace

hipError_t launch_split_kernel(const Params& p, int dtype, int grid, hipStream_t stream) {
  const bool packed = p.ffn1_packed != nullptr;
  auto* kernel = dtype == DT_F32 ? (packed ? moe_split_kernel<F32, true, 1> : moe_split_kernel<F32, false, 1>)
                 : p.split == 1  ? (packed ? moe_split_kernel<BF16, true, 1> : moe_split_kernel<BF16, false, 1>)
                                 : (packed ? moe_split_kernel<BF16, true, 2> : moe_split_kernel<BF16, false, 2>);
  hipLaunchKernelGGL(kernel, dim3(grid), dim3(512), split_lds_bytes(p.split), stream, p);
  return hipGetLastError();
}

hipError_t prepare_split_kernel() {
  for (const SplitUse& u : kSplitUses) {
    const hipError_t e = hipFuncSetAttribute(u.kernel, hipFuncAttributeMaxDynamicSharedMemorySize, u.lds);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

// the least of the kernels' numbers of workgroups a CU holds
hipError_t split_kernel_occupancy(int* per_cu) {
  *per_cu = 0x7FFFFFFF;
  for (const SplitUse& u : kSplitUses) {
    int n = 0;
    const hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, u.kernel, 512, u.lds);
    if (e != hipSuccess) return e;
    if (n < *per_cu) *per_cu = n;
  }
  return hipSuccess;
}

}  // namespace fmoe
