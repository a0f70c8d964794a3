// Shared host/device description of one launch of the fused MoE layer.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace fmoe {

enum : int { DT_F32 = 0, DT_BF16 = 1 };

// Error bits a kernel may raise in Control::error (sticky until the host
// clears it).
enum : unsigned {
  ERR_TIMEOUT = 1u,   // a bounded dependency wait ran out
  ERR_CAPACITY = 2u,  // more row tiles than the tables were sized for
};

// Rows of one expert handled by one tile task of the streaming ("skinny") path.
constexpr int SKINNY_MT = 64;
// Widths of one wave task: gate/up task = 32 gate + 32 up weight rows,
// down task = 64 weight rows.
constexpr int G1_NB = 2;  // 16-wide column blocks per gate/up wave task
constexpr int G2_NB = 4;  // 16-wide column blocks per down wave task
// Output columns summed by one combine task.
constexpr int COMBINE_COLS = 256;
constexpr int ROUTER_TOK = 8;    // streaming variant: tokens per router dot task
constexpr int ROUTER_EXP = 8;    // streaming variant: experts per router dot task
constexpr int DOT16_KC = 256;    // streaming variant, matrix-core router: k per LDS stage
constexpr int SCAN_LDS_WORDS = 1024;  // mask words (experts x 64-token words) the small-batch scan keeps in LDS
constexpr int SHORT_MASK_WORDS = 8192;  // the same for the tiled kernel's short prologue
constexpr int SPLIT_MAX_SLOTS = 2048;  // split-k kernel: (token, slot) entries its tables hold
constexpr int SPLIT_SELF_TOKENS = 32;  // ... tokens every workgroup may pick the winners of by itself
// Tokens whose winners one wave picks side by side (router_select_rows), where other waves have left the logits in memory.
// A winner costs a lane some 10 instructions and 5 for each expert it holds; of more than 128 experts those of four tokens
// are 16 a lane, of two 8. Twice as many counts of selections against that: so two while there are few tokens to a winner.
// us, one token / four / two, H=1024, I=256, E=256: k=32 T=1 43.9 / 44.6 / 40.7, T=31 97.0 / 101.1 / 96.8, k=16 T=8 56.4 /
// 57.1 / 54.8, k=8 T=8 42.9 / 40.6 / 39.6; tiled, E=160, k=32: T=384 106.7 / 113.6 / 111.1, T=768 145.1 / 142.9 / 141.2, k=16 T=600 105.4 /
// 103.7 / 104.0; float32 T=100 145.6 / 153.1 / 148.9.
constexpr __host__ __device__ int select_tokens(int E, int K, int T) { return E > 128 && T <= 24 * K ? 2 : 4; }
// Split-k kernel: every workgroup picks all winners for itself, while its eight waves do it in one go (E=256, k=8, T=24 so
// with four tokens a wave 62.6 us, from the selections of other workgroups with two 61.6; k=32, T=31 101.1 / 96.8).
constexpr __host__ __device__ bool split_self(int E, int K, int T) { return T <= 8 * select_tokens(E, K, T); }
constexpr int EARLY_MAX_TOKENS = 384;  // batches up to this size may take their gate/up weights before the routing is known
// Shapes whose columns do not divide into the bf16 tiled variant's tasks (256 of H, 128 of I): kernels of
// their own, which keep y as the streaming variant does (see tile_task).
constexpr __host__ __device__ bool tiled_ragged(int hidden, int intermediate) {
  return hidden % 256 != 0 || intermediate % 128 != 0;
}
// Elements from one row of h to the next in the bf16 tiled variant: whole 128-byte lines.
constexpr __host__ __device__ int tiled_h_pitch(int intermediate) { return (intermediate + 63) & ~63; }
constexpr int MAX_EXPERTS = 256;  // experts are spread 64 per wave register slot
constexpr int MAX_TOPK = 32;

// Dependency counters and the ticket dispenser, one 128-byte line each so that
// pollers of one counter do not queue behind atomics on another. Everything
// except `error` and `launches` is zero before a launch and is returned to zero
// by the last worker to leave.
struct alignas(128) ControlLine {
  unsigned v;
  unsigned pad[31];
};
struct alignas(128) LaunchLine {
  unsigned v;       // completed launches (diagnostic)
  unsigned posted;  // number the split-k kernel's last launch raised its posts to (see post_number)
  unsigned pad[30];
};
struct Control {
  ControlLine ticket;       // next task number
  ControlLine router_done;  // tokens whose routing is final
  ControlLine perm_done;    // scatter tasks finished
  ControlLine g2_done;      // down-projection tasks finished
  ControlLine exit_count;   // workers that have left the loop
  ControlLine n_mtiles;     // row tiles produced by the scan
  ControlLine error;        // sticky error bits
  LaunchLine launches;
  ControlLine xq[8];        // tiled variant: per-XCD ticket counters of the GEMM tasks
  ControlLine cticket;      // tiled variant: combine tickets
  ControlLine scan_done;    // tiled variant: per-expert scan tasks finished
};

// Phase flags, one line per workgroup: the worker that completes a phase
// writes every workgroup's copy, so waiting workers poll a line nobody else
// touches instead of queueing on one address.
// FLAG_ROUTED (streaming variant, early mode): every token's top-k entries are final.
enum : int { FLAG_SCAN = 0, FLAG_PERM = 1, FLAG_G2 = 2, FLAG_ROUTED = 3 };
struct alignas(128) WgFlags {
  unsigned f[32];
};

// Split-k kernel: a word a workgroup and hand-over, raised by the workgroup that has done its share, in every one of
// POST_COPIES rows; a workgroup watches one of those. Raised means the number of the launch, so nobody lowers it: launches
// of this kernel count from 1 (0: never raised), and behind the last number all posts return to zero.
// (POST_ROUTE: a word a routing task.)
enum : int { POST_ROUTE = 0, POST_GATE_UP = 1, POST_DOWN = 2, POST_PHASES = 3 };
constexpr int POST_COPIES = 8;
constexpr int POST_PITCH = 512;  // words of a row
constexpr __host__ __device__ unsigned post_number(unsigned posted) { return posted + 1u; }
constexpr __host__ __device__ unsigned posted_by(unsigned number) { return number == 0xFFFFFFFFu ? 0u : number; }
static_assert(post_number(posted_by(0xFFFFFFFFu)) == 1u && post_number(posted_by(0xFFFFFFFEu)) == 0xFFFFFFFFu,
              "no launch may take a post that was never raised, or one from before the count came round, for its own");

struct TileDesc {  // one row tile: `rows` consecutive permuted rows of one expert
  int expert;
  int row0;
  int rows;
  int shared;  // streaming variant: the expert has other row tiles, which read the same weights
};

// One record per executed task when tracing is on (times: 100 MHz wall clock).
struct TraceRec {
  unsigned ticket;
  unsigned kind;    // 0 router dot, 1 scan, 2 scatter, 3 gate/up, 4 down, 5 combine, 6 select or expert scan
  unsigned worker;  // streaming variant: workgroup * waves_per_group + wave; tiled one: workgroup
  unsigned aux;     // task-specific (row tile, token ...)
  long long t_fetch;  // before the ticket was drawn
  long long t_ready;  // dependencies satisfied, work starts
  long long t_end;    // work finished and signalled
  long long pad;
};

struct Params {
  int T, E, H, K, I;
  int W;          // 64-bit mask words per expert (row stride of `masks`)
  int n_workers;  // waves that take tickets (streaming variant) or items of the combine step
  int max_mtiles;
  long long spin_limit;  // bound on one dependency wait, 100 MHz ticks

  const void* tokens;  // [T,H]: what the router and the gate/up projection read (the caller's rows, or their RMSNorm)
  const void* residual;  // [T,H] rows added to the output (the caller's rows), or null
  const void* gate;    // [E,H]
  const void* ffn1;    // [E,2I,H]  rows 0..I-1 gate proj, I..2I-1 up proj
  const void* ffn2;    // [E,H,I]
  const float* bias;   // [E] or null
  // Optional re-laid-out copies of the expert weights for the streaming variant
  // (null: read the caller's layout). One gate/up or down wave task reads its
  // slice front to back: [expert][column block][k-step][weight block][lane][16 B].
  const void* ffn1_packed;
  const void* ffn2_packed;
  void* out;           // [T,H], may alias tokens

  int* topk_idx;              // [T,K]
  float* topk_w;              // [T,K]
  unsigned long long* masks;  // [E,W] bit t of word t/64: token t selected the expert
  int* word_prefix;           // [E,W] rows of the expert before word w
  int* expert_count;          // [E]
  int* expert_offset;         // [E+1]
  int* perm;                  // [T*K] permuted row -> t*K+slot
  float* row_w;               // [T*K] gate weight of the permuted row
  TileDesc* mtiles;           // [max_mtiles]
  void* h;                    // [T*K, I] SwiGLU output, layer dtype; bf16 tiled variant: rows of tiled_h_pitch(I) elements
  float* y;                   // [T*K, H] weighted down-projection rows, by t*K+slot; bf16 tiled variant, shapes that are
                              // not ragged: bf16 rows without the weight
  Control* ctl;
  WgFlags* wgflags;                // [n_groups]
  unsigned* posts;                 // [POST_PHASES][POST_COPIES][POST_PITCH]
  ControlLine* g1_done;            // [max_mtiles] gate/up tasks finished per row tile
  unsigned* cand;                  // [T,E] ordered_bits of the logits, from the chains to the selections
  unsigned* tok_arrive;            // [T] expert groups of the token whose keys are in
  int n_groups;                    // workgroups in the grid
  int fuse_scatter;                // 1: the scan task also writes the permutation
  int early;                       // 1, 2: row tile e belongs to expert e (empty or not), so gate/up tasks are
                                   //    handed out at launch and fetch their first weights under the routing
  int split;                       // 1, 2: the split-k kernel runs, on tiles of so many 16-row blocks
  int split_spec;                  //    1: its workgroups ask for gate/up weights before the routing is known
  int split_down;                  //    waves that share a down task: 4 or 8
  int dot16;                       // 1 (streaming variant, bf16): the logit chains run on the matrix core, 16 tokens x
                                   //    16 experts per workgroup, on the first workgroups before they take tickets;
                                   //    bf16 tiled variant: how it starts (see the launcher)
  // What the last worker out needs when a launch has raised an error bit: it fills `out`
  // with NaN, returns the workspace's leading zero_words 32-bit words (counters, flags,
  // masks; `ctl` is the workspace's first byte) to zero, and adds the bits to *host_error
  // (pinned host memory the host reads without waiting for the stream; may be null).
  unsigned* host_error;
  unsigned zero_words;
  int elem_bytes;     // of tokens / out: 2 or 4
  TraceRec* trace;    // null unless tracing; indexed by ticket
  unsigned trace_cap;
};

// How device code reaches the launch parameters. A kernel parameter whose address
// is passed to a function is copied to the wave's private memory first, and every
// field read in a task then goes through the vector memory pipeline, behind the
// weight loads. A kernel that defines FMOE_PARAMS_IN_KERNARG before including
// this header reads them in place in the kernel-argument segment instead
// (constant address space): a field costs a scalar load that the scalar cache
// serves. Both kernels do.
#if defined(__HIP_DEVICE_COMPILE__) && defined(FMOE_PARAMS_IN_KERNARG)
typedef const __attribute__((address_space(4))) Params& ParamsRef;
#else
typedef const Params& ParamsRef;
#endif

}  // namespace fmoe
