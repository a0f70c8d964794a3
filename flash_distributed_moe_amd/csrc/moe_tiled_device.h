// What the tiled kernels of both dtypes share: workgroup-wide waits and arrivals, the scan and
// scatter tasks, the XCD a workgroup runs on. Workgroups of 256 threads.
#pragma once
#ifndef FMOE_PARAMS_IN_KERNARG
#define FMOE_PARAMS_IN_KERNARG 1
#endif
#include "moe_device.h"

namespace fmoe {

constexpr int T_THREADS = 256;
constexpr int RT_TOK = 32;         // tokens per scatter task

// ---------------------------------------------------------- workgroup helpers
// Values that are the same in every lane but that the compiler cannot prove so
// (they come through a struct reference): pin them to scalar registers, so
// loops and branches on them stay scalar.
__device__ __forceinline__ int uni(int v) { return __builtin_amdgcn_readfirstlane(v); }
template <typename T>
__device__ __forceinline__ T* uni(T* ptr) {
  const unsigned long long v = reinterpret_cast<unsigned long long>(ptr);
  const unsigned lo = __builtin_amdgcn_readfirstlane(static_cast<unsigned>(v));
  const unsigned hi = __builtin_amdgcn_readfirstlane(static_cast<unsigned>(v >> 32));
  return reinterpret_cast<T*>((static_cast<unsigned long long>(hi) << 32) | lo);
}

struct WgShared {  // small static LDS block
  unsigned ticket;
  unsigned next;
  unsigned ok;
  unsigned flag[4];
};

// Thread 0 waits (bounded) for *p >= target; every thread learns the outcome.
__device__ __forceinline__ bool wg_wait_ge(ParamsRef p, const unsigned* ptr, unsigned target,
                                           WgShared* sh) {
  if (threadIdx.x == 0) {
    unsigned ok = 1u;
    if (ld_relaxed(ptr) < target) {
      const long long t0 = wall_clock64();
      unsigned spins = 0;
      while (ld_relaxed(ptr) < target) {
        if ((++spins & 31u) == 0u && ld_relaxed(&p.ctl->error.v) != 0u) {
          ok = 0u;
          break;
        }
        if (wall_clock64() - t0 > p.spin_limit) {
          or_relaxed(&p.ctl->error.v, ERR_TIMEOUT);
          ok = 0u;
          break;
        }
        __builtin_amdgcn_s_sleep(16);
      }
    }
    sh->ok = ok;
  }
  __syncthreads();
  const bool ok = sh->ok != 0u;
  __syncthreads();
  fence_acquire();
  return ok;
}

__device__ __forceinline__ bool wg_wait_flag(ParamsRef p, int which, WgShared* sh) {
  if (sh->flag[which] != 0u) return true;  // seen before by this workgroup
  const bool ok = wg_wait_ge(p, &p.wgflags[blockIdx.x].f[which], 1u, sh);
  if (ok && threadIdx.x == 0) sh->flag[which] = 1u;
  __syncthreads();
  return ok;
}

// A task's record, written by the lanes where `writes` holds: one, and only while tracing is on.
__device__ __forceinline__ void trace_task(ParamsRef p, bool writes, unsigned id, unsigned kind, unsigned aux,
                                           long long t_fetch, long long t_ready) {
  if (writes && id < p.trace_cap) {
    const long long t_end = wall_clock64();
    TraceRec* r = p.trace + id;
    st16(r, u32x4{id, kind, blockIdx.x, aux});
    st16(reinterpret_cast<char*>(r) + 16,
         u32x4{static_cast<unsigned>(t_fetch), static_cast<unsigned>(t_fetch >> 32),
               static_cast<unsigned>(t_ready), static_cast<unsigned>(t_ready >> 32)});
    st16(reinterpret_cast<char*>(r) + 32,
         u32x4{static_cast<unsigned>(t_end), static_cast<unsigned>(t_end >> 32), 0u, 0u});
  }
}
__device__ __forceinline__ long long trace_clock(bool traced) { return traced ? wall_clock64() : 0; }

// All threads' stores have completed, then one thread bumps the counter. Tile
// data (h, y) is written through to device-coherent memory, so completion is
// all a reader on another XCD needs (WRITEBACK adds an agent-scope release for
// data written with ordinary cached stores; no task does that at present).
// Readers of h and y use ordinary loads: every cache line of them has a single
// writer and is not read before it is final, so no reader can hold a stale copy.
template <bool WRITEBACK>
__device__ __forceinline__ unsigned wg_arrive(unsigned* counter, WgShared* sh) {
  fence_release();
  __syncthreads();
  if (threadIdx.x == 0) {
    if (WRITEBACK) __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
    sh->ticket = add_relaxed(counter, 1u);
  }
  __syncthreads();
  const unsigned old = sh->ticket;
  __syncthreads();
  return old;
}

__device__ __forceinline__ void wg_broadcast_flag(ParamsRef p, int which) {
  const int n = p.n_groups;
  WgFlags* flags = p.wgflags;
  for (int g = threadIdx.x; g < n; g += blockDim.x) st_relaxed(&flags[g].f[which], 1u);
}

// ----------------------------------------------------------------------- scan
// Same tables as the streaming variant's scan, in two steps. Expert scan: one
// wave per expert walks the expert's mask words 64 at a time and writes the
// running count in front of every word (word_prefix) and the expert's total.
// Final scan: one wave turns the totals into row offsets and the row-tile table
// (an expert's rows in as few tiles of at most TM rows as possible, of equal size).
constexpr int SCAN_EXPERTS = T_THREADS / 64;  // experts per expert-scan task

__device__ __noinline__ void tiled_expert_scan_task(ParamsRef pv, int blk) {
  ParamsRef p = uniform_params(pv);
  const int E = uni(p.E), W = uni(p.W), T = uni(p.T);
  const unsigned long long* masks = uni(p.masks);
  int* word_prefix = uni(p.word_prefix);
  int* expert_count = uni(p.expert_count);
  const int lane = threadIdx.x & 63;
  const int e = uni(blk) * SCAN_EXPERTS + uni(threadIdx.x >> 6);
  if (e >= E) return;
  const int wact = (T + 63) >> 6;
  int base = 0;
  for (int w0 = 0; w0 < wact; w0 += 64) {
    const int w = w0 + lane;
    const int c = w < wact ? __popcll(ldc(&masks[static_cast<size_t>(e) * W + w])) : 0;
    const int incl = wave_inclusive_scan(c);
    if (w < wact) stc(&word_prefix[static_cast<size_t>(e) * W + w], base + incl - c);
    base += __shfl(incl, 63, 64);
  }
  if (lane == 0) stc(&expert_count[e], base);
}

// Expert e's c rows, from permuted row `off` on, as balanced tiles of at most TM rows, whole blocks of
// BLK rows. Called by a whole wave, lanes in expert order; returns the number of tiles so far.
template <int TM, int BLK>
__device__ __forceinline__ int scan_tiles(const RouteTables& r, int e, int c, int off, int tile_base) {
  const int nt = (c + TM - 1) / TM;
  const int per = nt > 0 ? ((c + nt - 1) / nt + BLK - 1) / BLK * BLK : 0;
  const int tincl = wave_inclusive_scan(nt);
  const int toff = tile_base + tincl - nt;
  if (e < r.E) {
    stc(&r.expert_offset[e], off);
    int done = 0;
    for (int i = 0; i < nt; ++i) {
      const int tr = min(per, c - done);
      if (toff + i < r.max_mtiles) {
        stc16(&r.mtiles[toff + i],
              make_uint4(static_cast<unsigned>(e), static_cast<unsigned>(off + done), static_cast<unsigned>(tr),
                         nt > 1 ? 1u : 0u));
      }
      done += tr;
    }
  }
  return tile_base + __shfl(tincl, 63, 64);
}
// the totals behind it: rows of all experts and tiles
__device__ __forceinline__ void scan_totals(ParamsRef p, const RouteTables& r, int lane, int rows, int tiles) {
  if (lane == 0) {
    stc(&r.expert_offset[r.E], rows);
    if (tiles > r.max_mtiles) {
      or_relaxed(&p.ctl->error.v, ERR_CAPACITY);
      tiles = 0;
    }
    stc(&p.ctl->n_mtiles.v, static_cast<unsigned>(tiles));
  }
}

template <int TM, int BLK>
__device__ __noinline__ void tiled_scan_task(ParamsRef pv) {
  ParamsRef p = uniform_params(pv);
  const RouteTables r = route_tables(p);
  const int tid = threadIdx.x;
  if (tid < 64) {
    const int lane = tid;
    const int epl = (r.E + 63) >> 6;
    int base = 0, tile_base = 0;
    for (int j = 0; j < epl; ++j) {
      const int e = lane + 64 * j;
      const int c = e < r.E ? ldc(&r.expert_count[e]) : 0;
      const int incl = wave_inclusive_scan(c);
      tile_base = scan_tiles<TM, BLK>(r, e, c, base + incl - c, tile_base);
      base += __shfl(incl, 63, 64);
    }
    scan_totals(p, r, lane, base, tile_base);
  }
  fence_release();
  __syncthreads();
  wg_broadcast_flag(p, FLAG_SCAN);
}

__device__ void tiled_scatter_task(ParamsRef p, int blk) {
  const RouteTables r = route_tables(p);
  const int i0 = blk * RT_TOK * r.K;
  const int n = min(RT_TOK * r.K, r.T * r.K - i0);
  for (int i = threadIdx.x; i < n; i += T_THREADS) scatter_entry(r, i0 + i);
}

__device__ __forceinline__ int xcc_id() {
  // HW_REG_XCC_ID (20), bits 0..3
  return __builtin_amdgcn_s_getreg((3 << 11) | (0 << 6) | 20) & 7;
}


}  // namespace fmoe
