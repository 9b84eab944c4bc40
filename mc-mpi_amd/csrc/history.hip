/*
 * history.hip -- history-based transport kernel.
 *
 * One history per lane, run to termination with the loop condition of
 * Layer::simulate_particle (src/layer.cpp:195-200) around the event of
 * Layer::particle_step (src/layer.cpp:123-190).  Unlike the reference CUDA
 * kernel (src/culayer_kernel.cu:19-113: one launch per 325 steps, host
 * round trips and re-sorting between launches), the grid is persistent:
 * lanes whose histories end take new ones from the wave's run of the work
 * queue (mc_queue), so lanes stay busy until the queue is empty and there is
 * one launch per call.
 *
 * The event itself is mc_walk_many (mc_walk.h): a short common step with the
 * general event apart.
 *
 * Tallies: each block accumulates the exact fixed-point tally of its cells
 * in LDS (two 64-bit limbs per cell that never carry into each other,
 * mc_fx_split; for weights too large for them, two words with carry) and adds
 * it to the global 128-bit tally at the end, and before limbs could overflow.
 * Integer sums are exact, so the result is independent of which lane, wave or
 * block handled which history.  For layers too large for LDS the adds go to
 * the global (L2-resident) tally.  The per-cell cross-section pairs are staged
 * in LDS when they fit next to the tally, otherwise read through L2.
 *
 * Measured against the kernel with mc_event and a tally with carry: a lone
 * history 450 -> 284 ns per event (10,000 cells); 1,000 histories on the
 * 100-cell slab, whole call 264 -> 181 us; 1,000 on 10,000 cells 26.0 -> 9.8
 * ms (dealt over the CUs); 8e6 on 10,000 cells 267 -> 237 ms, there bound by
 * the cells' L2 reads (37 lines per wave and event).
 */
#include "internal.h"
#include <algorithm>

#include "mc_walk.h"

namespace {

template <bool SCORE> struct bank_io {
  const mc_transport_args &a;
  double score;
  static constexpr bool RESUMES = false;
  __device__ __forceinline__ int code(const mc_state &p, bool at_cap, const mc_layer_k &L) {
    return mc_end_code(p, at_cap, L);
  }
  __device__ __forceinline__ uint64_t load(int64_t i, mc_state &p) {
    load_state(a, i, p);
    score = 0.0;
    return 0;
  }
  __device__ __forceinline__ bool store(int64_t i, mc_state &p, int code, uint64_t ev,
                                        uint32_t col) {
    store_state(a, i, p, code);
    if (a.events) a.events[i] = ev;
    if (a.collisions) a.collisions[i] = col;
    if (SCORE) a.score[i] = score;
    return false;
  }
};

/* ------------------------------------------------------------- wide layers
   A layer of more cells than a block's LDS tally holds is cut into windows.
   A sweep transports the histories of every window, each block one window's;
   a history that crosses into another window is parked there for the next
   sweep, until none is left.  A history crosses a window's edge a few times at
   most (windows are thousands of cells, flights a good part of the layer), so
   parking costs little, where a global tally costs two returning atomics in
   memory per event: 200,000 histories on 20,000 cells 540 -> 118 ms. */
constexpr int MC_MAX_WINDOWS = 64;

struct mc_windows {
  int32_t nw, W;            /* window w: cells [w W, (w + 1) W) of the layer */
  uint32_t *count;          /* [nw] histories of this sweep */
  unsigned long long *next; /* [nw] queue counters */
  const uint32_t *list;     /* histories, by window */
  int32_t *win;             /* [n] a history's window, -1 when finished */
  uint64_t *ev;             /* [n] its events so far */
};

/* windows of a sweep and the blocks they get: one each, the rest by count */
struct mc_window_share {
  int32_t w;
  uint32_t block, blocks, first; /* index and number of blocks; list offset */
};

__device__ __forceinline__ mc_window_share mc_window_of(const mc_windows &win) {
  uint64_t total = 0;
  uint32_t busy = 0;
  for (int w = 0; w < win.nw; ++w) {
    total += win.count[w];
    busy += win.count[w] != 0;
  }
  mc_window_share s{-1, 0, 0, 0};
  uint32_t at = 0, first = 0;
  for (int w = 0; w < win.nw; ++w) {
    const uint32_t c = win.count[w];
    const uint32_t share = c ? 1u + (uint32_t)((uint64_t)c * (gridDim.x - busy) / total) : 0u;
    if (s.w < 0 && blockIdx.x < at + share) s = {w, blockIdx.x - at, share, first};
    at += share;
    first += c;
  }
  return s;
}

template <bool SCORE> struct window_io {
  static constexpr bool RESUMES = true;
  const mc_transport_args &a;
  const mc_windows &win;
  const uint32_t *list;
  double score;
  int64_t j;
  int to; /* window a history is parked in, -1: finished */
  __device__ __forceinline__ uint64_t load(int64_t i, mc_state &p) {
    j = list[i];
    load_state(a, j, p);
    if (SCORE) score = a.score[j];
    return win.ev[j];
  }
  __device__ __forceinline__ int code(const mc_state &p, bool at_cap, const mc_layer_k &) {
    to = mc_alive(p, a.L) && !at_cap ? (p.index - a.L.index_start) / win.W : -1;
    return to >= 0 ? 3 : mc_end_code(p, at_cap, a.L);
  }
  __device__ __forceinline__ bool store(int64_t, mc_state &p, int code, uint64_t ev, uint32_t col) {
    store_state(a, j, p, code);
    win.ev[j] = ev;
    win.win[j] = to;
    if (a.events) a.events[j] = ev;
    if (a.collisions) a.collisions[j] += col;
    if (SCORE) a.score[j] = score;
    return false;
  }
};

__global__ void k_windows_clear(mc_windows win, uint32_t *cursor) {
  const int t = threadIdx.x;
  if (t >= win.nw) return;
  win.count[t] = 0;
  cursor[t] = 0;
  win.next[t] = 0;
}

/* the histories of each window; OPEN: their first windows, from the bank */
template <bool OPEN> __global__ void k_windows_count(mc_transport_args a, mc_windows win) {
  __shared__ uint32_t s_n[MC_MAX_WINDOWS];
  if (threadIdx.x < MC_MAX_WINDOWS) s_n[threadIdx.x] = 0;
  __syncthreads();
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < a.n;
       i += (int64_t)gridDim.x * blockDim.x) {
    int w;
    if (OPEN) {
      mc_state p;
      load_state(a, i, p);
      const uint32_t c = (uint32_t)p.index - (uint32_t)a.L.index_start;
      w = c < (uint32_t)a.L.m ? (int)(c / (uint32_t)win.W) : 0;
      win.win[i] = w;
      win.ev[i] = 0;
      if (a.collisions) a.collisions[i] = 0;
      if (a.score) a.score[i] = 0.0;
    } else {
      w = win.win[i];
    }
    if (w >= 0) atomicAdd(&s_n[w], 1u);
  }
  __syncthreads();
  if (threadIdx.x < (unsigned)win.nw && s_n[threadIdx.x])
    atomicAdd(&win.count[threadIdx.x], s_n[threadIdx.x]);
}

/* the histories of each window one after the other (cursors zeroed) */
__global__ void k_windows_list(int64_t n, mc_windows win, uint32_t *list, uint32_t *cursor) {
  __shared__ uint32_t s_n[MC_MAX_WINDOWS], s_at[MC_MAX_WINDOWS];
  const int t = threadIdx.x;
  for (int64_t base = (int64_t)blockIdx.x * blockDim.x; base < n;
       base += (int64_t)gridDim.x * blockDim.x) { /* block-uniform */
    if (t < MC_MAX_WINDOWS) s_n[t] = 0;
    __syncthreads();
    const int64_t i = base + t;
    const int w = i < n ? win.win[i] : -1;
    uint32_t r = 0;
    if (w >= 0) r = atomicAdd(&s_n[w], 1u);
    __syncthreads();
    if (t < win.nw && s_n[t]) {
      uint32_t first = 0;
      for (int v = 0; v < t; ++v) first += win.count[v];
      s_at[t] = first + atomicAdd(&cursor[t], s_n[t]);
    }
    __syncthreads();
    if (w >= 0) list[s_at[w] + r] = (uint32_t)i;
    __syncthreads();
  }
}

/* one block's part of layer L (cells and global tally words at cells, fx_lo,
   fx_hi, ...): LDS, the walk, the tally and totals */
template <bool LDS_TALLY, bool LDS_CELLS, bool SCORE, typename IO>
__device__ __forceinline__ void history_block(const mc_transport_args &a, const mc_layer_k &L,
                                              int off, IO &io, mc_call_queue &queue, double wmc,
                                              int refill_k) {
  extern __shared__ __align__(16) unsigned char smem[];
  __shared__ int s_k;
  __shared__ unsigned long long s_tot[MC_TOTALS];
  const mc_walk_k K = mc_walk_live(L);
  const int m = L.m;
  double2 *tab = reinterpret_cast<double2 *>(smem);
  mc_tab_fill(tab);
  unsigned long long *t0 = reinterpret_cast<unsigned long long *>(smem + MC_TAB_BYTES), *t1 = t0 + m;
  if (LDS_TALLY) {
    for (int c = threadIdx.x; c < m; c += blockDim.x) {
      t0[c] = 0;
      t1[c] = 0;
    }
  }
  const mc_cell *cells = a.cells + off;
  const double *g = SCORE ? a.g + off : nullptr;
  if (LDS_CELLS) {
    mc_cell *lc = reinterpret_cast<mc_cell *>(t1 + m);
    cells = mc_cells_fill(lc, cells, m);
    if (SCORE) {
      double *lg = reinterpret_cast<double *>(lc + m + 2);
      for (int c = threadIdx.x; c < m; c += blockDim.x) lg[c] = g[c];
      g = lg;
    }
  }
  if (threadIdx.x < MC_TOTALS) s_tot[threadIdx.x] = 0;
  /* the block's weights: the largest among the first histories of its waves
     (a guess that sets the limbs' range; heavier ones go to the global tally) */
  if (threadIdx.x == 0) s_k = -1023;
  __syncthreads();
  if (LDS_TALLY) {
    atomicMax(&s_k, mc_ceil_log2(wmc));
    __syncthreads();
  }

  unsigned long long *fx_lo = a.fx + off, *fx_hi = fx_lo + a.L.m;
  uint32_t *flags = a.flags + off;
  unsigned int *status = &a.ctr->status;
  const mc_block_tally B =
      mc_block_tally_for(m, __builtin_amdgcn_readfirstlane(s_k), blockDim.x >> 6);
  if (LDS_TALLY && B.limbs) { /* block-uniform */
    mc_walk_bank<LDS_CELLS>(io, queue, L, K, cells, tab, refill_k, B.every, a.max_events, s_tot,
                 [&](mc_mask lanes, int c8, const mc_cell &, bool, double, double dw, double) {
                   mc_tally_limbs(t0, t1, B.S, fx_lo, fx_hi, flags, status, lanes, c8, dw);
                   if (SCORE && mc_in(lanes)) io.score = io.score + *mc_word(g, c8) * dw;
                 },
                 mc_mover{t0, t1, fx_lo, fx_hi, m, B.S.L, B.every, B.every});
    __syncthreads();
    mc_limbs_move(t0, t1, B.S.L, m, threadIdx.x, blockDim.x, fx_lo, fx_hi);
  } else {
    unsigned long long *lo = LDS_TALLY ? t0 : fx_lo, *hi = LDS_TALLY ? t1 : fx_hi;
    mc_walk_bank<LDS_CELLS>(io, queue, L, K, cells, tab, refill_k, 1 << 30, a.max_events, s_tot,
                 [&](mc_mask lanes, int c8, const mc_cell &, bool, double, double dw, double) {
                   if (mc_in(lanes)) {
                     mc_tally(lo, hi, flags, status, c8 >> 3, dw);
                     if (SCORE) io.score = io.score + *mc_word(g, c8) * dw;
                   }
                 },
                 [](int) {});
    __syncthreads();
    if (LDS_TALLY) {
      for (int c = threadIdx.x; c < m; c += blockDim.x) {
        mc_fx v;
        v.lo = t0[c];
        v.hi = t1[c];
        mc_fx_atomic_add(&fx_lo[c], &fx_hi[c], v);
      }
    }
  }
  if (threadIdx.x == 0) mc_totals_out(s_tot, a.ctr);
}

template <bool LDS_TALLY, bool LDS_CELLS, bool SCORE>
__global__ __launch_bounds__(1024) void k_history(mc_transport_args a, int refill_k, int per_cu) {
  mc_call_queue queue{mc_queue_open(a.n, per_cu, blockIdx.x, gridDim.x), &a.ctr->next};
  bank_io<SCORE> io{a, 0.0};
  const uint64_t i = queue.q.next + __lane_id();
  double wmc = 0.0;
  if (LDS_TALLY && i < queue.q.end) wmc = a.aos ? a.aos[i].wmc : a.soa.wmc[i];
  history_block<LDS_TALLY, LDS_CELLS, SCORE>(a, a.L, 0, io, queue, wmc, refill_k);
}

/* one sweep over the windows of a wide layer */
template <bool SCORE>
__global__ __launch_bounds__(1024) void k_history_windows(mc_transport_args a, mc_windows win,
                                                          int refill_k, int per_cu) {
  const mc_window_share sh = mc_window_of(win);
  if (sh.w < 0) return; /* block-uniform: no window left for this block */
  const int w = __builtin_amdgcn_readfirstlane(sh.w), off = w * win.W;
  mc_layer_k L = a.L;
  L.index_start += off;
  L.m = a.L.m - off < win.W ? a.L.m - off : win.W;
  mc_call_queue queue{mc_queue_open(win.count[w], per_cu, sh.block, sh.blocks), &win.next[w]};
  window_io<SCORE> io{a, win, win.list + sh.first, 0.0, 0, -1};
  const uint64_t i = queue.q.next + __lane_id();
  double wmc = 0.0;
  if (i < queue.q.end) wmc = a.aos ? a.aos[io.list[i]].wmc : a.soa.wmc[io.list[i]];
  history_block<true, false, SCORE>(a, L, off, io, queue, wmc, refill_k);
}

template <bool T, bool C, bool S>
int launch_one(mcgpu_context *ctx, const mc_transport_args &a, const mcgpu_options &o,
               hipStream_t s, size_t lds) {
  auto kern = k_history<T, C, S>;
  if (lds > 65536)
    (void)hipFuncSetAttribute(reinterpret_cast<const void *>(kern),
                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  int per_cu = 0;
  int block = o.block_size;
  if (block <= 0) {
    block = mc_auto_block(kern, lds, &per_cu);
  } else if (block > 1024 || block % 64) {
    return mc_fail(ctx, MCGPU_ERR_ARG, "block_size must be a multiple of 64 and <= 1024");
  } else if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kern, block, lds) !=
                 hipSuccess || per_cu < 1) {
    per_cu = 1;
  }
  int grid = o.grid_blocks;
  if (grid <= 0) {
    grid = per_cu * ctx->num_cus;
    if (a.n < grid) grid = (int)(a.n > 0 ? a.n : 1); /* a block per history at most */
  }
  int k = o.events_per_refill > 0 ? o.events_per_refill : 0; /* 0: adaptive */
  hipLaunchKernelGGL(kern, dim3(grid), dim3(block), lds, s, a, k, per_cu);
  MC_HIP(ctx, hipGetLastError());
  return MCGPU_OK;
}

/* Sweeps over a wide layer's windows until no history is parked.  Scratch (16
   bytes per history) from the context; MCGPU_ERR_NOMEM: there is none. */
template <bool S>
int launch_windows(mcgpu_context *ctx, const mc_transport_args &a, const mcgpu_options &o,
                   hipStream_t s, int nw, int W) {
  auto kern = k_history_windows<S>;
  const size_t lds = MC_TAB_BYTES + 16 * (size_t)W;
  if (lds > 65536)
    (void)hipFuncSetAttribute(reinterpret_cast<const void *>(kern),
                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  int per_cu = 0;
  int block = o.block_size;
  if (block <= 0)
    block = mc_auto_block(kern, lds, &per_cu);
  else if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kern, block, lds) != hipSuccess ||
           per_cu < 1)
    per_cu = 1;
  const int grid = o.grid_blocks > 0 ? o.grid_blocks : per_cu * ctx->num_cus;
  const int k = o.events_per_refill > 0 ? o.events_per_refill : 0;

  /* ev[n], win[n], list[n], queue counters, counts, cursors */
  const size_t n = (size_t)a.n, words = (16 * n + 255) / 256 * 256;
  int rc = mc_ensure(ctx, &ctx->work, &ctx->work_bytes, words + 16 * MC_MAX_WINDOWS);
  if (rc) return rc;
  unsigned char *base = (unsigned char *)ctx->work;
  mc_windows win;
  win.nw = nw;
  win.W = W;
  win.ev = (uint64_t *)base;
  win.win = (int32_t *)(base + 8 * n);
  uint32_t *list = (uint32_t *)(base + 12 * n);
  win.list = list;
  win.next = (unsigned long long *)(base + words);
  win.count = (uint32_t *)(win.next + MC_MAX_WINDOWS);
  uint32_t *cursor = win.count + MC_MAX_WINDOWS;
  uint32_t host[MC_MAX_WINDOWS];
  const unsigned blocks = (unsigned)std::min<size_t>((n + 1023) / 1024, 4 * (size_t)ctx->num_cus);

  for (bool first = true;; first = false) {
    hipLaunchKernelGGL(k_windows_clear, dim3(1), dim3(64), 0, s, win, cursor);
    MC_HIP(ctx, hipGetLastError());
    if (first)
      hipLaunchKernelGGL(k_windows_count<true>, dim3(blocks), dim3(1024), 0, s, a, win);
    else
      hipLaunchKernelGGL(k_windows_count<false>, dim3(blocks), dim3(1024), 0, s, a, win);
    MC_HIP(ctx, hipGetLastError());
    if (!first) { /* the first sweep's histories are all of them */
      MC_HIP(ctx, hipMemcpyAsync(host, win.count, 4 * (size_t)nw, hipMemcpyDeviceToHost, s));
      MC_HIP(ctx, hipStreamSynchronize(s));
      uint64_t left = 0;
      for (int w = 0; w < nw; ++w) left += host[w];
      if (left == 0) return MCGPU_OK;
    }
    hipLaunchKernelGGL(k_windows_list, dim3(blocks), dim3(1024), 0, s, a.n, win, list, cursor);
    MC_HIP(ctx, hipGetLastError());
    hipLaunchKernelGGL(kern, dim3(grid), dim3(block), lds, s, a, win, k, per_cu);
    MC_HIP(ctx, hipGetLastError());
  }
}

} // namespace

int mc_launch_history(mcgpu_context *ctx, const mc_transport_args &a, const mcgpu_options &o,
                      hipStream_t s) {
  const size_t m = (size_t)a.L.m;
  const size_t tally = 16 * m + MC_TAB_BYTES, cells = sizeof(mc_cell) * m + MC_PAD_BYTES;
  const size_t budget = ctx->lds_per_block - 256; /* the kernel's static LDS */
  const bool lds_tally = tally <= budget;
  /* wide layers: equal windows that fill the LDS; with scratch for them (not
     in the no-allocation entry point, whose context is quiet) and at least a
     block per window.  Else the global tally. */
  const size_t most = (budget - MC_TAB_BYTES) / 16, nw = (m + most - 1) / most;
  const bool block_ok = o.block_size <= 1024 && o.block_size % 64 == 0;
  if (!lds_tally && !ctx->quiet && nw <= MC_MAX_WINDOWS && a.n < (int64_t)0xFFFFFFFFu &&
      block_ok && (o.grid_blocks <= 0 || (size_t)o.grid_blocks >= nw) && !(a.score && !a.g)) {
    const int W = (int)((m + nw - 1) / nw);
    const int rc = a.score ? launch_windows<true>(ctx, a, o, s, (int)nw, W)
                           : launch_windows<false>(ctx, a, o, s, (int)nw, W);
    if (rc != MCGPU_ERR_NOMEM) return rc;
    ctx->err.clear();
  }
  if (a.score) { /* per-history score of a weighted tally (forward of the adjoint) */
    if (!a.g) return mc_fail(ctx, MCGPU_ERR_ARG, "score output needs target weights g");
    const size_t extra = 8 * m;
    const bool lds_cells = lds_tally && tally + cells + extra <= budget;
    if (lds_tally && lds_cells) return launch_one<true, true, true>(ctx, a, o, s, tally + cells + extra);
    if (lds_tally) return launch_one<true, false, true>(ctx, a, o, s, tally);
    return launch_one<false, false, true>(ctx, a, o, s, MC_TAB_BYTES);
  }
  const bool lds_cells = lds_tally && tally + cells <= budget;
  if (lds_tally && lds_cells) return launch_one<true, true, false>(ctx, a, o, s, tally + cells);
  if (lds_tally) return launch_one<true, false, false>(ctx, a, o, s, tally);
  return launch_one<false, false, false>(ctx, a, o, s, MC_TAB_BYTES);
}
