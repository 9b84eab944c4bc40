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
#include "mc_walk.h"

namespace {

template <bool SCORE> struct bank_io {
  const mc_transport_args &a;
  double score;
  static constexpr bool RESUMES = false;
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

template <bool LDS_TALLY, bool LDS_CELLS, bool SCORE>
__global__ __launch_bounds__(1024) void k_history(mc_transport_args a, int refill_k,
                                                   int per_cu) {
  extern __shared__ __align__(16) unsigned char smem[];
  __shared__ int s_k;
  __shared__ unsigned long long s_tot[MC_TOTALS];
  const mc_walk_k K = mc_walk_live(a.L);
  mc_call_queue queue{mc_queue_open(a.n, per_cu), &a.ctr->next};
  const int m = a.L.m;
  double2 *tab = reinterpret_cast<double2 *>(smem);
  mc_tab_fill(tab);
  unsigned long long *t0 = reinterpret_cast<unsigned long long *>(smem + MC_TAB_BYTES), *t1 = t0 + m;
  if (LDS_TALLY) {
    for (int c = threadIdx.x; c < m; c += blockDim.x) {
      t0[c] = 0;
      t1[c] = 0;
    }
  }
  const mc_cell *cells = a.cells;
  const double *g = a.g;
  if (LDS_CELLS) {
    mc_cell *lc = reinterpret_cast<mc_cell *>(smem + MC_TAB_BYTES + (size_t)16 * m);
    for (int c = threadIdx.x; c < m; c += blockDim.x) lc[c] = a.cells[c];
    cells = lc;
    if (SCORE) {
      double *lg = reinterpret_cast<double *>(smem + MC_TAB_BYTES + (size_t)32 * m);
      for (int c = threadIdx.x; c < m; c += blockDim.x) lg[c] = a.g[c];
      g = lg;
    }
  }
  if (threadIdx.x < MC_TOTALS) s_tot[threadIdx.x] = 0;
  /* the block's weights: the largest among the first histories of its waves
     (a guess that sets the limbs' range; heavier ones go to the global tally) */
  if (threadIdx.x == 0) s_k = -1023;
  __syncthreads();
  if (LDS_TALLY) {
    const uint64_t i = queue.q.next + __lane_id();
    if (i < queue.q.end) atomicMax(&s_k, mc_ceil_log2(a.aos ? a.aos[i].wmc : a.soa.wmc[i]));
    __syncthreads();
  }

  bank_io<SCORE> io{a, 0.0};
  unsigned long long *fx_lo = a.fx, *fx_hi = a.fx + m;
  uint32_t *flags = a.flags;
  unsigned int *status = &a.ctr->status;
  const mc_block_tally B =
      mc_block_tally_for(m, __builtin_amdgcn_readfirstlane(s_k), blockDim.x >> 6);
  if (LDS_TALLY && B.limbs) { /* block-uniform */
    mc_walk_bank(io, queue, a.L, K, cells, tab, refill_k, B.every, a.max_events, s_tot,
                 [&](mc_mask lanes, int c, const mc_cell &, bool, double, double dw, double) {
                   mc_tally_limbs(t0, t1, B.S, fx_lo, fx_hi, flags, status, lanes, c, dw);
                   if (SCORE && mc_in(lanes)) io.score = io.score + g[c] * dw;
                 },
                 mc_mover{t0, t1, fx_lo, fx_hi, m, B.S.L, B.every, B.every});
    __syncthreads();
    mc_limbs_move(t0, t1, B.S.L, m, threadIdx.x, blockDim.x, fx_lo, fx_hi);
  } else {
    unsigned long long *lo = LDS_TALLY ? t0 : fx_lo, *hi = LDS_TALLY ? t1 : fx_hi;
    mc_walk_bank(io, queue, a.L, K, cells, tab, refill_k, 1 << 30, a.max_events, s_tot,
                 [&](mc_mask lanes, int c, const mc_cell &, bool, double, double dw, double) {
                   if (mc_in(lanes)) {
                     mc_tally(lo, hi, flags, status, c, dw);
                     if (SCORE) io.score = io.score + g[c] * dw;
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

} // namespace

int mc_launch_history(mcgpu_context *ctx, const mc_transport_args &a, const mcgpu_options &o,
                      hipStream_t s) {
  const size_t m = (size_t)a.L.m;
  const size_t tally = 16 * m + MC_TAB_BYTES, cells = sizeof(mc_cell) * m;
  const size_t budget = ctx->lds_per_block - 256; /* the kernel's static LDS */
  const bool lds_tally = tally <= budget;
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
