/*
 * adjoint.hip -- gradient of a weighted tally by history replay.
 *
 * Target: T = sum_c g_c * tally_c, where tally_c is the absorbed weight of
 * cell c (src/layer.cpp:174-179).  Parameters: the per-cell cross sections
 * the step uses, sig_a_c and sig_i_c (src/layer.cpp:131-133).
 *
 * The forward pass (history kernel with target weights) stores, per history,
 * T_h = sum_j g_{c_j} dw_j.  The adjoint kernel replays every history from
 * its initial particle -- the particle's seed is its RNG state, so the replay
 * recomputes the path instead of storing it -- and for each event j (cell
 * c, flight length d_j, weight w_{j+1} after the event, collision flag,
 * P_j = sum_{k<j} g_{c_k} dw_k) adds
 *   pathwise, sig_a:      d_j * (g_c * w_{j+1} - (T_h - P_j - g_c * dw_j))
 *   score function, sig_i: ([collision] / sig_i - d_j) * (T_h - P_j)
 *                          (only where sig_i > EPS_PRECISION: there the flight
 *                          length is sampled with density sig_i e^{-sig_i d})
 * to two exact fixed-point per-cell tallies (same arithmetic as the absorbed
 * weight tally).  The kill at the minimum weight is not differentiated.
 * When T_h was not stored, each lane first replays the history once to
 * compute it, then replays it again for the gradient.
 *
 * Two adds in LDS for each of the two terms bound the adjoint, and the longest
 * histories, some five times the mean, end a run of few histories per lane.
 * 1,000 cells, 1 M histories: adjoint 11.3 -> 5.8 ms, forward with scores 6.8
 * -> 4.5 ms.
 */
#include "mc_adjoint.h"

namespace {

struct adj_args {
  mc_layer_k L;
  int64_t n;
  mcgpu_bank init; /* read only */
  const mc_cell *cells;
  const double *g;
  const double *score; /* may be null */
  unsigned long long *fx; /* ga lo [0,m), ga hi [m,2m), gi lo [2m,3m), gi hi [3m,4m) */
  uint32_t *flags;        /* ga flags [0,m), gi flags [m,2m) */
  mc_counters *ctr;
  uint64_t max_events;
};

/* the block's totals: this call counts events alone */
__device__ __forceinline__ void events_out(unsigned long long *s_tot, mc_counters *ctr) {
  if (threadIdx.x != 0) return;
  s_tot[1] = s_tot[2] = s_tot[3] = s_tot[4] = 0;
  mc_totals_out(s_tot, ctr, mc_counter_copy());
}

/* LDS_T: the two limb tallies in LDS; LDS_C: the cells and target weights too */
template <bool LDS_T, bool LDS_C, bool HAVE_SCORE>
__global__ __launch_bounds__(1024) void k_adjoint(adj_args a, int refill_k, int per_cu) {
  extern __shared__ __align__(16) unsigned char smem[];
  __shared__ mc_scale s_scale;
  __shared__ uint32_t s_thick;
  __shared__ unsigned long long s_tot[MC_TOTALS];
  constexpr int U = LDS_T ? MC_IN_LDS : MC_IN_MEMORY;
  mc_call_queue queue{mc_queue_open(a.n, per_cu, blockIdx.x, gridDim.x), &a.ctr->next};
  const int m = a.L.m;
  double2 *tab = reinterpret_cast<double2 *>(smem);
  mc_tab_fill(tab);
  mc_grad_tally G;
  G.t = reinterpret_cast<unsigned long long *>(smem + MC_TAB_BYTES);
  G.fx = a.fx;
  G.stride = m;
  G.flags_a = a.flags;
  G.flags_i = a.flags + m;
  G.status = &a.ctr->status;
  G.m = m;
  const mc_cell *cells = a.cells;
  const double *g = a.g;
  if (threadIdx.x < MC_TOTALS) s_tot[threadIdx.x] = 0;
  if (threadIdx.x == 0) {
    mc_scale_clear(&s_scale);
    s_thick = 0;
  }
  if (LDS_T)
    for (int c = threadIdx.x; c < 4 * m; c += blockDim.x) G.t[c] = 0;
  if (LDS_C) {
    mc_cell *lc = reinterpret_cast<mc_cell *>(G.t + 4 * m);
    double *lg = reinterpret_cast<double *>(lc + m + 2);
    for (int c = threadIdx.x; c < m; c += blockDim.x) lg[c] = a.g[c];
    cells = mc_cells_fill(lc, a.cells, m);
    g = lg;
  }
  __syncthreads();
  if (LDS_T) { /* the split */
    int kg = -1023;
    for (int c = threadIdx.x; c < m; c += blockDim.x) {
      const int k = mc_ceil_log2(g[c]);
      kg = k > kg ? k : kg;
    }
    atomicMax(&s_scale.g, kg);
    mc_scale_scatter(&s_scale, cells, m);
    mc_count_thick(&s_thick, cells, m, a.L.dx);
    const uint64_t i = queue.q.next + __lane_id();
    if (i < queue.q.end) atomicMax(&s_scale.w, mc_ceil_log2(a.init.wmc[i]));
    const uint64_t j =
        mc_scale_place(0, (uint64_t)a.n, (uint64_t)threadIdx.x * gridDim.x + blockIdx.x,
                       (uint64_t)blockDim.x * gridDim.x);
    if (j < (uint64_t)a.n) atomicMax(&s_scale.w, mc_ceil_log2(a.init.wmc[j]));
    __syncthreads();
  }
  const bool limbs = mc_grad_split(G, s_scale, a.L.dx, blockDim.x >> 6);

  mc_grad_io<HAVE_SCORE> io{a.init, a.score, 0.0, 0.0, 1};
  auto on_event = [&](mc_mask lanes, int c8, const mc_cell &cell, bool coll, double di, double dw,
                      double wmc) {
    mc_grad_event<MC_GRAD_LIMBS>(io, G, g, lanes, c8, cell, coll, di, dw, wmc);
  };
  if constexpr (LDS_T) { /* thick cells: as in the history kernel.  20,000
       histories of 2,300 collisions on 100 cells, their scores known, 4.80 ms
       with the common walk, 3.03 with this one, 2 M of 340 events 52.3 and 32.9 */
    const int thick = __builtin_amdgcn_readfirstlane((int)s_thick);
    if (limbs && 2 * thick > m) { /* block-uniform */
      mc_walk_bank<LDS_C, U, true>(io, queue, a.L, mc_walk_live<U>(a.L), cells, tab, refill_k,
                   G.every, a.max_events, s_tot, on_event, mc_grad_mover{G, G.every});
      __syncthreads();
      mc_grad_move(G, threadIdx.x, blockDim.x);
      events_out(s_tot, a.ctr);
      return;
    }
  }
  const mc_walk_k K = mc_walk_live<U>(a.L);
  if (LDS_T && limbs) { /* block-uniform */
    mc_walk_bank<LDS_C>(io, queue, a.L, K, cells, tab, refill_k, G.every, a.max_events, s_tot,
                 on_event, mc_grad_mover{G, G.every});
  } else {
    constexpr int MODE = LDS_T ? MC_GRAD_CARRY : MC_GRAD_GLOBAL;
    mc_walk_bank<LDS_C, U>(io, queue, a.L, K, cells, tab, refill_k, 1 << 30, a.max_events, s_tot,
                 [&](mc_mask lanes, int c8, const mc_cell &cell, bool coll, double di, double dw,
                     double wmc) {
                   mc_grad_event<MODE>(io, G, g, lanes, c8, cell, coll, di, dw, wmc);
                 },
                 [](int) {});
  }
  __syncthreads();
  if (LDS_T) mc_grad_move(G, threadIdx.x, blockDim.x, limbs);
  events_out(s_tot, a.ctr);
}

__global__ void k_setup_cells(int m, const double *sig_a, const double *sig_i, mc_cell *cells,
                              unsigned long long *fx, int fx_words_per_cell, uint32_t *flags,
                              int flag_words_per_cell, mc_counters *ctr) {
  const size_t c = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (c < (size_t)m) {
    mc_cell k;
    k.sig_a = sig_a[c];
    k.sig_i = sig_i[c];
    cells[c] = k;
    for (int w = 0; w < fx_words_per_cell; ++w) fx[(size_t)w * m + c] = 0;
    for (int w = 0; w < flag_words_per_cell; ++w) flags[(size_t)w * m + c] = 0;
  }
  mc_counters_clear(ctr, (uint64_t)c);
}

__global__ void k_finalize2(int m, const unsigned long long *fx, const uint32_t *flags,
                            double *ga, double *gi, mc_counters *ctr,
                            mc_counters *host_ctr) {
  mc_counters_fold(ctr, host_ctr);
  const size_t c = (size_t)blockIdx.x * blockDim.x + threadIdx.x, n = (size_t)m;
  if (c < n) {
    ga[c] = ga[c] + mc_fx_finalize(fx[c], fx[n + c], flags[c]);
    gi[c] = gi[c] + mc_fx_finalize(fx[2 * n + c], fx[3 * n + c], flags[n + c]);
  }
}

__global__ void k_finalize1(int m, const unsigned long long *fx, const uint32_t *flags, double *w,
                            mc_counters *ctr, mc_counters *host_ctr) {
  mc_counters_fold(ctr, host_ctr);
  const size_t c = (size_t)blockIdx.x * blockDim.x + threadIdx.x, n = (size_t)m;
  if (c < n && ctr->left == 0) w[c] = w[c] + mc_fx_finalize(fx[c], fx[n + c], flags[c]);
}

/* the counters that the finalizing kernel has handed over */
int read_counters(mcgpu_context *ctx, hipStream_t s, mcgpu_stats *stats) {
  MC_HIP(ctx, hipStreamSynchronize(s));
  const mc_counters *hc = (const mc_counters *)ctx->host_counters;
  if (stats) {
    float ms = 0.f;
    (void)hipEventElapsedTime(&ms, ctx->ev0, ctx->ev1);
    stats->events = hc->events;
    stats->collisions = hc->collisions;
    stats->n_left = (int64_t)hc->n_left;
    stats->n_right = (int64_t)hc->n_right;
    stats->n_killed = (int64_t)hc->n_killed;
    stats->kernel_ms = ms;
  }
  if (hc->status & 1u)
    return mc_fail(ctx, MCGPU_ERR_EVENT_CAP, "a history exceeded max_events_per_history");
  if (hc->status & 2u) return mc_fail(ctx, MCGPU_ERR_RANGE, "a tally term was outside +-2^39");
  return MCGPU_OK;
}

int cells_setup(mcgpu_context *ctx, int m, const double *sig_a, const double *sig_i, int fx_words,
                int flag_words, hipStream_t s) {
  int rc;
  if ((rc = mc_ensure(ctx, &ctx->cells, &ctx->cells_bytes, sizeof(mc_cell) * (size_t)m))) return rc;
  if ((rc = mc_ensure(ctx, &ctx->fx, &ctx->fx_bytes, 8 * (size_t)fx_words * m))) return rc;
  if ((rc = mc_ensure(ctx, &ctx->flags, &ctx->flags_bytes, 4 * (size_t)flag_words * m))) return rc;
  hipLaunchKernelGGL(k_setup_cells, dim3(((unsigned)m + 255) / 256), dim3(256), 0, s, m, sig_a, sig_i,
                     (mc_cell *)ctx->cells, (unsigned long long *)ctx->fx, fx_words,
                     (uint32_t *)ctx->flags, flag_words, (mc_counters *)ctx->counters);
  MC_HIP(ctx, hipGetLastError());
  return MCGPU_OK;
}

template <bool T, bool C, bool S>
int launch_adj(mcgpu_context *ctx, const adj_args &a, const mcgpu_options &o, hipStream_t s,
               size_t lds) {
  auto kern = k_adjoint<T, C, S>;
  if (lds > 65536)
    (void)hipFuncSetAttribute(reinterpret_cast<const void *>(kern),
                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  int per_cu = 0;
  int block = o.block_size;
  if (block <= 0) {
    block = mc_auto_block(ctx, kern, lds, &per_cu);
  } else if (block > 1024 || block % 64) {
    return mc_fail(ctx, MCGPU_ERR_ARG, "block_size must be a multiple of 64 and <= 1024");
  } else if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kern, block, lds) !=
                 hipSuccess || per_cu < 1) {
    per_cu = 1;
  }
  const int grid = o.grid_blocks > 0 ? o.grid_blocks : mc_auto_grid(ctx, a.L.m, a.n, per_cu);
  const int k = o.events_per_refill > 0 ? o.events_per_refill : 0; /* 0: adaptive */
  hipLaunchKernelGGL(kern, dim3(grid), dim3(block), lds, s, a, k, per_cu);
  MC_HIP(ctx, hipGetLastError());
  return MCGPU_OK;
}

/* the two tallies, cells and target weights in LDS when they fit, else the
   tallies, else nothing */
template <bool S>
int launch_adj_fit(mcgpu_context *ctx, const adj_args &a, const mcgpu_options &o, hipStream_t s) {
  const size_t m = (size_t)a.L.m, budget = ctx->lds_per_block - 256;
  if (MC_TAB_BYTES + MC_PAD_BYTES + 56 * m <= budget)
    return launch_adj<true, true, S>(ctx, a, o, s, MC_TAB_BYTES + MC_PAD_BYTES + 56 * m);
  if (MC_TAB_BYTES + 32 * m <= budget)
    return launch_adj<true, false, S>(ctx, a, o, s, MC_TAB_BYTES + 32 * m);
  return launch_adj<false, false, S>(ctx, a, o, s, MC_TAB_BYTES);
}

} // namespace

extern "C" {

int mcgpu_forward_cells(mcgpu_context *ctx, int64_t n, const mcgpu_bank *bank,
                        const double *sig_a, const double *sig_i, double *weights_absorbed,
                        int32_t min_index, int32_t max_index, double dx,
                        double particle_min_weight, const double *g, double *history_score,
                        int8_t *result, const mcgpu_options *opt, mcgpu_stats *stats,
                        void *stream) {
  if (!ctx) return MCGPU_ERR_ARG;
  ctx->err.clear();
  if (n < 0 || !bank || !sig_a || !sig_i || !weights_absorbed ||
      mc_layer_cells(min_index, max_index) == 0 ||
      (history_score && !g))
    return mc_fail(ctx, MCGPU_ERR_ARG, "forward_cells: bad arguments");
  MC_HIP(ctx, hipSetDevice(ctx->device));
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const int m = mc_layer_cells(min_index, max_index);
  int rc = cells_setup(ctx, m, sig_a, sig_i, 2, 1, s);
  if (rc) return rc;
  mcgpu_options o;
  mcgpu_default_options(&o);
  if (opt) o = *opt;
  if (history_score && o.kernel != MCGPU_KERNEL_HISTORY)
    return mc_fail(ctx, MCGPU_ERR_ARG, "per-history scores need the history kernel");
  mc_transport_args a;
  memset(&a, 0, sizeof a);
  a.L.index_start = min_index;
  a.L.m = m;
  a.L.dx = dx;
  a.L.min_weight = particle_min_weight;
  a.n = n;
  a.soa = *bank;
  a.result8 = result;
  a.cells = (const mc_cell *)ctx->cells;
  a.fx = (unsigned long long *)ctx->fx;
  a.flags = (uint32_t *)ctx->flags;
  a.ctr = (mc_counters *)ctx->counters;
  a.max_events = o.max_events_per_history ? o.max_events_per_history : (1ULL << 27);
  a.g = g;
  a.score = history_score;
  MC_HIP(ctx, hipEventRecord(ctx->ev0, s));
  int sweep = 0;
  do {
    if (n > 0) {
      rc = o.kernel == MCGPU_KERNEL_EVENT ? mc_launch_event(ctx, a, o, s)
                                          : mc_launch_history(ctx, a, o, s, sweep++);
      if (rc) return rc;
    }
    MC_HIP(ctx, hipEventRecord(ctx->ev1, s));
    hipLaunchKernelGGL(k_finalize1, dim3(((unsigned)m + 255) / 256), dim3(256), 0, s, m,
                       (const unsigned long long *)ctx->fx, (const uint32_t *)ctx->flags,
                       weights_absorbed, a.ctr, (mc_counters *)ctx->host_counters);
    MC_HIP(ctx, hipGetLastError());
    rc = read_counters(ctx, s, stats);
  } while (rc != MCGPU_ERR_HIP && ((const mc_counters *)ctx->host_counters)->left != 0);
  return rc;
}

int mcgpu_adjoint_cells(mcgpu_context *ctx, int64_t n, const mcgpu_bank *initial,
                        const double *sig_a, const double *sig_i, int32_t min_index,
                        int32_t max_index, double dx, double particle_min_weight,
                        const double *g, const double *history_score, double *grad_sig_a,
                        double *grad_sig_i, const mcgpu_options *opt, mcgpu_stats *stats,
                        void *stream) {
  if (!ctx) return MCGPU_ERR_ARG;
  ctx->err.clear();
  if (n < 0 || !initial || !sig_a || !sig_i || !g || !grad_sig_a || !grad_sig_i ||
      mc_layer_cells(min_index, max_index) == 0)
    return mc_fail(ctx, MCGPU_ERR_ARG, "adjoint_cells: bad arguments");
  if (n > 0 && (!initial->seed || !initial->x || !initial->mu || !initial->wmc || !initial->index))
    return mc_fail(ctx, MCGPU_ERR_ARG, "adjoint_cells: bank has a null array");
  MC_HIP(ctx, hipSetDevice(ctx->device));
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const int m = mc_layer_cells(min_index, max_index);
  int rc = cells_setup(ctx, m, sig_a, sig_i, 4, 2, s);
  if (rc) return rc;
  mcgpu_options o;
  mcgpu_default_options(&o);
  if (opt) o = *opt;
  adj_args a;
  memset(&a, 0, sizeof a);
  a.L.index_start = min_index;
  a.L.m = m;
  a.L.dx = dx;
  a.L.min_weight = particle_min_weight;
  a.n = n;
  a.init = *initial;
  a.cells = (const mc_cell *)ctx->cells;
  a.g = g;
  a.score = history_score;
  a.fx = (unsigned long long *)ctx->fx;
  a.flags = (uint32_t *)ctx->flags;
  a.ctr = (mc_counters *)ctx->counters;
  a.max_events = o.max_events_per_history ? o.max_events_per_history : (1ULL << 27);
  MC_HIP(ctx, hipEventRecord(ctx->ev0, s));
  if (n > 0) {
    rc = history_score ? launch_adj_fit<true>(ctx, a, o, s) : launch_adj_fit<false>(ctx, a, o, s);
    if (rc) return rc;
  }
  MC_HIP(ctx, hipEventRecord(ctx->ev1, s));
  hipLaunchKernelGGL(k_finalize2, dim3(((unsigned)m + 255) / 256), dim3(256), 0, s, m,
                     (const unsigned long long *)ctx->fx, (const uint32_t *)ctx->flags,
                     grad_sig_a, grad_sig_i, a.ctr, (mc_counters *)ctx->host_counters);
  MC_HIP(ctx, hipGetLastError());
  return read_counters(ctx, s, stats);
}

} /* extern "C" */
