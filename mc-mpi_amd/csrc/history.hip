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

constexpr size_t TAB_BYTES = 16 * MC_ABS_N; /* the absorbed-fraction rows in LDS */

/* A wave's histories, one per lane.  tally(lanes, c, dw) adds deposits;
   moves(k) is called before every (at most) k events per lane, k <= k_max. */
template <bool SCORE, typename Tally, typename Moves>
__device__ __forceinline__ void walk_bank(const mc_transport_args &a, const mc_cell *cells,
                                          const double *g, const double2 *tab, int refill_k,
                                          mc_queue q, const mc_walk_k &K,
                                          unsigned long long *s_tot, int k_max, Tally tally,
                                          Moves moves) {
  mc_walk p;
  p.s2 = 0;
  p.x = p.mu = p.wmc = p.rh = p.rl = p.fe = p.fs = 0.0;
  p.c = p.st = 0;
  int64_t idx = 0;
  bool has = false, capped = false;
  mc_mask run = 0, pend = 0; /* lanes whose history goes on / waits for the general event */
  uint64_t ev = 0;
  uint32_t col = 0;
  double score = 0.0;
  unsigned long long tot_ev = 0, tot_col = 0, nl = 0, nr = 0, nk = 0;

  /* events between refills: refill_k if positive, else adapted per wave
     from the lanes found idle at each refill (many idle: the histories are
     short against the interval, halve it; almost none: double it, since
     each refill costs a queue atomic and a pass through this loop) */
  const bool adapt = refill_k <= 0;
  int kk = adapt ? 128 : refill_k;
  int wait = 1;
  /* wave-uniform bound on every lane's event count (a waiting event counted);
     recomputed exactly (the largest in the wave) when an interval could reach
     the cap, which then shortens the interval: no history passes the cap */
  uint64_t ev_bound = 0;
  for (;;) {
    if (mc_queue_more(q)) { /* wave-uniform */
      const mc_mask need = mc_lanes(!has);
      if (adapt) {
        const int idle = __popcll(need);
        kk = idle > 16 ? (kk > 8 ? kk >> 1 : 8) : (idle < 4 ? (kk < 256 ? kk << 1 : 256) : kk);
      }
      if (need) {
        const int64_t i = mc_queue_take(q, need, &a.ctr->next);
        bool on = false;
        if (!has && i >= 0) {
          mc_state in;
          load_state(a, i, in);
          mc_walk_from(p, in, a.L);
          idx = i;
          has = true;
          on = mc_walk_alive(p, a.L);
          ev = 0;
          col = 0;
          score = 0.0;
        }
        run |= mc_lanes(on);
      }
    }
    if (mc_lanes(has) == 0) break; /* wave-uniform */
    int ki = kk < k_max ? kk : k_max - 1; /* a waiting lane may add one */
    if (ev_bound + (uint64_t)ki >= a.max_events) {
      ev_bound = mc_wave_max_u64(has ? ev + (mc_in(pend) ? 1u : 0u) : 0ull);
      if (ev_bound + (uint64_t)ki >= a.max_events) ki = (int)(a.max_events - ev_bound);
    }
    ev_bound += (uint64_t)ki;
    moves(ki + 1);
    uint32_t ei = 0; /* events of this interval */
    const int general =
        mc_walk_many(p, run, pend, ki, wait, cells, tab, K, ei, col,
                     [&](mc_mask lanes, int c, const mc_cell &, bool, double, double dw, double) {
                       tally(lanes, c, dw);
                       if (SCORE && mc_in(lanes)) score = score + g[c] * dw;
                     });
    wait = mc_walk_wait(wait, general, ki);
    ev += ei;
    const bool on = mc_in(run), waits = mc_in(pend);
    if (has && !waits && (!on || ev >= a.max_events)) {
      mc_state out;
      mc_walk_to(out, p, a.L);
      int code = mc_exit_code(out, a.L);
      if (on) { /* runaway history stopped by the guard */
        capped = true;
        code = 2;
      }
      store_state(a, idx, out, code);
      if (a.events) a.events[idx] = ev;
      if (a.collisions) a.collisions[idx] = col;
      if (SCORE) a.score[idx] = score;
      tot_ev += ev;
      tot_col += col;
      nl += code == -1;
      nr += code == 1;
      nk += code == 0;
      has = false;
    }
    run &= mc_lanes(has);
  }

  mc_totals_wave(s_tot, tot_ev, tot_col, nl, nr, nk);
  if (capped) atomicOr(&a.ctr->status, 1u);
}

template <bool LDS_TALLY, bool LDS_CELLS, bool SCORE>
__global__ __launch_bounds__(1024) void k_history(mc_transport_args a, int refill_k,
                                                   int per_cu) {
  extern __shared__ __align__(16) unsigned char smem[];
  __shared__ int s_k;
  __shared__ unsigned long long s_tot[5];
  const mc_walk_k K = mc_walk_live(a.L);
  const mc_queue q = mc_queue_open(a.n, per_cu);
  const int m = a.L.m;
  double2 *tab = reinterpret_cast<double2 *>(smem);
  for (int j = threadIdx.x; j < MC_ABS_N; j += blockDim.x)
    tab[j] = make_double2(mc_abs_tab[j][0], mc_abs_tab[j][1]);
  unsigned long long *t0 = reinterpret_cast<unsigned long long *>(smem + TAB_BYTES), *t1 = t0 + m;
  if (LDS_TALLY) {
    for (int c = threadIdx.x; c < m; c += blockDim.x) {
      t0[c] = 0;
      t1[c] = 0;
    }
  }
  const mc_cell *cells = a.cells;
  const double *g = a.g;
  if (LDS_CELLS) {
    mc_cell *lc = reinterpret_cast<mc_cell *>(smem + TAB_BYTES + (size_t)16 * m);
    for (int c = threadIdx.x; c < m; c += blockDim.x) lc[c] = a.cells[c];
    cells = lc;
    if (SCORE) {
      double *lg = reinterpret_cast<double *>(smem + TAB_BYTES + (size_t)32 * m);
      for (int c = threadIdx.x; c < m; c += blockDim.x) lg[c] = a.g[c];
      g = lg;
    }
  }
  unsigned long long *fx_lo = a.fx, *fx_hi = a.fx + m;
  uint32_t *flags = a.flags;
  unsigned int *status = &a.ctr->status;
  if (threadIdx.x < 5) s_tot[threadIdx.x] = 0;
  mc_counters *ctr = a.ctr;
  auto totals = [&]() { /* after a barrier */
    if (threadIdx.x == 0)
      mc_totals_block(s_tot, &ctr->events, &ctr->collisions, &ctr->n_left, &ctr->n_right,
                      &ctr->n_killed);
  };
  if (!LDS_TALLY) {
    __syncthreads();
    walk_bank<SCORE>(a, cells, g, tab, refill_k, q, K, s_tot, 1 << 30,
                     [&](mc_mask lanes, int c, double dw) {
                       if (mc_in(lanes)) mc_tally(fx_lo, fx_hi, flags, status, c, dw);
                     },
                     [](int) {});
    __syncthreads();
    totals();
    return;
  }

  /* the block's weights: the largest among the first histories of its waves
     (a guess that sets the limbs' range; heavier ones go to the global tally) */
  if (threadIdx.x == 0) s_k = -1023;
  __syncthreads();
  {
    const uint64_t i = q.next + __lane_id();
    if (i < q.end) atomicMax(&s_k, mc_ceil_log2(a.aos ? a.aos[i].wmc : a.soa.wmc[i]));
  }
  __syncthreads();
  const int waves = blockDim.x >> 6;
  const mc_block_tally B = mc_block_tally_for(m, __builtin_amdgcn_readfirstlane(s_k), waves);
  if (B.limbs) { /* block-uniform */
    int left = B.every;
    walk_bank<SCORE>(a, cells, g, tab, refill_k, q, K, s_tot, B.every,
                     [&](mc_mask lanes, int c, double dw) {
                       mc_tally_limbs(t0, t1, B.S, fx_lo, fx_hi, flags, status, lanes, c, dw);
                     },
                     [&](int k) {
                       if (left < k) { /* wave-uniform */
                         mc_limbs_move(t0, t1, B.S.L, m, __lane_id(), 64, fx_lo, fx_hi);
                         left = B.every;
                       }
                       left -= k;
                     });
    __syncthreads();
    mc_limbs_move(t0, t1, B.S.L, m, threadIdx.x, blockDim.x, fx_lo, fx_hi);
  } else {
    walk_bank<SCORE>(a, cells, g, tab, refill_k, q, K, s_tot, 1 << 30,
                     [&](mc_mask lanes, int c, double dw) {
                       if (mc_in(lanes)) mc_tally(t0, t1, flags, status, c, dw);
                     },
                     [](int) {});
    __syncthreads();
    for (int c = threadIdx.x; c < m; c += blockDim.x) {
      mc_fx v;
      v.lo = t0[c];
      v.hi = t1[c];
      mc_fx_atomic_add(&fx_lo[c], &fx_hi[c], v);
    }
  }
  totals(); /* the barrier after the walk stands before */
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
  const size_t tally = 16 * m + TAB_BYTES, cells = sizeof(mc_cell) * m;
  const size_t budget = ctx->lds_per_block - 256; /* the kernel's static LDS */
  const bool lds_tally = tally <= budget;
  if (a.score) { /* per-history score of a weighted tally (forward of the adjoint) */
    if (!a.g) return mc_fail(ctx, MCGPU_ERR_ARG, "score output needs target weights g");
    const size_t extra = 8 * m;
    const bool lds_cells = lds_tally && tally + cells + extra <= budget;
    if (lds_tally && lds_cells) return launch_one<true, true, true>(ctx, a, o, s, tally + cells + extra);
    if (lds_tally) return launch_one<true, false, true>(ctx, a, o, s, tally);
    return launch_one<false, false, true>(ctx, a, o, s, TAB_BYTES);
  }
  const bool lds_cells = lds_tally && tally + cells <= budget;
  if (lds_tally && lds_cells) return launch_one<true, true, false>(ctx, a, o, s, tally + cells);
  if (lds_tally) return launch_one<true, false, false>(ctx, a, o, s, tally);
  return launch_one<false, false, false>(ctx, a, o, s, TAB_BYTES);
}
