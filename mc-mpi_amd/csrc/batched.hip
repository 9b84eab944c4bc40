/*
 * batched.hip -- many independent slab problems in one persistent launch.
 *
 * The reference runs one Layer per MPI rank and transports each layer's bank
 * with Layer::simulate (src/layer.cpp:239-361).  Here thousands of
 * independent slabs (each one Layer's worth of work) share a single launch:
 *  - the host cuts every slab's bank into tiles of particles_per_lane *
 *    block_size particles, or of a block's part (mc_tile_size), and orders
 *    them by their time (mc_tile_work), so the long tiles start early;
 *  - each persistent block takes the next tile from a global counter, zeroes
 *    its LDS tally for that slab's cells (and stages the slab's cross sections
 *    in LDS when both fit), runs the tile's histories with lanes refilled
 *    from an LDS counter (as in the history kernel), and adds the exact
 *    fixed-point tally to the slab's global cells once per tile;
 *  - setup (cross-section table, zeroed tallies and counters), transport and
 *    finalize (tally -> weights_absorbed) are captured once into a hipGraph
 *    and replayed; zeroing is done by kernels (no memset nodes).
 * Per history the arithmetic is the single-slab kernels' arithmetic, so each
 * slab's results are bit-identical to transporting it alone.
 *
 * The event is the common step of mc_walk.h; what bounds a launch besides it
 * is the tiles: a block waits for its tile's longest history, and few large
 * tiles leave CUs idle.  Measured, 512 slabs of 32 to 8,192 cells with 100 to
 * 1e5 histories each: 110 -> 50 ms with mc_walk.h and tiles of half a part, 43
 * ms with histories that set out apart, 38.7 in tiles of a whole part, 33.0
 * sorted by time (2.8e11 events/s; 4.9e11 where all lies in LDS and no block
 * waits).
 */
#include <algorithm>
#include <vector>

#include "mc_walk.h"

namespace {

struct batch_args {
  const mc_slab_k *slabs;
  const mc_tile_k *tiles;
  int32_t n_tiles;
  uint32_t lds;            /* dynamic LDS bytes of a block */
  int32_t lds_cells_max_m; /* slabs with m <= this stage cross sections in LDS */
  int32_t lds_tally_max_m; /* slabs with m <= this keep their tally in LDS; larger
                              ones add straight into the global tally */
  mcgpu_bank soa;
  const mc_cell *cells;
  unsigned long long *fx; /* lo words [0, total), hi words [total, 2 total) */
  int64_t total_cells;
  uint32_t *flags;
  int8_t *result8;
  mc_counters *ctr;
  uint64_t max_events;
};

struct tile_io {
  const batch_args &a;
  static constexpr bool RESUMES = false;
  __device__ __forceinline__ int code(const mc_state &p, bool at_cap, const mc_layer_k &L) {
    return mc_end_code(p, at_cap, L);
  }
  __device__ __forceinline__ uint64_t load(int64_t i, mc_state &p) {
    p.seed = a.soa.seed[i];
    p.x = a.soa.x[i];
    p.mu = a.soa.mu[i];
    p.wmc = a.soa.wmc[i];
    p.index = a.soa.index[i];
    return 0;
  }
  __device__ __forceinline__ bool store(int64_t i, mc_state &p, int code, uint64_t ev, uint32_t) {
    if (a.result8) a.result8[i] = (int8_t)code;
    if (ev == 0) return false; /* its state stays as it came (store_state) */
    a.soa.seed[i] = p.seed;
    a.soa.x[i] = p.x;
    a.soa.mu[i] = p.mu;
    a.soa.wmc[i] = p.wmc;
    a.soa.index[i] = p.index;
    return false;
  }
};

/* The tile loop is the history kernel's (mc_walk_bank) with the tile's LDS
   counter as its queue; the tally and cell pointers are LDS or global in
   branches of their own, so every access compiles to the matching
   instruction.  WIDE: some slabs' tallies do not fit LDS beside the rows of
   the absorbed fraction; those that fit without them take all of LDS
   (mc_full_tally), the others the global tally. */
template <bool WIDE>
__global__ __launch_bounds__(1024) void k_batched(batch_args a, int refill_k) {
  extern __shared__ __align__(16) unsigned char smem[];
  __shared__ int s_tile;
  __shared__ mc_scale s_scale;
  __shared__ uint32_t s_thick;
  __shared__ unsigned long long s_next;
  __shared__ unsigned long long s_tot[MC_TOTALS];
  double2 *tab = reinterpret_cast<double2 *>(smem);
  mc_tab_fill(tab);
  unsigned long long *t0 = reinterpret_cast<unsigned long long *>(smem + MC_TAB_BYTES);
  const int B = blockDim.x;
  const int tid = threadIdx.x;
  if (tid < MC_TOTALS) s_tot[tid] = 0;
  if (tid == 0) {
    mc_scale_clear(&s_scale);
    s_thick = 0;
  }
  tile_io io{a};
  bool rows = true; /* in LDS */

  for (;;) {
    if (tid == 0) s_tile = (int)atomicAdd(&a.ctr->next, 1ull);
    __syncthreads();
    const int t = __builtin_amdgcn_readfirstlane(s_tile);
    if (t >= a.n_tiles) break; /* block-uniform */
    const mc_tile_k tile = a.tiles[t];
    const mc_slab_k sl = a.slabs[__builtin_amdgcn_readfirstlane(tile.slab)];
    mc_layer_k L;
    L.index_start = __builtin_amdgcn_readfirstlane(sl.index_start);
    L.m = __builtin_amdgcn_readfirstlane(sl.m);
    L.dx = mc_uniform(sl.dx);
    L.min_weight = mc_uniform(sl.min_weight);
    const int m = L.m;
    const int64_t cell_off = (int64_t)mc_readlane64((unsigned long long)sl.cell_off, 0);
    const bool lds_tally = m <= a.lds_tally_max_m; /* block-uniform */
    const bool lds_cells = m <= a.lds_cells_max_m; /* implies lds_tally */
    const int sh = lds_cells ? mc_limbs_copies(m, a.lds - MC_TAB_BYTES - MC_PAD_BYTES -
                                                      sizeof(mc_cell) * m)
                             : 0;
    const mc_limbs T = mc_limbs_at(t0, m, sh), mine = mc_limbs_mine(T);
    unsigned long long *t1 = t0 + m; /* words with carry: one copy */
    mc_cell *lc = reinterpret_cast<mc_cell *>(t0 + (2 * (size_t)m << sh));
    const mc_cell *gc = a.cells + cell_off;
    const int most = (int)(a.lds / 16);
    const bool full = WIDE && !lds_tally && m <= most + MC_FULL_BEYOND; /* block-uniform */
    if (lds_tally) {
      for (int c = tid; c < 2 * m << sh; c += B) t0[c] = 0;
      if (lds_cells) lc = mc_cells_fill(lc, gc, m);
    }
    mc_full_tally F;
    F.t = reinterpret_cast<unsigned long long *>(smem);
    F.m = m < most ? m : most;
    if (WIDE) {
      if (full)
        for (int c = tid; c < 2 * F.m; c += B) F.t[c] = 0;
      else if (!rows)
        mc_tab_fill(tab);
      rows = !full;
    }
    if (tid == 0) s_next = (unsigned long long)tile.begin;
    /* the tile's weights, from one history per thread (as the history kernel) */
    {
      const uint64_t i = mc_scale_place(tile.begin, tile.end, tid, B);
      if (i < (uint64_t)tile.end) atomicMax(&s_scale.w, mc_ceil_log2(a.soa.wmc[i]));
    }
    if ((lds_tally || full) && m >= MC_THICK_CELLS) mc_scale_cells(&s_scale, gc, m, L.dx);
    if (lds_cells) mc_count_thick(&s_thick, gc, m, L.dx);
    __syncthreads();

    const mc_walk_k K = mc_walk_live(L);
    const mc_block_tally bt = mc_block_tally_for(m, s_scale, B >> 6);
    mc_tile_queue queue{&s_next, mc_readlane64((unsigned long long)tile.end, 0), false};
    unsigned long long *fx_lo = a.fx + cell_off, *fx_hi = fx_lo + a.total_cells;
    uint32_t *flags = a.flags + cell_off;
    unsigned int *status = &a.ctr->status;
    auto limbs = [&](mc_mask lanes, int c8, const mc_cell &, bool, double, double dw, double) {
      mc_tally_limbs(mine, bt.S, fx_lo, fx_hi, flags, status, lanes, c8, dw);
    };
    const mc_mover mover{T, fx_lo, fx_hi, m, bt.S.L, bt.every, bt.every};
    if (lds_tally && bt.limbs) {
      if (lds_cells && 2 * s_thick > (uint32_t)m) /* block-uniform */
        mc_walk_bank<true, MC_IN_LDS, true>(io, queue, L, K, lc, tab, refill_k, bt.every,
                     a.max_events, s_tot, limbs, mover);
      else if (lds_cells)
        mc_walk_bank<true>(io, queue, L, K, lc, tab, refill_k, bt.every, a.max_events, s_tot, limbs,
                     mover);
      else
        mc_walk_bank<false>(io, queue, L, K, gc, tab, refill_k, bt.every, a.max_events, s_tot, limbs,
                     mover);
    } else if (lds_tally) { /* heavy weights */
      mc_walk_bank<false>(io, queue, L, K, gc, tab, refill_k, 1 << 30, a.max_events, s_tot,
                   [&](mc_mask lanes, int c8, const mc_cell &, bool, double, double dw, double) {
                     if (mc_in(lanes)) mc_tally(t0, t1, flags, status, c8 >> 3, dw);
                   },
                   [](int) {});
    } else if (full) {
      F.B = bt;
      F.fx_lo = fx_lo;
      F.fx_hi = fx_hi;
      F.flags = flags;
      F.status = status;
      F.left = bt.every;
      mc_walk_bank<false>(io, queue, L, K, gc, reinterpret_cast<const double2 *>(mc_abs_tab),
                   refill_k, F.every(), a.max_events, s_tot,
                   [&](mc_mask lanes, int c8, const mc_cell &, bool, double, double dw, double) {
                     F.add(lanes, c8, dw);
                   },
                   [&](int n) { F.moves(n); });
    } else if (WIDE) {
      mc_walk_bank<false, MC_IN_MEMORY>(
                   io, queue, L, mc_walk_live<MC_IN_MEMORY>(L), gc, tab, refill_k, 1 << 30,
                   a.max_events, s_tot,
                   [&](mc_mask lanes, int c, const mc_cell &, bool, double, double dw, double) {
                     if (mc_in(lanes)) mc_tally(fx_lo, fx_hi, flags, status, c, dw);
                   },
                   [](int) {});
    }

    __syncthreads();
    if (lds_tally && bt.limbs) {
      mc_limbs_move(T, bt.S.L, m, tid, B, fx_lo, fx_hi);
    } else if (lds_tally) {
      for (int c = tid; c < m; c += B) {
        mc_fx v;
        v.lo = t0[c];
        v.hi = t1[c];
        mc_fx_atomic_add(&fx_lo[c], &fx_hi[c], v);
      }
    } else if (full) {
      F.out();
    }
    if (tid == 0) {
      mc_scale_clear(&s_scale);
      s_thick = 0;
    }
    __syncthreads();
  }
  /* the break follows a barrier after the last tile's totals */
  if (tid == 0) mc_totals_out(s_tot, a.ctr, mc_counter_copy());
}

__global__ void k_batch_setup(int64_t total, const double *sigs, const double *ar, mc_cell *cells,
                              unsigned long long *fx, uint32_t *flags, mc_counters *ctr) {
  const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (c < total) {
    cells[c] = mc_make_cell(sigs[c], ar[c]);
    fx[c] = 0;
    fx[total + c] = 0;
    flags[c] = 0;
  }
  mc_counters_clear(ctr, (uint64_t)c);
}

__global__ void k_batch_finalize(int64_t total, const unsigned long long *fx,
                                 const uint32_t *flags, double *weights, mc_counters *ctr,
                                 mc_counters *host_ctr) {
  mc_counters_fold(ctr, host_ctr);
  const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (c < total) weights[c] = weights[c] + mc_fx_finalize(fx[c], fx[total + c], flags[c]);
}

void (*batched_kernel(const mc_batched_shape &sh))(batch_args, int) {
  return sh.wide ? k_batched<true> : k_batched<false>;
}

} // namespace

int mc_batched_plan_shape(mcgpu_context *ctx, int max_m, int block, int grid, int refill,
                          mc_batched_shape *out) {
  if (block > 1024 || block < 0 || block % 64)
    return mc_fail(ctx, MCGPU_ERR_ARG, "block_size must be a multiple of 64 and <= 1024");
  mc_batched_shape sh;
  sh.refill = refill > 0 ? refill : 0; /* 0: adaptive */
  /* LDS: the largest slab's tally plus its cross sections, as far as they fit
     (next to the absorbed-fraction rows and the kernel's static LDS); slabs
     whose tally does not fit add into the global tally directly */
  const size_t budget = ctx->lds_per_block - 256 - MC_TAB_BYTES;
  const size_t lds = std::min(budget, (size_t)32 * (size_t)std::max(max_m, 1) + MC_PAD_BYTES);
  sh.lds = mc_lds_with_copies(lds + MC_TAB_BYTES, max_m);
  sh.lds_cells_max_m = (int)((lds - MC_PAD_BYTES) / 32);
  sh.lds_tally_max_m = (int)(lds / 16);
  sh.wide = max_m > sh.lds_tally_max_m;
  const auto kern = batched_kernel(sh);
  if (sh.lds > 65536)
    (void)hipFuncSetAttribute(reinterpret_cast<const void *>(kern),
                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)sh.lds);
  int per_cu = 0;
  if (block == 0) block = mc_auto_block(ctx, kern, sh.lds, &per_cu);
  sh.block = block;
  sh.grid = grid;
  if (sh.grid <= 0) {
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kern, block, sh.lds) !=
            hipSuccess ||
        per_cu < 1)
      per_cu = 1;
    sh.grid = per_cu * ctx->num_cus;
  }
  *out = sh;
  return MCGPU_OK;
}

int mc_launch_batched(mcgpu_context *ctx, const mc_batched_shape &sh, const mc_slab_k *slabs,
                      const mc_tile_k *tiles, int32_t n_tiles, const mcgpu_bank &bank,
                      const mc_cell *cells, unsigned long long *fx, int64_t total_cells,
                      uint32_t *flags, int8_t *result8, mc_counters *ctr, uint64_t max_events,
                      hipStream_t s) {
  batch_args a;
  a.slabs = slabs;
  a.tiles = tiles;
  a.n_tiles = n_tiles;
  a.lds_cells_max_m = sh.lds_cells_max_m;
  a.lds_tally_max_m = sh.lds_tally_max_m;
  a.lds = (uint32_t)sh.lds;
  a.soa = bank;
  a.cells = cells;
  a.fx = fx;
  a.total_cells = total_cells;
  a.flags = flags;
  a.result8 = result8;
  a.ctr = ctr;
  a.max_events = max_events;
  hipLaunchKernelGGL(batched_kernel(sh), dim3(sh.grid), dim3(sh.block), sh.lds, s, a, sh.refill);
  MC_HIP(ctx, hipGetLastError());
  return MCGPU_OK;
}

struct mcgpu_batch {
  mcgpu_context *ctx = nullptr;
  std::vector<mcgpu_slab> host_slabs;
  mcgpu_options opt{};
  /* inputs (caller-owned device memory) */
  const double *sigs = nullptr, *ar = nullptr;
  double *weights = nullptr;
  int64_t total_cells = 0, total_particles = 0;
  mcgpu_bank bank{};
  int8_t *result = nullptr;
  /* plan-owned device memory */
  mc_slab_k *d_slabs = nullptr;
  mc_tile_k *d_tiles = nullptr;
  int32_t n_tiles = 0;
  size_t tiles_cap = 0;
  mc_cell *d_cells = nullptr;
  unsigned long long *d_fx = nullptr;
  uint32_t *d_flags = nullptr;
  mc_counters *d_ctr = nullptr;
  mc_counters *h_ctr = nullptr;
  int max_m = 0;
  size_t lds = 0;
  int lds_cells_max_m = 0;
  int lds_tally_max_m = 0;
  int block = 1024, grid = 0;
  hipStream_t stream = nullptr;
  hipGraph_t graph = nullptr;
  hipGraphExec_t exec = nullptr;
  hipEvent_t e0 = nullptr, e1 = nullptr;
};

namespace {

int batch_tiles(mcgpu_batch *b) {
  mcgpu_context *ctx = b->ctx;
  const int ppl = b->opt.particles_per_lane > 0 ? b->opt.particles_per_lane : 16;
  const int64_t T = (int64_t)ppl * b->block;
  double share = 0.0; /* automatic: mc_tile_size */
  if (b->opt.particles_per_lane <= 0)
    for (const mcgpu_slab &h : b->host_slabs)
      share += (double)h.n * mc_layer_cells(h.min_index, h.max_index) / b->grid;
  std::vector<mc_tile_k> tiles;
  std::vector<double> work;
  for (size_t s = 0; s < b->host_slabs.size(); ++s) {
    const mcgpu_slab &h = b->host_slabs[s];
    const int m = mc_layer_cells(h.min_index, h.max_index);
    const int64_t Ts = b->opt.particles_per_lane > 0 ? T : mc_tile_size(T, share, h.n, m, b->block);
    for (int64_t p0 = 0; p0 < h.n; p0 += Ts) {
      mc_tile_k t;
      t.slab = (int32_t)s;
      t.pad_ = 0;
      t.begin = h.particle_offset + p0;
      t.end = h.particle_offset + std::min(h.n, p0 + Ts);
      tiles.push_back(t);
      work.push_back(mc_tile_work(t.end - t.begin, m));
    }
  }
  std::vector<size_t> order(tiles.size());
  for (size_t i = 0; i < order.size(); ++i) order[i] = i;
  std::stable_sort(order.begin(), order.end(), [&](size_t x, size_t y) { return work[x] > work[y]; });
  std::vector<mc_tile_k> sorted(tiles.size());
  for (size_t i = 0; i < order.size(); ++i) sorted[i] = tiles[order[i]];
  b->n_tiles = (int32_t)sorted.size();
  if (sorted.size() > b->tiles_cap) {
    if (b->d_tiles) MC_HIP(ctx, hipFree(b->d_tiles));
    b->d_tiles = nullptr;
    MC_HIP(ctx, hipMalloc(&b->d_tiles, sizeof(mc_tile_k) * (sorted.size() + 1)));
    b->tiles_cap = sorted.size();
  }
  if (!sorted.empty())
    MC_HIP(ctx, hipMemcpy(b->d_tiles, sorted.data(), sizeof(mc_tile_k) * sorted.size(),
                          hipMemcpyHostToDevice));
  return MCGPU_OK;
}

int batch_capture(mcgpu_batch *b) {
  mcgpu_context *ctx = b->ctx;
  int rc;
  mc_batched_shape sh;
  if ((rc = mc_batched_plan_shape(ctx, b->max_m, b->opt.block_size > 0 ? b->opt.block_size : 0,
                                  b->opt.grid_blocks, b->opt.events_per_refill, &sh)))
    return rc;
  b->block = sh.block;
  b->lds = sh.lds;
  b->lds_cells_max_m = sh.lds_cells_max_m;
  b->lds_tally_max_m = sh.lds_tally_max_m;
  b->grid = sh.grid;
  if ((rc = batch_tiles(b))) return rc;
  if (b->exec) {
    (void)hipGraphExecDestroy(b->exec);
    b->exec = nullptr;
  }
  if (b->graph) {
    (void)hipGraphDestroy(b->graph);
    b->graph = nullptr;
  }
  batch_args a;
  a.slabs = b->d_slabs;
  a.tiles = b->d_tiles;
  a.n_tiles = b->n_tiles;
  a.lds_cells_max_m = b->lds_cells_max_m;
  a.lds_tally_max_m = b->lds_tally_max_m;
  a.lds = (uint32_t)b->lds;
  a.soa = b->bank;
  a.cells = b->d_cells;
  a.fx = b->d_fx;
  a.total_cells = b->total_cells;
  a.flags = b->d_flags;
  a.result8 = b->result;
  a.ctr = b->d_ctr;
  a.max_events = b->opt.max_events_per_history ? b->opt.max_events_per_history : (1ULL << 27);
  const int64_t tc = b->total_cells;
  MC_HIP(ctx, hipStreamBeginCapture(b->stream, hipStreamCaptureModeThreadLocal));
  hipLaunchKernelGGL(k_batch_setup, dim3((unsigned)((tc + 255) / 256)), dim3(256), 0, b->stream,
                     tc, b->sigs, b->ar, b->d_cells, b->d_fx, b->d_flags, b->d_ctr);
  hipLaunchKernelGGL(batched_kernel(sh), dim3(sh.grid), dim3(sh.block), sh.lds, b->stream, a,
                     sh.refill);
  hipLaunchKernelGGL(k_batch_finalize, dim3((unsigned)((tc + 255) / 256)), dim3(256), 0,
                     b->stream, tc, (const unsigned long long *)b->d_fx,
                     (const uint32_t *)b->d_flags, b->weights, b->d_ctr, b->h_ctr);
  hipError_t e = hipStreamEndCapture(b->stream, &b->graph);
  if (e != hipSuccess) return mc_fail(ctx, MCGPU_ERR_HIP, "hipStreamEndCapture", e);
  MC_HIP(ctx, hipGraphInstantiate(&b->exec, b->graph, nullptr, nullptr, 0));
  b->opt.block_size = b->block;
  b->opt.grid_blocks = b->grid;
  /* 0 where the plan adapts (mcgpu_batch_options) */
  b->opt.events_per_refill = std::max(b->opt.events_per_refill, 0);
  b->opt.particles_per_lane = std::max(b->opt.particles_per_lane, 0);
  return MCGPU_OK;
}

int batch_launch(mcgpu_batch *b, hipStream_t s, mcgpu_stats *stats) {
  mcgpu_context *ctx = b->ctx;
  MC_HIP(ctx, hipEventRecord(b->e0, s));
  MC_HIP(ctx, hipGraphLaunch(b->exec, s));
  MC_HIP(ctx, hipEventRecord(b->e1, s));
  MC_HIP(ctx, hipStreamSynchronize(s));
  if (stats) {
    float ms = 0.f;
    (void)hipEventElapsedTime(&ms, b->e0, b->e1);
    stats->events = b->h_ctr->events;
    stats->collisions = b->h_ctr->collisions;
    stats->n_left = (int64_t)b->h_ctr->n_left;
    stats->n_right = (int64_t)b->h_ctr->n_right;
    stats->n_killed = (int64_t)b->h_ctr->n_killed;
    stats->kernel_ms = ms;
  }
  if (b->h_ctr->status & 1u)
    return mc_fail(ctx, MCGPU_ERR_EVENT_CAP, "a history exceeded max_events_per_history");
  if (b->h_ctr->status & 2u) return mc_fail(ctx, MCGPU_ERR_RANGE, "a tally term was outside +-2^39");
  return MCGPU_OK;
}

} // namespace

extern "C" {

int mcgpu_batch_destroy(mcgpu_batch *b) {
  if (!b) return MCGPU_OK;
  (void)hipSetDevice(b->ctx->device);
  if (b->stream) (void)hipStreamSynchronize(b->stream);
  if (b->exec) (void)hipGraphExecDestroy(b->exec);
  if (b->graph) (void)hipGraphDestroy(b->graph);
  void *bufs[] = {b->d_slabs, b->d_tiles, b->d_cells, b->d_fx, b->d_flags, b->d_ctr};
  for (void *p : bufs)
    if (p) (void)hipFree(p);
  if (b->h_ctr) (void)hipHostFree(b->h_ctr);
  if (b->e0) (void)hipEventDestroy(b->e0);
  if (b->e1) (void)hipEventDestroy(b->e1);
  if (b->stream) (void)hipStreamDestroy(b->stream);
  delete b;
  return MCGPU_OK;
}

int mcgpu_batch_create(mcgpu_context *ctx, int32_t n_slabs, const mcgpu_slab *slabs,
                       const double *sigs, const double *absorption_rates,
                       double *weights_absorbed, int64_t total_cells, const mcgpu_bank *bank,
                       int8_t *result, const mcgpu_options *opt, mcgpu_batch **out) {
  if (!ctx || !out) return MCGPU_ERR_ARG;
  *out = nullptr;
  ctx->err.clear();
  if (n_slabs <= 0 || !slabs || !sigs || !absorption_rates || !weights_absorbed || !bank ||
      total_cells <= 0)
    return mc_fail(ctx, MCGPU_ERR_ARG, "batch: null pointer or empty batch");
  MC_HIP(ctx, hipSetDevice(ctx->device));
  mcgpu_batch *b = new mcgpu_batch();
  b->ctx = ctx;
  b->host_slabs.assign(slabs, slabs + n_slabs);
  mcgpu_default_options(&b->opt);
  if (opt) b->opt = *opt;
  b->sigs = sigs;
  b->ar = absorption_rates;
  b->weights = weights_absorbed;
  b->total_cells = total_cells;
  b->bank = *bank;
  b->result = result;
  std::vector<mc_slab_k> ks(n_slabs);
  int rc = MCGPU_OK;
  for (int s = 0; s < n_slabs && !rc; ++s) {
    const mcgpu_slab &h = slabs[s];
    const int m = mc_layer_cells(h.min_index, h.max_index);
    if (m <= 0 || h.n < 0 || h.cell_offset < 0 || h.cell_offset + m > total_cells ||
        h.particle_offset < 0)
      rc = mc_fail(ctx, MCGPU_ERR_ARG, "batch: invalid slab descriptor");
    ks[s].index_start = h.min_index;
    ks[s].m = m;
    ks[s].dx = h.dx;
    ks[s].min_weight = h.particle_min_weight;
    ks[s].cell_off = h.cell_offset;
    b->max_m = std::max(b->max_m, m);
    b->total_particles = std::max(b->total_particles, h.particle_offset + h.n);
  }
  if (!rc && b->total_particles > 0 &&
      (!bank->seed || !bank->x || !bank->mu || !bank->wmc || !bank->index))
    rc = mc_fail(ctx, MCGPU_ERR_ARG, "batch: bank has a null array");
#define B_HIP(call)                                                           \
  if (!rc) {                                                                  \
    hipError_t e_ = (call);                                                   \
    if (e_ != hipSuccess) rc = mc_fail(ctx, MCGPU_ERR_HIP, #call, e_);        \
  }
  B_HIP(hipMalloc(&b->d_slabs, sizeof(mc_slab_k) * n_slabs));
  B_HIP(hipMemcpy(b->d_slabs, ks.data(), sizeof(mc_slab_k) * n_slabs, hipMemcpyHostToDevice));
  B_HIP(hipMalloc(&b->d_cells, sizeof(mc_cell) * total_cells));
  B_HIP(hipMalloc(&b->d_fx, 16 * (size_t)total_cells));
  B_HIP(hipMalloc(&b->d_flags, 4 * (size_t)total_cells));
  B_HIP(hipMalloc(&b->d_ctr, MC_COUNTER_BYTES));
  B_HIP(hipHostMalloc(&b->h_ctr, sizeof(mc_counters), hipHostMallocDefault));
  B_HIP(hipStreamCreateWithFlags(&b->stream, hipStreamNonBlocking));
  B_HIP(hipEventCreate(&b->e0));
  B_HIP(hipEventCreate(&b->e1));
#undef B_HIP
  if (!rc) rc = batch_capture(b);
  if (rc) {
    mcgpu_batch_destroy(b);
    return rc;
  }
  *out = b;
  return MCGPU_OK;
}

int mcgpu_batch_run(mcgpu_batch *b, void *stream, mcgpu_stats *stats) {
  if (!b) return MCGPU_ERR_ARG;
  b->ctx->err.clear();
  MC_HIP(b->ctx, hipSetDevice(b->ctx->device));
  return batch_launch(b, reinterpret_cast<hipStream_t>(stream), stats);
}

int mcgpu_batch_options(const mcgpu_batch *b, mcgpu_options *opt) {
  if (!b || !opt) return MCGPU_ERR_ARG;
  *opt = b->opt;
  return MCGPU_OK;
}

int mcgpu_batch_autotune(mcgpu_batch *b, int32_t n_candidates, double *times_ms,
                         mcgpu_options *chosen) {
  if (!b) return MCGPU_ERR_ARG;
  mcgpu_context *ctx = b->ctx;
  ctx->err.clear();
  MC_HIP(ctx, hipSetDevice(ctx->device));
  struct cand {
    int block, ppl, refill;
  };
  /* the first: the automatic shape (tiles of a block's part, the interval
     adapted per wave) */
  static const cand cands[] = {{0, 0, 0},      {1024, 16, 8}, {1024, 4, 8},  {1024, 64, 8},
                               {1024, 16, 32}, {512, 16, 8},  {256, 64, 8},  {1024, 1, 8}};
  const int n_all = (int)(sizeof(cands) / sizeof(cands[0]));
  const int nc = n_candidates > 0 && n_candidates < n_all ? n_candidates : n_all;
  /* device copies of everything a run overwrites */
  const int64_t np = b->total_particles;
  void *save = nullptr;
  const size_t bank_bytes = (size_t)np * (8 + 8 + 8 + 8 + 4);
  const size_t w_bytes = 8 * (size_t)b->total_cells;
  MC_HIP(ctx, hipMalloc(&save, bank_bytes + w_bytes + 64));
  unsigned char *sv = (unsigned char *)save;
  auto snapshot = [&](bool restore) -> int {
    struct {
      void *p;
      size_t bytes;
    } parts[] = {{b->bank.seed, 8 * (size_t)np}, {b->bank.x, 8 * (size_t)np},
                 {b->bank.mu, 8 * (size_t)np},   {b->bank.wmc, 8 * (size_t)np},
                 {b->bank.index, 4 * (size_t)np}, {b->weights, w_bytes}};
    size_t off = 0;
    for (auto &pt : parts) {
      if (pt.bytes) {
        hipError_t e = restore ? hipMemcpyAsync(pt.p, sv + off, pt.bytes, hipMemcpyDeviceToDevice, b->stream)
                               : hipMemcpyAsync(sv + off, pt.p, pt.bytes, hipMemcpyDeviceToDevice, b->stream);
        if (e != hipSuccess) return mc_fail(ctx, MCGPU_ERR_HIP, "autotune snapshot", e);
      }
      off += pt.bytes;
    }
    hipError_t e = hipStreamSynchronize(b->stream);
    return e == hipSuccess ? MCGPU_OK : mc_fail(ctx, MCGPU_ERR_HIP, "autotune sync", e);
  };
  int rc = snapshot(false);
  double best = 1e300;
  int best_i = 0;
  const mcgpu_options base = b->opt;
  for (int i = 0; i < nc && !rc; ++i) {
    b->opt = base;
    b->opt.block_size = cands[i].block;
    b->opt.particles_per_lane = cands[i].ppl;
    b->opt.events_per_refill = cands[i].refill;
    b->opt.grid_blocks = 0;
    rc = batch_capture(b);
    mcgpu_stats st{};
    if (!rc) rc = batch_launch(b, b->stream, &st);
    if (!rc) rc = snapshot(true);
    if (times_ms) times_ms[i] = rc ? -1.0 : st.kernel_ms;
    if (!rc && st.kernel_ms < best) {
      best = st.kernel_ms;
      best_i = i;
    }
  }
  b->opt = base;
  b->opt.block_size = cands[best_i].block;
  b->opt.particles_per_lane = cands[best_i].ppl;
  b->opt.events_per_refill = cands[best_i].refill;
  b->opt.grid_blocks = 0;
  if (!rc) rc = batch_capture(b);
  (void)hipFree(save);
  if (!rc && chosen) *chosen = b->opt;
  return rc;
}

} /* extern "C" */
