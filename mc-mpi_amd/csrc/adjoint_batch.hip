/*
 * adjoint_batch.hip -- forward-with-scores and adjoint over many independent
 * slabs, one persistent launch each.
 *
 * The single-slab entry points (mcgpu_forward_cells, mcgpu_adjoint_cells)
 * fill the GPU when a slab has millions of histories; a batch of slabs shares
 * one launch instead, as the batched transport does:
 *  - the host cuts every slab's particles into tiles of particles_per_lane x
 *    block_size histories, or of a block's part (mc_tile_size), and orders
 *    them by their time (mc_tile_work), the longest first;
 *  - a persistent block takes the next tile from a global counter, stages the
 *    slab's cells, target weights and (zeroed) fixed-point accumulators in
 *    LDS when they fit (if not, the accumulators alone, or it adds straight into
 *    the global ones),
 *    runs the tile's histories with lanes refilled from an LDS counter, and
 *    adds its accumulators to the slab's global cells once per tile.
 * Per history the arithmetic is that of the single-slab kernels (the same
 * step, the same score and gradient terms in event order, exact sums), so
 * every slab's outputs are bit-identical to running it alone.
 *
 * Bound by the tiles' longest histories and, between them, by the LDS adds
 * (two a deposit, four a gradient event).  64 slabs of 1,000 cells and 50,000
 * histories: 45.6 -> 24.0 ms (forward 10.6, adjoint 13.5).
 */
#include <algorithm>
#include <vector>

#include "mc_adjoint.h"

namespace {

struct bslab_k {
  int32_t index_start;
  int32_t m;
  double dx;
  double min_weight;
  int64_t cell_off;
};

struct btile_k {
  int32_t slab;
  int32_t pad_;
  int64_t begin; /* absolute particle indices [begin, end) */
  int64_t end;
};

struct bcell_args {
  const bslab_k *slabs;
  const btile_k *tiles;
  int32_t n_tiles;
  int32_t lds_max_m;      /* slabs with m <= this stage their cells in LDS */
  uint32_t lds;           /* dynamic LDS bytes */
  mcgpu_bank bank;        /* forward: in/out; adjoint: initial bank, read only */
  const mc_cell *cells;   /* [total] */
  const double *g;        /* [total] */
  const double *score_in; /* adjoint: per-history scores, may be null */
  double *score_out;      /* forward: per-history scores, may be null */
  int8_t *result8;        /* forward: exit codes, may be null */
  unsigned long long *fx; /* forward: 2 words per cell; adjoint: 4 (ga lo, ga hi, gi lo, gi hi) */
  int64_t total;
  uint32_t *flags;        /* forward: [total]; adjoint: [2 total] */
  mc_counters *ctr;
  uint64_t max_events;
};

/* block-uniform: claim the next tile */
__device__ __forceinline__ int next_tile(mc_counters *ctr, int *s_tile) {
  if (threadIdx.x == 0) *s_tile = (int)atomicAdd(&ctr->next, 1ull);
  __syncthreads();
  return __builtin_amdgcn_readfirstlane(*s_tile);
}

/* a tile and its slab, every field wave-uniform */
struct btile {
  mc_layer_k L;
  int64_t cell_off;
  uint64_t begin, end;
};

__device__ __forceinline__ btile read_tile(const bcell_args &a, int t) {
  const btile_k tile = a.tiles[t];
  const bslab_k sl = a.slabs[__builtin_amdgcn_readfirstlane(tile.slab)];
  btile b;
  b.L.index_start = __builtin_amdgcn_readfirstlane(sl.index_start);
  b.L.m = __builtin_amdgcn_readfirstlane(sl.m);
  b.L.dx = mc_uniform(sl.dx);
  b.L.min_weight = mc_uniform(sl.min_weight);
  b.cell_off = (int64_t)mc_readlane64((unsigned long long)sl.cell_off, 0);
  b.begin = mc_readlane64((unsigned long long)tile.begin, 0);
  b.end = mc_readlane64((unsigned long long)tile.end, 0);
  return b;
}

template <bool SCORE> struct fwd_io {
  const bcell_args &a;
  double score;
  static constexpr bool RESUMES = false;
  __device__ __forceinline__ int code(const mc_state &p, bool at_cap, const mc_layer_k &L) {
    return mc_end_code(p, at_cap, L);
  }
  __device__ __forceinline__ uint64_t load(int64_t i, mc_state &p) {
    p.seed = a.bank.seed[i];
    p.x = a.bank.x[i];
    p.mu = a.bank.mu[i];
    p.wmc = a.bank.wmc[i];
    p.index = a.bank.index[i];
    score = 0.0;
    return 0;
  }
  __device__ __forceinline__ bool store(int64_t i, mc_state &p, int code, uint64_t ev, uint32_t) {
    if (a.result8) a.result8[i] = (int8_t)code;
    if (SCORE) a.score_out[i] = score;
    if (ev == 0) return false; /* its state stays as it came (store_state) */
    a.bank.seed[i] = p.seed;
    a.bank.x[i] = p.x;
    a.bank.mu[i] = p.mu;
    a.bank.wmc[i] = p.wmc;
    a.bank.index[i] = p.index;
    return false;
  }
};

/* Forward: mcgpu_forward_cells per slab.  Per tile as the batched transport
   (k_batched), with each history's score.  WIDE: some slabs' cells do not fit
   LDS beside the tally.  Those keep the tally there while it fits (10,135
   cells) and read cells and targets through L2: eight slabs of 4,080 cells and
   3,000 histories, with scores, 25.5 -> 7.3 ms; of 5,100, without, 23.0 -> 7.0. */
template <bool SCORE, bool WIDE>
__global__ __launch_bounds__(1024) void k_forward_cells_batch(bcell_args a, int refill_k) {
  extern __shared__ __align__(16) unsigned char smem[];
  __shared__ int s_tile;
  __shared__ mc_scale s_scale;
  __shared__ uint32_t s_thick;
  __shared__ unsigned long long s_next;
  __shared__ unsigned long long s_tot[MC_TOTALS];
  const int B = blockDim.x, tid = threadIdx.x;
  if (tid < MC_TOTALS) s_tot[tid] = 0;
  if (tid == 0) {
    mc_scale_clear(&s_scale);
    s_thick = 0;
  }
  double2 *tab = reinterpret_cast<double2 *>(smem);
  mc_tab_fill(tab);
  unsigned long long *t0 = reinterpret_cast<unsigned long long *>(smem + MC_TAB_BYTES);
  fwd_io<SCORE> io{a, 0.0};

  for (;;) {
    const int t = next_tile(a.ctr, &s_tile);
    if (t >= a.n_tiles) break;
    const btile b = read_tile(a, t);
    const int m = b.L.m;
    const bool in_lds = !WIDE || m <= a.lds_max_m; /* block-uniform */
    const int sh = in_lds ? mc_limbs_copies(m, a.lds - MC_TAB_BYTES - MC_PAD_BYTES -
                                                   (sizeof(mc_cell) + (SCORE ? 8 : 0)) * m)
                          : 0;
    const mc_limbs T = mc_limbs_at(t0, m, sh), mine = mc_limbs_mine(T);
    unsigned long long *t1 = t0 + m; /* words with carry: one copy */
    mc_cell *lc = reinterpret_cast<mc_cell *>(t0 + (2 * (size_t)m << sh));
    double *lg = reinterpret_cast<double *>(lc + m + 2);
    const bool lds_tally = WIDE && !in_lds && 16 * (int64_t)m <= (int64_t)a.lds - (int64_t)MC_TAB_BYTES;
    mc_full_tally F;
    F.t = t0;
    F.m = m;
    if (WIDE && lds_tally)
      for (int c = tid; c < 2 * m; c += B) t0[c] = 0;
    if (in_lds) {
      for (int c = tid; c < 2 * m << sh; c += B) t0[c] = 0;
      for (int c = tid; c < m; c += B) {
        if (SCORE) lg[c] = a.g[b.cell_off + c];
      }
      lc = mc_cells_fill(lc, a.cells + b.cell_off, m);
    }
    if (tid == 0) s_next = b.begin;
    {
      const uint64_t i = mc_scale_place(b.begin, b.end, tid, B);
      if (i < (uint64_t)b.end) atomicMax(&s_scale.w, mc_ceil_log2(a.bank.wmc[i]));
    }
    if ((in_lds || lds_tally) && m >= MC_THICK_CELLS)
      mc_scale_cells(&s_scale, a.cells + b.cell_off, m, b.L.dx);
    if (in_lds) mc_count_thick(&s_thick, a.cells + b.cell_off, m, b.L.dx);
    __syncthreads();

    const mc_walk_k K = mc_walk_live(b.L);
    const mc_block_tally bt = mc_block_tally_for(m, s_scale, B >> 6);
    mc_tile_queue queue{&s_next, b.end, false};
    unsigned long long *fx_lo = a.fx + b.cell_off, *fx_hi = fx_lo + a.total;
    uint32_t *flags = a.flags + b.cell_off;
    unsigned int *status = &a.ctr->status;
    const double *gg = SCORE ? a.g + b.cell_off : nullptr;
    if (WIDE && lds_tally) {
      F.B = bt;
      F.fx_lo = fx_lo;
      F.fx_hi = fx_hi;
      F.flags = flags;
      F.status = status;
      F.left = bt.every;
      mc_walk_bank<false>(io, queue, b.L, K, a.cells + b.cell_off, tab, refill_k, F.every(),
                   a.max_events, s_tot,
                   [&](mc_mask lanes, int c8, const mc_cell &, bool, double, double dw, double) {
                     F.add(lanes, c8, dw);
                     if (SCORE && mc_in(lanes)) io.score = io.score + *mc_word(gg, c8) * dw;
                   },
                   [&](int n) { F.moves(n); });
    } else if (!(WIDE && !in_lds) && bt.limbs) {
      auto limbs = [&](mc_mask lanes, int c8, const mc_cell &, bool, double, double dw, double) {
        mc_tally_limbs(mine, bt.S, fx_lo, fx_hi, flags, status, lanes, c8, dw);
        if (SCORE && mc_in(lanes)) io.score = io.score + *mc_word(lg, c8) * dw;
      };
      const mc_mover mover{T, fx_lo, fx_hi, m, bt.S.L, bt.every, bt.every};
      if (2 * s_thick > (uint32_t)m) /* block-uniform */
        mc_walk_bank<true, MC_IN_LDS, true>(io, queue, b.L, K, lc, tab, refill_k, bt.every,
                     a.max_events, s_tot, limbs, mover);
      else
        mc_walk_bank<true>(io, queue, b.L, K, lc, tab, refill_k, bt.every, a.max_events, s_tot, limbs,
                     mover);
    } else if (!WIDE || in_lds) { /* weights too heavy for the limbs */
      mc_walk_bank<true>(io, queue, b.L, K, lc, tab, refill_k, 1 << 30, a.max_events, s_tot,
                   [&](mc_mask lanes, int c8, const mc_cell &, bool, double, double dw, double) {
                     if (mc_in(lanes)) {
                       mc_tally(t0, t1, flags, status, c8 >> 3, dw);
                       if (SCORE) io.score = io.score + *mc_word(lg, c8) * dw;
                     }
                   },
                   [](int) {});
    } else {
      mc_walk_bank<false, MC_IN_MEMORY>(
                   io, queue, b.L, mc_walk_live<MC_IN_MEMORY>(b.L), a.cells + b.cell_off, tab,
                   refill_k, 1 << 30, a.max_events, s_tot,
                   [&](mc_mask lanes, int c, const mc_cell &, bool, double, double dw, double) {
                     if (mc_in(lanes)) {
                       mc_tally(fx_lo, fx_hi, flags, status, c, dw);
                       if (SCORE) io.score = io.score + gg[c] * dw;
                     }
                   },
                   [](int) {});
    }
    __syncthreads();
    if (WIDE && lds_tally) {
      F.out();
    } else if (!WIDE || in_lds) {
      if (bt.limbs)
        mc_limbs_move(T, bt.S.L, m, tid, B, fx_lo, fx_hi);
      else
        for (int c = tid; c < m; c += B)
          mc_fx_atomic_add(&fx_lo[c], &fx_hi[c], mc_fx{t0[c], t1[c]});
    }
    if (tid == 0) {
      mc_scale_clear(&s_scale);
      s_thick = 0;
    }
    __syncthreads();
  }
  if (tid == 0) mc_totals_out(s_tot, a.ctr, mc_counter_copy());
}

/* Adjoint: mcgpu_adjoint_cells per slab (replay from the initial bank).  WIDE
   as above (5,067 cells): eight slabs of 2,910 cells 22.1 -> 6.9 ms. */
template <bool HAVE_SCORE, bool WIDE>
__global__ __launch_bounds__(1024) void k_adjoint_cells_batch(bcell_args a, int refill_k) {
  extern __shared__ __align__(16) unsigned char smem[];
  __shared__ int s_tile;
  __shared__ mc_scale s_scale;
  __shared__ uint32_t s_thick;
  __shared__ unsigned long long s_next;
  __shared__ unsigned long long s_tot[MC_TOTALS];
  const int B = blockDim.x, tid = threadIdx.x;
  if (tid < MC_TOTALS) s_tot[tid] = 0;
  if (tid == 0) {
    mc_scale_clear(&s_scale);
    s_thick = 0;
  }
  double2 *tab = reinterpret_cast<double2 *>(smem);
  mc_tab_fill(tab);
  mc_grad_tally G;
  G.t = reinterpret_cast<unsigned long long *>(smem + MC_TAB_BYTES);
  G.stride = a.total;
  G.status = &a.ctr->status;
  mc_grad_io<HAVE_SCORE> io{a.bank, a.score_in, 0.0, 0.0, 1};

  for (;;) {
    const int t = next_tile(a.ctr, &s_tile);
    if (t >= a.n_tiles) break;
    const btile b = read_tile(a, t);
    const int m = b.L.m;
    const bool in_lds = !WIDE || m <= a.lds_max_m; /* block-uniform */
    const bool lds_tally = WIDE && !in_lds && 32 * (int64_t)m <= (int64_t)a.lds - (int64_t)MC_TAB_BYTES;
    mc_cell *lc = reinterpret_cast<mc_cell *>(G.t + 4 * (size_t)m);
    double *lg = reinterpret_cast<double *>(lc + m + 2);
    const double *gg = a.g + b.cell_off;
    G.fx = a.fx + b.cell_off;
    G.flags_a = a.flags + b.cell_off;
    G.flags_i = a.flags + a.total + b.cell_off;
    G.m = m;
    if (in_lds || lds_tally) {
      int kg = -1023;
      for (int c = tid; c < m; c += B) {
        for (int w = 0; w < 4; ++w) G.t[w * m + c] = 0;
        const double v = gg[c];
        if (in_lds) lg[c] = v;
        const int k = mc_ceil_log2(v);
        kg = k > kg ? k : kg;
      }
      atomicMax(&s_scale.g, kg);
      mc_scale_scatter(&s_scale, a.cells + b.cell_off, m);
      if (in_lds) mc_count_thick(&s_thick, a.cells + b.cell_off, m, b.L.dx);
      if (in_lds) lc = mc_cells_fill(lc, a.cells + b.cell_off, m);
    }
    if (tid == 0) s_next = b.begin;
    {
      const uint64_t i = mc_scale_place(b.begin, b.end, tid, B);
      if (i < (uint64_t)b.end) atomicMax(&s_scale.w, mc_ceil_log2(a.bank.wmc[i]));
    }
    __syncthreads();

    const mc_walk_k K = mc_walk_live(b.L);
    const bool limbs = mc_grad_split(G, s_scale, b.L.dx, B >> 6);
    mc_tile_queue queue{&s_next, b.end, false};
    auto add = [&](mc_mask lanes, int c8, const mc_cell &cell, bool coll, double di, double dw,
                   double wmc) {
      mc_grad_event<MC_GRAD_LIMBS>(io, G, lg, lanes, c8, cell, coll, di, dw, wmc);
    };
    if (in_lds && limbs && 2 * s_thick > (uint32_t)m) /* block-uniform */
      mc_walk_bank<true, MC_IN_LDS, true>(io, queue, b.L, K, lc, tab, refill_k, G.every,
                   a.max_events, s_tot, add, mc_grad_mover{G, G.every});
    else if (in_lds && limbs)
      mc_walk_bank<true>(io, queue, b.L, K, lc, tab, refill_k, G.every, a.max_events, s_tot, add,
                   mc_grad_mover{G, G.every});
    else if (in_lds)
      mc_walk_bank<true>(io, queue, b.L, K, lc, tab, refill_k, 1 << 30, a.max_events, s_tot,
                   [&](mc_mask lanes, int c8, const mc_cell &cell, bool coll, double di, double dw,
                       double wmc) {
                     mc_grad_event<MC_GRAD_CARRY>(io, G, lg, lanes, c8, cell, coll, di, dw, wmc);
                   },
                   [](int) {});
    else if (WIDE && lds_tally && limbs)
      mc_walk_bank<false>(io, queue, b.L, K, a.cells + b.cell_off, tab, refill_k, G.every,
                   a.max_events, s_tot,
                   [&](mc_mask lanes, int c8, const mc_cell &cell, bool coll, double di, double dw,
                       double wmc) {
                     mc_grad_event<MC_GRAD_LIMBS>(io, G, gg, lanes, c8, cell, coll, di, dw, wmc);
                   },
                   mc_grad_mover{G, G.every});
    else if (WIDE && lds_tally)
      mc_walk_bank<false>(io, queue, b.L, K, a.cells + b.cell_off, tab, refill_k, 1 << 30,
                   a.max_events, s_tot,
                   [&](mc_mask lanes, int c8, const mc_cell &cell, bool coll, double di, double dw,
                       double wmc) {
                     mc_grad_event<MC_GRAD_CARRY>(io, G, gg, lanes, c8, cell, coll, di, dw, wmc);
                   },
                   [](int) {});
    else if (WIDE)
      mc_walk_bank<false, MC_IN_MEMORY>(
                   io, queue, b.L, mc_walk_live<MC_IN_MEMORY>(b.L), a.cells + b.cell_off, tab,
                   refill_k, 1 << 30, a.max_events, s_tot,
                   [&](mc_mask lanes, int c, const mc_cell &cell, bool coll, double di, double dw,
                       double wmc) {
                     mc_grad_event<MC_GRAD_GLOBAL>(io, G, gg, lanes, c, cell, coll, di, dw, wmc);
                   },
                   [](int) {});
    __syncthreads();
    if (in_lds || lds_tally) mc_grad_move(G, tid, B, limbs);
    if (tid == 0) {
      mc_scale_clear(&s_scale);
      s_thick = 0;
    }
    __syncthreads();
  }
  if (tid == 0) { /* this call counts events alone */
    s_tot[1] = s_tot[2] = s_tot[3] = s_tot[4] = 0;
    mc_totals_out(s_tot, a.ctr, mc_counter_copy());
  }
}

/* cells from (sig_a, sig_i); zeroed accumulators (words per cell) and counters */
__global__ void k_batch_cells_setup(int64_t total, const double *sig_a, const double *sig_i,
                                    mc_cell *cells, unsigned long long *fx, int fx_words,
                                    uint32_t *flags, int flag_words, mc_counters *ctr) {
  const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (c < total) {
    mc_cell k;
    k.sig_a = sig_a[c];
    k.sig_i = sig_i[c];
    cells[c] = k;
    for (int w = 0; w < fx_words; ++w) fx[(size_t)w * total + c] = 0;
    for (int w = 0; w < flag_words; ++w) flags[(size_t)w * total + c] = 0;
  }
  mc_counters_clear(ctr, (uint64_t)c);
}

/* out_k[c] += the k-th accumulator (k < n_out) */
__global__ void k_batch_cells_finalize(int64_t total, const unsigned long long *fx,
                                       const uint32_t *flags, double *out0, double *out1,
                                       mc_counters *ctr, mc_counters *host_ctr) {
  mc_counters_fold(ctr, host_ctr);
  const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= total) return;
  out0[c] = out0[c] + mc_fx_finalize(fx[c], fx[total + c], flags[c]);
  if (out1) out1[c] = out1[c] + mc_fx_finalize(fx[2 * total + c], fx[3 * total + c], flags[total + c]);
}

/* Validates the slab table and builds the device slab and tile tables in
   ctx->tables; returns the largest slab's cell count in *max_m. */
int build_tables(mcgpu_context *ctx, int32_t n_slabs, const mcgpu_slab *slabs,
                 int64_t total_cells, int ppl, int block, int grid, const bslab_k **d_slabs,
                 const btile_k **d_tiles, int32_t *n_tiles, int *max_m, int64_t *max_particle) {
  std::vector<bslab_k> ks(n_slabs);
  std::vector<btile_k> tiles;
  std::vector<double> work;
  *max_m = 0;
  *max_particle = 0;
  const int64_t most = (int64_t)(ppl > 0 ? ppl : 16) * block;
  double share = 0.0; /* automatic: mc_tile_size */
  if (ppl <= 0)
    for (int s = 0; s < n_slabs; ++s)
      share += (double)slabs[s].n * ((double)slabs[s].max_index - slabs[s].min_index) / grid;
  for (int s = 0; s < n_slabs; ++s) {
    const mcgpu_slab &h = slabs[s];
    const int m = mc_layer_cells(h.min_index, h.max_index);
    if (m <= 0 || h.n < 0 || h.cell_offset < 0 || h.cell_offset + m > total_cells ||
        h.particle_offset < 0)
      return mc_fail(ctx, MCGPU_ERR_ARG, "batch: invalid slab descriptor");
    ks[s].index_start = h.min_index;
    ks[s].m = m;
    ks[s].dx = h.dx;
    ks[s].min_weight = h.particle_min_weight;
    ks[s].cell_off = h.cell_offset;
    *max_m = std::max(*max_m, m);
    *max_particle = std::max(*max_particle, h.particle_offset + h.n);
    const int64_t tile_size = ppl > 0 ? most : mc_tile_size(most, share, h.n, m, block);
    for (int64_t p0 = 0; p0 < h.n; p0 += tile_size) {
      btile_k t;
      t.slab = s;
      t.pad_ = 0;
      t.begin = h.particle_offset + p0;
      t.end = h.particle_offset + std::min(h.n, p0 + tile_size);
      tiles.push_back(t);
      work.push_back(mc_tile_work(t.end - t.begin, m));
    }
  }
  std::vector<size_t> order(tiles.size());
  for (size_t i = 0; i < order.size(); ++i) order[i] = i;
  std::stable_sort(order.begin(), order.end(), [&](size_t x, size_t y) { return work[x] > work[y]; });
  /* both tables in one copy */
  const size_t slab_bytes = (sizeof(bslab_k) * ks.size() + 255) / 256 * 256;
  std::vector<unsigned char> both(slab_bytes + sizeof(btile_k) * tiles.size());
  memcpy(both.data(), ks.data(), sizeof(bslab_k) * ks.size());
  for (size_t i = 0; i < order.size(); ++i)
    memcpy(both.data() + slab_bytes + sizeof(btile_k) * i, &tiles[order[i]], sizeof(btile_k));
  int rc = mc_ensure(ctx, &ctx->tables, &ctx->tables_bytes, both.size() + sizeof(btile_k));
  if (rc) return rc;
  unsigned char *base = (unsigned char *)ctx->tables;
  MC_HIP(ctx, hipMemcpy(base, both.data(), both.size(), hipMemcpyHostToDevice));
  *d_slabs = (const bslab_k *)base;
  *d_tiles = (const btile_k *)(base + slab_bytes);
  *n_tiles = (int32_t)tiles.size();
  return MCGPU_OK;
}

/* the counters that the finalizing kernel has handed over */
int read_batch_counters(mcgpu_context *ctx, hipStream_t s, mcgpu_stats *stats) {
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

/* o's block, grid and refill as batch_prepare set them */
template <typename K>
int launch_persistent(mcgpu_context *ctx, K kern, const bcell_args &a, const mcgpu_options &o,
                      size_t lds, hipStream_t s) {
  hipLaunchKernelGGL(kern, dim3(o.grid_blocks), dim3(o.block_size), lds, s, a, o.events_per_refill);
  MC_HIP(ctx, hipGetLastError());
  return MCGPU_OK;
}

/* the LDS for a slab's cells, beside the rows and the kernels' static LDS */
size_t batch_budget(const mcgpu_context *ctx) {
  return ctx->lds_per_block - 256 - MC_TAB_BYTES - MC_PAD_BYTES;
}

int largest_slab(int32_t n_slabs, const mcgpu_slab *slabs) {
  int m = 0;
  for (int s = 0; s < n_slabs; ++s)
    m = std::max(m, (int)mc_layer_cells(slabs[s].min_index, slabs[s].max_index));
  return m;
}

/* whether some slab's cells do not fit LDS */
bool batch_wide(const mcgpu_context *ctx, int32_t n_slabs, const mcgpu_slab *slabs,
                size_t lds_bytes_per_cell) {
  return (size_t)largest_slab(n_slabs, slabs) > batch_budget(ctx) / lds_bytes_per_cell;
}

/* Common set-up of both batched calls: options and launch shape of `kern`,
   tables, cells, accumulators, LDS size.  fx_words / flag_words: accumulator
   words per cell. */
template <typename K>
int batch_prepare(mcgpu_context *ctx, K kern, int32_t n_slabs, const mcgpu_slab *slabs,
                  int64_t total_cells, const mcgpu_bank *bank, const double *sig_a,
                  const double *sig_i, int fx_words, int flag_words, size_t lds_bytes_per_cell,
                  const mcgpu_options *opt, hipStream_t s, mcgpu_options *o, bcell_args *a,
                  size_t *lds) {
  mcgpu_default_options(o);
  if (opt) *o = *opt;
  if (o->block_size > 1024 || o->block_size % 64)
    return mc_fail(ctx, MCGPU_ERR_ARG, "block_size must be a multiple of 64 and <= 1024");
  memset(a, 0, sizeof *a);
  int max_m = largest_slab(n_slabs, slabs);
  /* LDS for the largest slab that fits; all of it if there are larger ones */
  const size_t budget = batch_budget(ctx);
  a->lds_max_m = (int)std::min<size_t>((size_t)max_m, budget / lds_bytes_per_cell);
  *lds = MC_TAB_BYTES + MC_PAD_BYTES +
         (max_m > a->lds_max_m ? budget : lds_bytes_per_cell * (size_t)a->lds_max_m);
  if (flag_words == 1) *lds = mc_lds_with_copies(*lds, a->lds_max_m); /* the forward */
  a->lds = (uint32_t)*lds;
  if (*lds > 65536)
    (void)hipFuncSetAttribute(reinterpret_cast<const void *>(kern),
                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)*lds);
  int per_cu = 0;
  if (o->block_size <= 0)
    o->block_size = mc_auto_block(ctx, kern, *lds, &per_cu);
  else if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kern, o->block_size, *lds) !=
               hipSuccess || per_cu < 1)
    per_cu = 1;
  const int block = o->block_size;
  if (o->grid_blocks <= 0) o->grid_blocks = per_cu * ctx->num_cus;
  if (o->events_per_refill < 0) o->events_per_refill = 0; /* 0: adaptive */
  int64_t max_particle = 0;
  int rc = build_tables(ctx, n_slabs, slabs, total_cells, o->particles_per_lane, block,
                        o->grid_blocks, &a->slabs, &a->tiles, &a->n_tiles, &max_m, &max_particle);
  if (rc) return rc;
  if (max_particle > 0 && (!bank->seed || !bank->x || !bank->mu || !bank->wmc || !bank->index))
    return mc_fail(ctx, MCGPU_ERR_ARG, "batch: bank has a null array");
  if ((rc = mc_ensure(ctx, &ctx->cells, &ctx->cells_bytes, sizeof(mc_cell) * (size_t)total_cells)))
    return rc;
  if ((rc = mc_ensure(ctx, &ctx->fx, &ctx->fx_bytes, 8 * (size_t)fx_words * total_cells))) return rc;
  if ((rc = mc_ensure(ctx, &ctx->flags, &ctx->flags_bytes, 4 * (size_t)flag_words * total_cells)))
    return rc;
  hipLaunchKernelGGL(k_batch_cells_setup, dim3((unsigned)((total_cells + 255) / 256)), dim3(256), 0,
                     s, total_cells, sig_a, sig_i, (mc_cell *)ctx->cells,
                     (unsigned long long *)ctx->fx, fx_words, (uint32_t *)ctx->flags, flag_words,
                     (mc_counters *)ctx->counters);
  MC_HIP(ctx, hipGetLastError());
  a->bank = *bank;
  a->cells = (const mc_cell *)ctx->cells;
  a->fx = (unsigned long long *)ctx->fx;
  a->total = total_cells;
  a->flags = (uint32_t *)ctx->flags;
  a->ctr = (mc_counters *)ctx->counters;
  a->max_events = o->max_events_per_history ? o->max_events_per_history : (1ULL << 27);
  return MCGPU_OK;
}

} // namespace

extern "C" {

int mcgpu_forward_cells_batch(mcgpu_context *ctx, int32_t n_slabs, const mcgpu_slab *slabs,
                              int64_t total_cells, const mcgpu_bank *bank, const double *sig_a,
                              const double *sig_i, double *weights_absorbed, const double *g,
                              double *history_score, int8_t *result, const mcgpu_options *opt,
                              mcgpu_stats *stats, void *stream) {
  if (!ctx) return MCGPU_ERR_ARG;
  ctx->err.clear();
  if (n_slabs <= 0 || !slabs || total_cells <= 0 || !bank || !sig_a || !sig_i ||
      !weights_absorbed || (history_score && !g))
    return mc_fail(ctx, MCGPU_ERR_ARG, "forward_cells_batch: bad arguments");
  MC_HIP(ctx, hipSetDevice(ctx->device));
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  mcgpu_options o;
  bcell_args a;
  size_t lds = 0;
  const bool score = history_score != nullptr;
  const int per_cell = score ? 40 : 32;
  const bool wide = batch_wide(ctx, n_slabs, slabs, per_cell);
  const auto kern = score ? (wide ? k_forward_cells_batch<true, true> : k_forward_cells_batch<true, false>)
                          : (wide ? k_forward_cells_batch<false, true> : k_forward_cells_batch<false, false>);
  int rc = batch_prepare(ctx, kern, n_slabs, slabs, total_cells, bank, sig_a, sig_i, 2, 1,
                         per_cell, opt, s, &o, &a, &lds);
  if (rc) return rc;
  a.g = g;
  a.score_out = history_score;
  a.result8 = result;
  MC_HIP(ctx, hipEventRecord(ctx->ev0, s));
  if (a.n_tiles > 0) {
    rc = launch_persistent(ctx, kern, a, o, lds, s);
    if (rc) return rc;
  }
  MC_HIP(ctx, hipEventRecord(ctx->ev1, s));
  hipLaunchKernelGGL(k_batch_cells_finalize, dim3((unsigned)((total_cells + 255) / 256)), dim3(256),
                     0, s, total_cells, (const unsigned long long *)ctx->fx,
                     (const uint32_t *)ctx->flags, weights_absorbed, (double *)nullptr, a.ctr,
                     (mc_counters *)ctx->host_counters);
  MC_HIP(ctx, hipGetLastError());
  return read_batch_counters(ctx, s, stats);
}

int mcgpu_adjoint_cells_batch(mcgpu_context *ctx, int32_t n_slabs, const mcgpu_slab *slabs,
                              int64_t total_cells, const mcgpu_bank *initial,
                              const double *sig_a, const double *sig_i, const double *g,
                              const double *history_score, double *grad_sig_a,
                              double *grad_sig_i, const mcgpu_options *opt, mcgpu_stats *stats,
                              void *stream) {
  if (!ctx) return MCGPU_ERR_ARG;
  ctx->err.clear();
  if (n_slabs <= 0 || !slabs || total_cells <= 0 || !initial || !sig_a || !sig_i || !g ||
      !grad_sig_a || !grad_sig_i)
    return mc_fail(ctx, MCGPU_ERR_ARG, "adjoint_cells_batch: bad arguments");
  MC_HIP(ctx, hipSetDevice(ctx->device));
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  mcgpu_options o;
  bcell_args a;
  size_t lds = 0;
  const bool wide = batch_wide(ctx, n_slabs, slabs, 56);
  const auto kern = history_score
                        ? (wide ? k_adjoint_cells_batch<true, true> : k_adjoint_cells_batch<true, false>)
                        : (wide ? k_adjoint_cells_batch<false, true> : k_adjoint_cells_batch<false, false>);
  int rc = batch_prepare(ctx, kern, n_slabs, slabs, total_cells, initial, sig_a, sig_i, 4, 2, 56, opt,
                         s, &o, &a, &lds);
  if (rc) return rc;
  a.g = g;
  a.score_in = history_score;
  MC_HIP(ctx, hipEventRecord(ctx->ev0, s));
  if (a.n_tiles > 0) {
    rc = launch_persistent(ctx, kern, a, o, lds, s);
    if (rc) return rc;
  }
  MC_HIP(ctx, hipEventRecord(ctx->ev1, s));
  hipLaunchKernelGGL(k_batch_cells_finalize, dim3((unsigned)((total_cells + 255) / 256)), dim3(256),
                     0, s, total_cells, (const unsigned long long *)ctx->fx,
                     (const uint32_t *)ctx->flags, grad_sig_a, grad_sig_i, a.ctr,
                     (mc_counters *)ctx->host_counters);
  MC_HIP(ctx, hipGetLastError());
  return read_batch_counters(ctx, s, stats);
}

} /* extern "C" */
