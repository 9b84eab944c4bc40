/*
 * internal.h -- shared definitions of the library's translation units:
 * the context, device counter block and kernel launchers.
 */
#ifndef MCGPU_INTERNAL_H
#define MCGPU_INTERNAL_H

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <string>

#include "../../include/mcgpu.h"
#include "mc_device.h"

/* Device-side counters of one transport call. */
struct mc_counters {
  unsigned long long next;       /* work-queue head (history kernel) */
  unsigned long long events;
  unsigned long long collisions;
  unsigned long long n_left;
  unsigned long long n_right;
  unsigned long long n_killed;
  unsigned int status;           /* bit 0: event cap hit, bit 1: tally range */
  unsigned int left;             /* windows: histories not known to be finished */
};

/* On the device the counters lie at the start of MC_COUNTER_BYTES, with more
   copies of the totals (events to n_killed) behind: blocks add to different
   ones (mc_counter_copy), and the call's last kernel folds them.  The
   adds of all blocks to one line follow one another: on 20,000 histories of a
   dozen events, a full grid of 1,024 blocks, they took 37 of 105 us. */
constexpr int MC_COUNTER_COPIES = 8;
constexpr size_t MC_COUNTER_STEP = 256; /* bytes; in different channels */
constexpr size_t MC_COUNTER_BYTES = MC_COUNTER_COPIES * MC_COUNTER_STEP;
constexpr unsigned MC_COUNTER_WORDS = sizeof(mc_counters) / 8;
static_assert(sizeof(mc_counters) == 56, "words 1 to 5 are the totals");

__device__ __forceinline__ unsigned long long *mc_counter_word(mc_counters *ctr, unsigned copy,
                                                               unsigned word) {
  return reinterpret_cast<unsigned long long *>(ctr) + copy * (MC_COUNTER_STEP / 8) + word;
}

/* the copy of a block's totals */
__device__ __forceinline__ unsigned mc_counter_copy() { return blockIdx.x % MC_COUNTER_COPIES; }

/* by a kernel's threads: word t of them all */
__device__ __forceinline__ void mc_counters_clear(mc_counters *ctr, uint64_t t) {
  if (t < MC_COUNTER_COPIES * MC_COUNTER_WORDS)
    *mc_counter_word(ctr, (unsigned)t / MC_COUNTER_WORDS, (unsigned)t % MC_COUNTER_WORDS) = 0;
}

/* By the call's last kernel: the copies' totals into the counters (the copies
   then hold zero), and the counters to the host (pinned memory; null: not),
   without a copy of their own. */
__device__ __forceinline__ void mc_counters_fold(mc_counters *ctr, mc_counters *host) {
  const unsigned t = threadIdx.x;
  if (blockIdx.x != 0 || blockIdx.y != 0 || t >= MC_COUNTER_WORDS) return;
  unsigned long long v = *mc_counter_word(ctr, 0, t);
  if (t >= 1 && t <= 5) {
    for (unsigned c = 1; c < MC_COUNTER_COPIES; ++c) v += *mc_counter_word(ctr, c, t);
    for (unsigned c = 1; c < MC_COUNTER_COPIES; ++c) *mc_counter_word(ctr, c, t) = 0;
    *mc_counter_word(ctr, 0, t) = v;
  }
  if (host) reinterpret_cast<unsigned long long *>(host)[t] = v;
}

/* the launch shape of a persistent kernel with so much LDS (mc_auto_block) */
struct mc_block_shape {
  const void *kern = nullptr;
  size_t lds = 0;
  int block = 0, per_cu = 0;
};

struct mcgpu_context {
  int device = 0;
  int num_cus = 0;
  size_t lds_per_block = 0;
  bool quiet = false; /* no error text (a stack context of the no-allocation entry point) */
  hipStream_t stream = nullptr;
  hipEvent_t ev0 = nullptr, ev1 = nullptr;
  std::string err;

  /* shapes found by the last calls, the oldest replaced */
  mc_block_shape shapes[8];
  unsigned next_shape = 0;

  /* grow-only scratch (device) */
  void *cells = nullptr;      size_t cells_bytes = 0;     /* mc_cell[m] */
  void *fx = nullptr;         size_t fx_bytes = 0;        /* u64[2m] tally */
  void *flags = nullptr;      size_t flags_bytes = 0;     /* u32[m] */
  void *counters = nullptr;                               /* mc_counters */
  void *host_counters = nullptr;                          /* pinned mc_counters */
  void *aos = nullptr;        size_t aos_bytes = 0;       /* staging mcgpu_particle[n] */
  void *res32 = nullptr;      size_t res32_bytes = 0;     /* int32[n] */
  void *sig_in = nullptr;     size_t sig_in_bytes = 0;    /* double[2m] sigs, ar */
  void *w_in = nullptr;       size_t w_in_bytes = 0;      /* double[m] weights */
  void *work = nullptr;       size_t work_bytes = 0;      /* event kernel banks */
  void *tables = nullptr;     size_t tables_bytes = 0;    /* batched calls: slab + tile tables */
};

/* the cells of a layer [min_index, max_index): 0 if there are none, or more than
   the 2^31 - 1 that its 32-bit cell numbers take */
static inline int32_t mc_layer_cells(int32_t min_index, int32_t max_index) {
  const int64_t m = (int64_t)max_index - min_index;
  return m > 0 && m <= INT32_MAX ? (int32_t)m : 0;
}

/* grow-only device buffer */
int mc_ensure(mcgpu_context *ctx, void **buf, size_t *cap, size_t need);
int mc_fail(mcgpu_context *ctx, int status, const char *what, hipError_t e = hipSuccess);
#define MC_HIP(ctx, call)                                          \
  do {                                                             \
    hipError_t e_ = (call);                                        \
    if (e_ != hipSuccess) return mc_fail((ctx), MCGPU_ERR_HIP, #call, e_); \
  } while (0)

/* Arguments common to the transport kernels. */
struct mc_transport_args {
  mc_layer_k L;
  int64_t n;
  mcgpu_particle *aos; /* exactly one of aos / soa is used */
  mcgpu_bank soa;
  const mc_cell *cells;
  unsigned long long *fx; /* [2m]: lo words then hi words */
  uint32_t *flags;
  int8_t *result8;
  int32_t *result32;
  uint64_t *events;
  uint64_t *collisions;
  mc_counters *ctr;
  uint64_t max_events;
  const double *g; /* optional per-cell target weights (history kernel) */
  double *score;   /* optional per-history sum of g[c] * dw, in event order */
};

/* particle i of the call's bank (AoS staging or SoA device bank) */
static __device__ __forceinline__ void load_state(const mc_transport_args &a, int64_t i, mc_state &p) {
  if (a.aos) {
    const mcgpu_particle *q = a.aos + i;
    p.seed = q->seed;
    p.x = q->x;
    p.mu = q->mu;
    p.wmc = q->wmc;
    p.index = q->index;
  } else {
    p.seed = a.soa.seed[i];
    p.x = a.soa.x[i];
    p.mu = a.soa.mu[i];
    p.wmc = a.soa.wmc[i];
    p.index = a.soa.index[i];
  }
}

/* moved: the history had an event; else its state in the bank stays as it came
   (the walk keeps 63 bits of the seed) */
static __device__ __forceinline__ void store_state(const mc_transport_args &a, int64_t i,
                                            const mc_state &p, int code, bool moved) {
  if (a.aos) {
    if (a.result32) a.result32[i] = code;
    if (!moved) return;
    mcgpu_particle *q = a.aos + i;
    q->seed = p.seed;
    q->x = p.x;
    q->mu = p.mu;
    q->wmc = p.wmc;
    q->index = p.index;
  } else {
    if (a.result8) a.result8[i] = (int8_t)code;
    if (!moved) return;
    a.soa.seed[i] = p.seed;
    a.soa.x[i] = p.x;
    a.soa.mu[i] = p.mu;
    a.soa.wmc[i] = p.wmc;
    a.soa.index[i] = p.index;
  }
}

/* Threads per block of a persistent kernel with `lds` bytes of dynamic LDS
   per block, when the caller gave none: of 256, 512 and 1024, the one with
   the most resident waves per CU by the occupancy calculator (which counts
   registers and LDS); ties go to the smaller block.  With LDS-resident
   tables a small block can leave most of the CU idle: 56 KB per block fits
   two blocks in 160 KB, 8 waves at 256 threads but 16 at 512.
   *per_cu receives the resident blocks per CU of the choice (at least 1).
   The context keeps the last shapes: the calculator's three answers take some
   10 us of a small call's 300. */
template <typename K>
static inline int mc_auto_block(mcgpu_context *ctx, K kern, size_t lds, int *per_cu) {
  const void *key = reinterpret_cast<const void *>(kern);
  for (const mc_block_shape &s : ctx->shapes)
    if (s.kern == key && s.lds == lds) {
      *per_cu = s.per_cu;
      return s.block;
    }
  int best = 256, best_waves = -1, best_per_cu = 1;
  for (int b = 256; b <= 1024; b *= 2) {
    int pc = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&pc, kern, b, lds) != hipSuccess) {
      (void)hipGetLastError();
      pc = 0;
    }
    const int waves = pc * (b / 64);
    if (waves > best_waves) {
      best = b;
      best_waves = waves;
      best_per_cu = pc > 0 ? pc : 1;
    }
  }
  *per_cu = best_per_cu;
  if (best_waves > 0) ctx->shapes[ctx->next_shape++ % 8] = {key, lds, best, best_per_cu};
  return best;
}

/* Blocks of a persistent kernel for n histories in a layer of m cells: all that
   the chip holds, a block per history at most, so that few histories spread over
   it.  In a layer of a few cells all blocks move their tallies to the same words,
   one after the other, and histories are short: one block per CU while that is a
   wave per SIMD.  One cell, 20,000 histories, by a full grid and so, in us: 48 and
   26 (1 event each), 82 and 70 (42); their gradients 86 and 47, 280 and 255.  Ten
   cells 109 and 105, 64 cells 255 and 280. */
static inline int mc_auto_grid(const mcgpu_context *ctx, int m, int64_t n, int per_cu) {
  int grid = per_cu * ctx->num_cus;
  if (m <= 8 && n <= 256 * (int64_t)ctx->num_cus) grid = ctx->num_cus;
  return n < grid ? (int)(n > 0 ? n : 1) : grid;
}

/* sweep: 0, or, where ctr->left is not 0 after it, the number of the sweep over a
   wide layer's windows that goes on with the histories left */
int mc_launch_history(mcgpu_context *ctx, const mc_transport_args &a, const mcgpu_options &o,
                      hipStream_t s, int sweep = 0);

/* The steps of one transport call around the kernel (capi.hip), on buffers
   the caller provides:
   mc_launch_setup:    cells[c] = (sigs*ar, sigs*(1-ar)), tally words and
                       flags of m cells and the counter block zeroed (a
                       kernel, no memset);
   mc_launch_finalize: weights[c] += the tally of cell c, rounded once, unless
                       ctr->left; the counters to host_ctr (pinned) if given;
   mc_status_from_counters: stats from the counter block read back (with
                       the kernel time given) and the call's status. */
int mc_launch_setup(mcgpu_context *ctx, int m, const double *sigs, const double *ar,
                    mc_cell *cells, unsigned long long *fx, uint32_t *flags, mc_counters *ctr,
                    hipStream_t s);
int mc_launch_finalize(mcgpu_context *ctx, int m, const unsigned long long *fx,
                       const uint32_t *flags, double *weights, mc_counters *ctr,
                       mc_counters *host_ctr, hipStream_t s);
int mc_status_from_counters(mcgpu_context *ctx, const mc_counters &hc, float kernel_ms,
                            mcgpu_stats *stats);

/* Device properties and the address of the no-allocation entry point's
   scratch array on the current device, set up once per device (noalloc.hip;
   also called by mcgpu_context_create for its device). */
int mc_noalloc_device_setup(int device);
int mc_launch_event(mcgpu_context *ctx, const mc_transport_args &a, const mcgpu_options &o,
                    hipStream_t s);

/* Particles first .. first+n-1 of a lazy source (Layer::create_particles,
   src/layer.cpp:89-121) into bank[0..n), on stream s (capi.hip). */
int mc_launch_create(mcgpu_context *ctx, uint64_t seed, int64_t first, int64_t n, double x_ini,
                     double wmc, int32_t index, const mcgpu_bank &bank, hipStream_t s);

/* The batched transport (batched.hip): a persistent launch over a work
   queue of tiles, each a particle range [begin, end) of the bank belonging
   to one slab (a layer: global cell range, dx, min weight, offset of its
   cells in the concatenated cell / tally arrays). */
struct mc_slab_k {
  int32_t index_start;
  int32_t m;
  double dx;
  double min_weight;
  int64_t cell_off;
};

struct mc_tile_k {
  int32_t slab;
  int32_t pad_;
  int64_t begin; /* absolute particle indices [begin, end) */
  int64_t end;
};

struct mc_batched_shape {
  int block, grid, refill;
  size_t lds;          /* dynamic LDS bytes per block */
  int lds_cells_max_m; /* slabs with m <= this stage their cells in LDS */
  int lds_tally_max_m; /* slabs with m <= this keep their tally in LDS */
  bool wide;           /* some slab's tally does not fit beside the rows */
};

/* Histories of a tile of a slab of n histories and m cells: n in equal tiles
   of at most `most`, or, when `share` (a block's part of all slabs' histories
   x cells) is given, of at most that part (few or uneven slabs), up to four
   times `most` where that is a quarter of the part (many), though of at least
   one history per four threads.  So there are at most as many tiles as blocks,
   and n / most and one for each slab.
   A block waits for its tile's longest history, several times the mean one,
   so small tiles cost more than they balance.  In tiles of 4/3, 1, 1/1.3, 1/2
   and 1/3 of a part: 512 slabs of 32 to 8,192 cells 39.8, 39.3, 41.8, 45.5 and
   46.5 ms; forward and adjoint of 64 slabs of 50,000 histories on 1,000 cells
   27.1, 24.3, 26.0, 28.0 and 29.5 ms; the cycle loop of 20 cycles of 100,000
   histories with one rank 8.7 ms in whole parts, 9.2 in halves, 13.3 in tiles
   of 4,096 (half the blocks without one).  4,096 slabs of 5.8e8 histories 2.56
   s with `most` (16 a thread) and 2.36 with up to four times that, where 512
   slabs lose without the quarter (32.3 and 37.4 ms).  A quarter of a CU's
   waves run twice as fast as all of them: 120 slabs of 20 to 2,000 histories
   15.2 ms with at least one history per thread, 11.5 with one per four. */
inline int64_t mc_tile_size(int64_t most, double share, int64_t n, int m, int block) {
  double fit = (double)most;
  if (share > 0.0) {
    const double part = share / m;
    if (part / 4.0 > fit) fit = part / 4.0 < 4.0 * fit ? part / 4.0 : 4.0 * fit;
    if (part < fit) fit = part;
  }
  if (fit < (double)block / 4) fit = (double)block / 4;
  const int64_t tiles = (int64_t)((double)n / fit) + ((double)n / fit > (int64_t)((double)n / fit));
  if (tiles <= 1) return n > 0 ? n : 1;
  return ((n + tiles - 1) / tiles + 63) / 64 * 64;
}

/* What tiles are sorted by, the largest first: about the time of a tile of n
   histories of m cells, whose longest history counts as much as some 10,000
   mean ones do on a full block, and whose collisions, load and store as much
   as some 240 crossings each.  Sorted by n m, small tiles of many cells came
   last and the whole launch waited for them: 512 slabs 38.7 -> 32.6 ms, 80
   slabs 14.3 -> 10.5 ms (1,000, 3,000 and 30,000 in place of 10,000: the
   same). */
inline double mc_tile_work(int64_t n, int m) { return ((double)n + 1e4) * ((double)m + 240.0); }

/* Launch shape for slabs of up to max_m cells; block 0 takes the size with
   the most resident waves, grid <= 0 resident blocks per CU x CUs. */
int mc_batched_plan_shape(mcgpu_context *ctx, int max_m, int block, int grid, int refill,
                          mc_batched_shape *out);
/* One launch over n_tiles tiles; fx / flags / ctr must be zeroed first
   (ctr->next is the tile queue head). */
int mc_launch_batched(mcgpu_context *ctx, const mc_batched_shape &sh, const mc_slab_k *slabs,
                      const mc_tile_k *tiles, int32_t n_tiles, const mcgpu_bank &bank,
                      const mc_cell *cells, unsigned long long *fx, int64_t total_cells,
                      uint32_t *flags, int8_t *result8, mc_counters *ctr, uint64_t max_events,
                      hipStream_t s);

#endif
