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
 * block handled which history.  Layers too large for LDS are transported in
 * windows (below).  The per-cell cross-section pairs are staged
 * in LDS when they fit next to the tally, otherwise read through L2.
 *
 * Measured against the kernel with the full event and a tally with carry: a lone
 * history 450 -> 284 ns per event (10,000 cells); 1,000 histories on the
 * 100-cell slab, whole call 264 -> 175 us; 1,000 on 10,000 cells 26.0 -> 9.4
 * ms (dealt over the CUs); 8e6 on 10,000 cells 267 -> 160 ms (4.9e11 events/s,
 * tally and cells in LDS: its pipe and the vector instructions, some 58 cycles
 * of a CU for a wave's event each, of 80 in all); 2e6 into a 1,000-cell layer
 * 11.7 -> 4.9 ms.
 */
#include "internal.h"
#include <algorithm>

#include "mc_ring.h"
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
    store_state(a, i, p, code, ev != 0);
    if (a.events) a.events[i] = ev;
    if (a.collisions) a.collisions[i] = col;
    if (SCORE) a.score[i] = score;
    return false;
  }
};

/* ------------------------------------------------------------- wide layers
   A layer of more cells than a block's LDS tally holds is cut into windows
   whose cells and tally fit; each block transports the histories of one
   window.  A history that crosses into another window is parked: its state
   goes to memory and its number into that window's ring, from which the
   window's blocks refill their lanes.  A block that has run dry, or has few
   histories left while many wait elsewhere, empties its tally, parks what it
   has and takes the window with the most waiting histories per block.  So all
   windows are worked at once, wherever the histories are, and the whole call
   is one launch; a history crosses a window's edge a few times at most
   (windows are thousands of cells, flights a good part of the layer).
   Histories whose ring slot was lost (a full ring, a wave that gave up
   waiting for it) are found by the next sweep; usually there is none.
   Measured against a global tally (two returning atomics in memory per event)
   and against sweeps in which a parked history waits for the next launch:
   200,000 histories on 20,000 cells 540, 106 and 45 ms; 2 M 161 ms (228 by
   sweeps); 200,000 on 50,000 cells 102 ms (236); 1,000 on 20,000 21.6 ms (56).
   With histories that set out apart the first two take 36 and 123 ms; the
   first then lasts little longer than its longest history (89,000 events).
   Histories taken up together at an edge set out one event apart (mc_walk.h);
   before, they met in the LDS banks, and 8 M histories on 10,000 cells took
   208 ms in two windows (now 161; 234 in one, whose cells do not fit). */
constexpr int MC_MAX_WINDOWS = 64;

/* between rings, which would otherwise lie a power of two apart: 8 M histories
   on 10,000 cells 169.8 ms without, 163.4 with (163.3 with rings of as many
   slots as histories) */
constexpr uint32_t MC_RING_PAD = 1056;

struct mc_windows {
  int32_t nw, W;            /* window w: cells [w W, (w + 1) W) of the layer */
  uint32_t *count;          /* [nw] histories at the sweep's start */
  unsigned long long *next; /* [nw] queue counters */
  const uint32_t *list;     /* those histories, by window */
  int32_t *at;              /* [n] the cell of a parked history, -1 when finished */
  uint64_t *ev;             /* [n] its events so far */
  /* histories parked in the course of a sweep: window w's are a ring of cap
     slots (mc_ring.h) at ring(w), put[w] - got[w] of them waiting */
  uint32_t *parked, *put, *got; /* [nw (cap + MC_RING_PAD)], [nw], [nw] */
  uint32_t *blocks;             /* [nw] blocks that transport window w */
  uint32_t *left;               /* histories not known to be finished */
  uint32_t *thick;              /* thick cells, or null: not asked (k_history_if_thick) */
  uint32_t cap;
  int patience; /* looks of an idle block before it ends */
  __device__ __forceinline__ uint32_t *ring(int w) const {
    return parked + (size_t)w * (cap + MC_RING_PAD);
  }
};
constexpr uint32_t MC_NOT_PUT = 0xFFFFFFFFu;

/* histories x windows of a call with rings at most (2 GiB, 4 GiB where the
   histories are just above a power of two) */
constexpr size_t MC_RING_WORDS = (size_t)1 << 29;

/* words of different windows lie on different lines */
constexpr int MC_WINDOW_STEP = 32;

/* LDS words of a block */
struct mc_window_block {
  unsigned long long run; /* the block's run of parked histories (mc_ring.h) */
  unsigned int looked;    /* clock of the last look at the windows' counts */
  int looking;
  int busy;               /* lanes with a history */
  int leave;              /* the block parks its histories and takes another window */
  uint32_t done;          /* histories finished */
  int w;                  /* the window chosen */
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

/* Words that another block may have written, or will read, within the sweep:
   past the caches of this XCD (agent scope) */
template <typename T> __device__ __forceinline__ T ld_shared(const T *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename T> __device__ __forceinline__ void st_shared(T *p, T v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

template <typename T> __device__ __forceinline__ T ld_block(const T *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

template <bool SCORE> struct window_io {
  static constexpr bool RESUMES = true;
  const mc_transport_args &a;
  const mc_windows &win;
  int32_t w; /* the block's window */
  mc_window_block *blk;
  double score;
  int to; /* cell a history is parked in, -1: finished */
  __device__ __forceinline__ uint64_t load(int64_t j, mc_state &p) {
    if (a.aos) {
      const mcgpu_particle *q = a.aos + j;
      p.seed = ld_shared(&q->seed);
      p.x = ld_shared(&q->x);
      p.mu = ld_shared(&q->mu);
      p.wmc = ld_shared(&q->wmc);
      p.index = ld_shared(&q->index);
    } else {
      p.seed = ld_shared(&a.soa.seed[j]);
      p.x = ld_shared(&a.soa.x[j]);
      p.mu = ld_shared(&a.soa.mu[j]);
      p.wmc = ld_shared(&a.soa.wmc[j]);
      p.index = ld_shared(&a.soa.index[j]);
    }
    if (SCORE) score = ld_shared(&a.score[j]);
    return ld_shared(&win.ev[j]);
  }
  __device__ __forceinline__ int code(const mc_state &p, bool at_cap, const mc_layer_k &) {
    to = mc_alive(p, a.L) && !at_cap ? p.index - a.L.index_start : -1;
    return to >= 0 ? 3 : mc_end_code(p, at_cap, a.L);
  }
  __device__ __forceinline__ bool store(int64_t j, mc_state &p, int code, uint64_t ev,
                                        uint32_t col) {
    if (a.collisions) st_shared(&a.collisions[j], ld_shared(&a.collisions[j]) + col);
    if (SCORE) st_shared(&a.score[j], score);
    if (to < 0) {
      store_state(a, j, p, code, ev != 0);
      if (a.events) a.events[j] = ev;
      win.at[j] = -1;
      atomicAdd(&blk->done, 1u);
      return false;
    }
    if (a.aos) {
      mcgpu_particle *q = a.aos + j;
      st_shared(&q->seed, p.seed);
      st_shared(&q->x, p.x);
      st_shared(&q->mu, p.mu);
      st_shared(&q->wmc, p.wmc);
      st_shared(&q->index, p.index);
    } else {
      st_shared(&a.soa.seed[j], p.seed);
      st_shared(&a.soa.x[j], p.x);
      st_shared(&a.soa.mu[j], p.mu);
      st_shared(&a.soa.wmc[j], p.wmc);
      st_shared(&a.soa.index[j], p.index);
    }
    st_shared(&win.ev[j], ev);
    st_shared(&win.at[j], (int32_t)to);
    /* all of it in memory before the history's number can be seen there */
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    const int32_t v = to / win.W;
    if (win.cap) {
      put(j, v, v < w);
      put(j, v, v == w);
      put(j, v, v > w);
    }
    return false;
  }
  /* the lanes with `mine`, all of the same window v */
  __device__ __forceinline__ void put(int64_t j, int32_t v, bool mine) {
    if (!mine) return;
    const mc_mask lanes = mc_lanes(true);
    const uint32_t rank = (uint32_t)mc_mbcnt64(lanes);
    uint32_t base = 0;
    if (rank == 0) base = atomicAdd(&win.put[v * MC_WINDOW_STEP], (uint32_t)__popcll(lanes));
    base = (uint32_t)__builtin_amdgcn_readfirstlane((int)base);
    st_shared(win.ring(v) + mc_ring_slot(base + rank, win.cap), (uint32_t)j);
  }
};

/* the parked histories of window v (0: none), read past the caches */
__device__ __forceinline__ uint32_t mc_window_waiting(const mc_windows &win, int v) {
  const uint32_t got = ld_shared(win.got + v * MC_WINDOW_STEP);
  const uint32_t have = ld_shared(win.put + v * MC_WINDOW_STEP) - got;
  return (int32_t)have > 0 ? have : 0u;
}

/* `want` of a window's parked histories, or a share of many, for a block (by
   one lane): its run, 0 if there are none */
__device__ __forceinline__ unsigned long long mc_window_claim(const mc_windows &win, int w,
                                                              uint32_t want) {
  uint32_t *got = win.got + w * MC_WINDOW_STEP;
  uint32_t at = ld_shared(got);
  for (int t = 0; t < 8; ++t) {
    const uint32_t have = ld_shared(win.put + w * MC_WINDOW_STEP) - at;
    if ((int32_t)have <= 0) return 0;
    const uint32_t share = have / (2u * gridDim.x);
    uint32_t size = share > want ? share : want;
    size = size < have ? size : have;
    const uint32_t was = atomicCAS(got, at, at + size);
    if (was == at) return mc_ring_run(at, size);
    at = was;
  }
  return 0;
}

/* A wave's histories of a window: those of its list, then those parked in it
   meanwhile.  Nothing waits long for a history to be parked: one that no wave
   takes is in the next sweep's list. */
struct mc_window_queue {
  static constexpr bool LEAVES = true;
  mc_call_queue open; /* none after the block's first window */
  const uint32_t *list;
  const mc_windows &win;
  mc_window_block *blk;
  int32_t w;
  int lanes; /* of the wave, counted in blk->busy */
  bool starved;
  __device__ __forceinline__ bool more() const { return true; }
  __device__ __forceinline__ int least() const { return starved ? 64 : 8; }
  __device__ __forceinline__ int64_t take(mc_mask need) {
    int64_t j = -1;
    if (open.more()) { /* wave-uniform */
      const int64_t i = open.take(need);
      if (mc_in(need) && i >= 0) j = list[i];
      need &= ~mc_lanes(j >= 0);
      if (need == 0 || open.more()) return j;
    }
    const uint32_t cnt = (uint32_t)__popcll(need);
    uint32_t next = 0, have = 0;
    if (__lane_id() == 0 && win.cap) {
      if (mc_ring_left(ld_block(&blk->run)) != 0) {
        const unsigned long long run = atomicAdd(&blk->run, (unsigned long long)cnt);
        next = mc_ring_next(run);
        have = mc_ring_left(run);
      }
    }
    next = (uint32_t)__builtin_amdgcn_readfirstlane((int)next);
    have = (uint32_t)__builtin_amdgcn_readfirstlane((int)have);
    const uint32_t rank = (uint32_t)mc_mbcnt64(need);
    starved = have < cnt;
    if (mc_in(need) && rank < have) {
      uint32_t *slot = win.ring(w) + mc_ring_slot(next + rank, win.cap);
      uint32_t v = MC_NOT_PUT;
      /* put[] counts it, so its number is on the way; if it does not come in
         time, it stays for the next sweep */
      for (int t = 0; t < 1024 && v == MC_NOT_PUT; ++t) v = ld_shared(slot);
      if (v != MC_NOT_PUT) v = atomicExch(slot, MC_NOT_PUT);
      if (v != MC_NOT_PUT) j = v;
    }
    return j;
  }
  /* counts the wave's lanes in use; when the block's run is used up, one wave
     every 40,000 cycles takes another, or finds that the block had better
     leave for another window.  Returns whether the wave is to park its
     histories and leave. */
  __device__ __forceinline__ bool leave(int used) {
    if (used != lanes) {
      if (__lane_id() == 0) atomicAdd(&blk->busy, used - lanes);
      lanes = used;
    }
    if (starved && win.cap) look();
    return __builtin_amdgcn_readfirstlane(ld_block(&blk->leave)) != 0 && !open.more();
  }
  __device__ __forceinline__ bool has_run() const {
    return mc_ring_left(ld_block(&blk->run)) != 0;
  }
  __device__ __forceinline__ void look() {
    const unsigned int now = (unsigned int)__builtin_readcyclecounter();
    int mine = 0;
    if (__lane_id() == 0) {
      if ((int32_t)(now - ld_block(&blk->looked)) > 40000 && atomicCAS(&blk->looking, 0, 1) == 0) {
        mine = !has_run() && ld_block(&blk->leave) == 0; /* under the lock: no other wave claims */
        if (!mine) atomicExch(&blk->looking, 0);
      }
    }
    if (!__builtin_amdgcn_readfirstlane(mine)) return;
    const int v = (int)__lane_id();
    const int busy = __builtin_amdgcn_readfirstlane(ld_block(&blk->busy));
    const int idle = (int)blockDim.x - busy;
    const uint32_t have = v < win.nw ? mc_window_waiting(win, v) : 0u;
    if (v == 0) blk->looked = now;
    if (mc_lanes(v == w && have != 0)) {
      if (v == 0) {
        const unsigned long long run = mc_window_claim(win, w, idle > 64 ? (uint32_t)idle : 64u);
        if (run) atomicExch(&blk->run, run);
      }
    } else if (busy * 4 < (int)blockDim.x) {
      const uint32_t least = busy > 128 ? 4u * (uint32_t)busy : 512u;
      if (mc_lanes(have >= least) && v == 0) atomicExch(&blk->leave, 1);
    }
    if (v == 0) atomicExch(&blk->looking, 0);
  }
  /* with no history: whether the block still transports some of the window */
  __device__ __forceinline__ bool wait() const {
    if (win.cap == 0) return false;
    if (__builtin_amdgcn_readfirstlane(has_run())) return true;
    if (__builtin_amdgcn_readfirstlane(ld_block(&blk->busy)) == 0) return false;
    __builtin_amdgcn_s_sleep(127);
    return true;
  }
};

/* by the first wave of a block without histories: a window with parked ones
   and a run of them, in blk; blk->w = -1: none came up while the block waited */
__device__ __forceinline__ void mc_window_choose(const mc_windows &win, mc_window_block *blk) {
  const int v = (int)__lane_id();
  int chosen = -1;
  unsigned long long run = 0;
  for (int t = 0; t < win.patience; ++t) { /* wave-uniform */
    uint64_t key = 0;
    if (v < win.nw) {
      const uint32_t have = mc_window_waiting(win, v);
      const uint32_t there = ld_shared(win.blocks + v * MC_WINDOW_STEP);
      if (have) key = ((((uint64_t)have << 6) / (there + 1u) + 1u) << 8) | (uint64_t)v;
    }
    const uint64_t best = mc_wave_max_u64(key);
    if (best) {
      const int w = __builtin_amdgcn_readfirstlane((int)(best & 255u));
      if (v == 0) {
        run = mc_window_claim(win, w, blockDim.x);
        if (run) atomicAdd(&win.blocks[w * MC_WINDOW_STEP], 1u);
      }
      if (mc_readlane64(run, 0)) {
        chosen = w;
        break;
      }
    } else {
      if (__builtin_amdgcn_readfirstlane((int)ld_shared(win.left)) <= 0) break;
      for (int r = 0; r < 10; ++r) __builtin_amdgcn_s_sleep(127);
    }
  }
  if (v == 0) {
    blk->w = chosen;
    blk->run = run;
    blk->busy = blk->leave = 0;
  }
}

__global__ void k_windows_clear(mc_windows win, uint32_t *cursor) {
  const int t = threadIdx.x;
  if (t >= win.nw) return;
  win.count[t] = 0;
  cursor[t] = 0;
  win.next[t] = 0;
  win.put[t * MC_WINDOW_STEP] = win.got[t * MC_WINDOW_STEP] = MC_RING_START;
  win.blocks[t * MC_WINDOW_STEP] = 0;
  if (t == 0) *win.left = 0;
  if (t == 0 && win.thick) *win.thick = 0;
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
      w = c < (uint32_t)a.L.m ? (int)c : 0;
      win.at[i] = w;
      win.ev[i] = 0;
      if (a.collisions) a.collisions[i] = 0;
      if (a.score) a.score[i] = 0.0;
    } else {
      w = win.at[i];
    }
    if (w >= 0) atomicAdd(&s_n[w / win.W], 1u);
  }
  if (OPEN && win.thick) {
    uint32_t thick = 0;
    for (int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; c < a.L.m;
         c += (int64_t)gridDim.x * blockDim.x)
      thick += mc_thick(a.cells[c], a.L.dx) ? 1u : 0u;
    thick = mc_wave_sum_u32(thick);
    if (__lane_id() == 0 && thick != 0) atomicAdd(win.thick, thick);
  }
  __syncthreads();
  if (threadIdx.x < (unsigned)win.nw && s_n[threadIdx.x]) {
    atomicAdd(&win.count[threadIdx.x], s_n[threadIdx.x]);
    atomicAdd(win.left, s_n[threadIdx.x]);
  }
}

/* the histories of each window one after the other (cursors zeroed), and
   room for those parked in the sweep */
__global__ void k_windows_list(int64_t n, mc_windows win, uint32_t *list, uint32_t *cursor) {
  __shared__ uint32_t s_n[MC_MAX_WINDOWS], s_at[MC_MAX_WINDOWS];
  const int t = threadIdx.x;
  const size_t words = win.cap ? (size_t)win.nw * (win.cap + MC_RING_PAD) : 0;
  for (size_t i = (size_t)blockIdx.x * blockDim.x + t; i < words;
       i += (size_t)gridDim.x * blockDim.x)
    win.parked[i] = MC_NOT_PUT;
  for (int64_t base = (int64_t)blockIdx.x * blockDim.x; base < n;
       base += (int64_t)gridDim.x * blockDim.x) { /* block-uniform */
    if (t < MC_MAX_WINDOWS) s_n[t] = 0;
    __syncthreads();
    const int64_t i = base + t;
    const int at = i < n ? win.at[i] : -1, w = at >= 0 ? at / win.W : -1;
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
   fx_hi, ...): LDS, the walk, the tally and totals.  k: mc_ceil_log2 of the
   weights this thread has looked at */
template <bool LDS_TALLY, bool LDS_CELLS, bool SCORE, typename IO, typename Queue>
__device__ __forceinline__ void history_block(const mc_transport_args &a, const mc_layer_k &L,
                                              int off, IO &io, Queue &queue, int k, int sh,
                                              int refill_k) {
  extern __shared__ __align__(16) unsigned char smem[];
  __shared__ mc_scale s_scale;
  __shared__ uint32_t s_thick;
  __shared__ unsigned long long s_tot[MC_TOTALS];
  /* Layers of thick cells: a walk of their own, and nothing of the common one
     alive in it, which would otherwise spill.  Not in windows, where with it
     8 M histories on 10,000 cells took 163 -> 168 ms and 200,000 on 20,000 cells
     35.8 -> 37.1, thick ones on 20,000 cells 14.5 -> 9.7. */
  constexpr bool THICK = LDS_TALLY && !Queue::LEAVES;
  constexpr int U = LDS_TALLY ? MC_IN_LDS : MC_IN_MEMORY;
  const int m = L.m;
  double2 *tab = reinterpret_cast<double2 *>(smem);
  mc_tab_fill(tab);
  unsigned long long *t0 = reinterpret_cast<unsigned long long *>(smem + MC_TAB_BYTES);
  unsigned long long *t1 = t0 + m; /* words with carry: one copy */
  const mc_limbs T = mc_limbs_at(t0, m, sh), mine = mc_limbs_mine(T);
  if (LDS_TALLY)
    for (int c = threadIdx.x; c < 2 * m << sh; c += blockDim.x) t0[c] = 0;
  const mc_cell *cells = a.cells + off;
  const double *g = SCORE ? a.g + off : nullptr;
  if (LDS_CELLS) {
    mc_cell *lc = reinterpret_cast<mc_cell *>(t0 + (2 * (size_t)m << sh));
    cells = mc_cells_fill(lc, cells, m);
    if (SCORE) {
      double *lg = reinterpret_cast<double *>(lc + m + 2);
      for (int c = threadIdx.x; c < m; c += blockDim.x) lg[c] = g[c];
      g = lg;
    }
  }
  if (threadIdx.x < MC_TOTALS) s_tot[threadIdx.x] = 0;
  if (threadIdx.x == 0) {
    mc_scale_clear(&s_scale);
    s_thick = 0;
  }
  __syncthreads();
  if (LDS_TALLY) {
    atomicMax(&s_scale.w, k);
    if (THICK) mc_count_thick(&s_thick, cells, m, L.dx);
    if (m >= MC_THICK_CELLS) mc_scale_cells(&s_scale, cells, m, L.dx);
    __syncthreads();
  }

  unsigned long long *fx_lo = a.fx + off, *fx_hi = fx_lo + a.L.m;
  uint32_t *flags = a.flags + off;
  unsigned int *status = &a.ctr->status;
  const mc_block_tally B = mc_block_tally_for(m, s_scale, blockDim.x >> 6);
  bool limbs = false;
  if constexpr (LDS_TALLY) limbs = B.limbs;
  auto on_event = [&](mc_mask lanes, int c8, const mc_cell &, bool, double, double dw, double) {
    mc_tally_limbs(mine, B.S, fx_lo, fx_hi, flags, status, lanes, c8, dw);
    if (SCORE && mc_in(lanes)) io.score = io.score + *mc_word(g, c8) * dw;
  };
  const mc_mover mover{T, fx_lo, fx_hi, m, B.S.L, B.every, B.every};
  if constexpr (THICK) {
    const int thick = __builtin_amdgcn_readfirstlane((int)s_thick);
    if (limbs && 2 * thick > m) { /* block-uniform */
      mc_walk_bank<LDS_CELLS, U, true>(io, queue, L, mc_walk_live<U>(L), cells, tab, refill_k,
                   B.every, a.max_events, s_tot, on_event, mover);
      __syncthreads();
      mc_limbs_move(T, B.S.L, m, threadIdx.x, blockDim.x, fx_lo, fx_hi);
      if (threadIdx.x == 0) mc_totals_out(s_tot, a.ctr, mc_counter_copy());
      return;
    }
  }
  const mc_walk_k K = mc_walk_live<U>(L);
  if (limbs) { /* block-uniform */
    mc_walk_bank<LDS_CELLS>(io, queue, L, K, cells, tab, refill_k, B.every, a.max_events, s_tot,
                 on_event, mover);
    __syncthreads();
    mc_limbs_move(T, B.S.L, m, threadIdx.x, blockDim.x, fx_lo, fx_hi);
  } else {
    unsigned long long *lo = LDS_TALLY ? t0 : fx_lo, *hi = LDS_TALLY ? t1 : fx_hi;
    mc_walk_bank<LDS_CELLS, U>(io, queue, L, K, cells, tab, refill_k, 1 << 30, a.max_events, s_tot,
                 [&](mc_mask lanes, int c8, const mc_cell &, bool, double, double dw, double) {
                   if (mc_in(lanes)) {
                     mc_tally(lo, hi, flags, status, mc_cell_of<U>(c8), dw);
                     if (SCORE) io.score = io.score + *mc_word<U>(g, c8) * dw;
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
  /* (windows, whose calls are long, keep to the first copy: with the others 200,000
     histories on 20,000 cells took 36.5 -> 38.1 ms) */
  if (threadIdx.x == 0) mc_totals_out(s_tot, a.ctr, Queue::LEAVES ? 0u : mc_counter_copy());
}

/* mc_ceil_log2 of the largest weight among the wave's first histories and one
   anywhere */
__device__ __forceinline__ int look_at_weights(const mc_transport_args &a, const mc_queue &q) {
  int k = -1023;
  auto look = [&](uint64_t i, uint64_t end) {
    const int of = i < end ? mc_ceil_log2(a.aos ? a.aos[i].wmc : a.soa.wmc[i]) : -1023;
    k = of > k ? of : k;
  };
  look(q.next + __lane_id(), q.end);
  look(mc_scale_place(0, (uint64_t)a.n, (uint64_t)threadIdx.x * gridDim.x + blockIdx.x,
                      (uint64_t)blockDim.x * gridDim.x), (uint64_t)a.n);
  return k;
}

template <bool LDS_TALLY, bool LDS_CELLS, bool SCORE>
__global__ __launch_bounds__(1024) void k_history(mc_transport_args a, int refill_k, int per_cu,
                                                  int sh) {
  mc_call_queue queue{mc_queue_open(a.n, per_cu, blockIdx.x, gridDim.x), &a.ctr->next};
  bank_io<SCORE> io{a, 0.0};
  const int k = LDS_TALLY ? look_at_weights(a, queue.q) : -1023;
  history_block<LDS_TALLY, LDS_CELLS, SCORE>(a, a.L, 0, io, queue, k, LDS_CELLS ? sh : 0,
                                             refill_k);
}

/* A long run on a layer whose tally fits LDS but not its cells, if they are thick:
   k_history_windows leaves it, as their walk and windows do not go into one
   kernel (history_block).  8,000 cells, 2 M histories of some 160 events, all
   collisions, in two windows 21.6 ms, here 15.9. */
template <bool SCORE>
__global__ __launch_bounds__(1024) void k_history_if_thick(mc_transport_args a, int refill_k,
                                                           int per_cu, const uint32_t *thick) {
  if (2 * (int64_t)*thick <= a.L.m) return;
  if (blockIdx.x == 0 && threadIdx.x == 0) a.ctr->left = 0;
  mc_call_queue queue{mc_queue_open(a.n, per_cu, blockIdx.x, gridDim.x), &a.ctr->next};
  bank_io<SCORE> io{a, 0.0};
  const int k = look_at_weights(a, queue.q);
  history_block<true, false, SCORE>(a, a.L, 0, io, queue, k, 0, refill_k);
}

/* the tally of the first `most` cells in all of the block's LDS (mc_full_tally) */
__global__ __launch_bounds__(1024) void k_history_full(mc_transport_args a, int refill_k,
                                                       int per_cu, int most) {
  extern __shared__ __align__(16) unsigned char smem[];
  __shared__ mc_scale s_scale;
  __shared__ unsigned long long s_tot[MC_TOTALS];
  mc_call_queue queue{mc_queue_open(a.n, per_cu, blockIdx.x, gridDim.x), &a.ctr->next};
  bank_io<false> io{a, 0.0};
  const int k = look_at_weights(a, queue.q);
  const mc_walk_k K = mc_walk_live(a.L);
  mc_full_tally F;
  F.t = reinterpret_cast<unsigned long long *>(smem);
  F.m = a.L.m < most ? a.L.m : most;
  for (int c = threadIdx.x; c < 2 * F.m; c += blockDim.x) F.t[c] = 0;
  if (threadIdx.x < MC_TOTALS) s_tot[threadIdx.x] = 0;
  if (threadIdx.x == 0) mc_scale_clear(&s_scale);
  __syncthreads();
  atomicMax(&s_scale.w, k);
  mc_scale_cells(&s_scale, a.cells, a.L.m, a.L.dx);
  __syncthreads();
  F.B = mc_block_tally_for(a.L.m, s_scale, blockDim.x >> 6);
  F.fx_lo = a.fx;
  F.fx_hi = a.fx + a.L.m;
  F.flags = a.flags;
  F.status = &a.ctr->status;
  F.left = F.B.every;
  mc_walk_bank<false>(io, queue, a.L, K, a.cells, reinterpret_cast<const double2 *>(mc_abs_tab),
               refill_k, F.every(), a.max_events, s_tot,
               [&](mc_mask lanes, int c8, const mc_cell &, bool, double, double dw, double) {
                 F.add(lanes, c8, dw);
               },
               [&](int n) { F.moves(n); });
  __syncthreads();
  F.out();
  if (threadIdx.x == 0) mc_totals_out(s_tot, a.ctr, mc_counter_copy());
}

/* one sweep over the windows of a wide layer */
template <bool LDS_CELLS, bool SCORE>
__global__ __launch_bounds__(1024) void k_history_windows(mc_transport_args a, mc_windows win,
                                                          int refill_k, int per_cu) {
  if (win.thick && 2 * (int64_t)*win.thick > a.L.m) return; /* k_history_if_thick's */
  __shared__ mc_window_block blk;
  const mc_window_share sh = mc_window_of(win);
  if (threadIdx.x == 0) {
    blk = {0, 0, 0, 0, 0, 0, sh.w};
    if (sh.w >= 0) atomicAdd(&win.blocks[sh.w * MC_WINDOW_STEP], 1u);
  }
  __syncthreads();
  int w = __builtin_amdgcn_readfirstlane(sh.w);
  for (bool first = true;; first = false) {
    if (!first || w < 0) { /* block-uniform */
      __syncthreads();
      if (threadIdx.x == 0) {
        if (w >= 0) atomicSub(&win.blocks[w * MC_WINDOW_STEP], 1u);
        if (blk.done) atomicSub(win.left, blk.done);
        blk.done = 0;
      }
      if (threadIdx.x < 64) mc_window_choose(win, &blk);
      __syncthreads();
      w = __builtin_amdgcn_readfirstlane(blk.w);
      if (w < 0) return;
    }
    const int off = w * win.W;
    mc_layer_k L = a.L;
    L.index_start += off;
    L.m = a.L.m - off < win.W ? a.L.m - off : win.W;
    const bool listed = first && sh.w >= 0;
    mc_window_queue queue{
        {mc_queue_open(listed ? win.count[w] : 0, per_cu, listed ? sh.block : 0u,
                       listed ? sh.blocks : 1u), &win.next[w]},
        win.list + sh.first, win, &blk, w, 0, false};
    window_io<SCORE> io{a, win, w, &blk, 0.0, -1};
    const uint64_t i = queue.open.q.next + __lane_id();
    int k = -1023;
    auto look = [&](int64_t j) {
      const int of = mc_ceil_log2(ld_shared(a.aos ? &a.aos[j].wmc : &a.soa.wmc[j]));
      k = of > k ? of : k;
    };
    if (listed) { /* the first histories, and one anywhere in the list */
      const uint64_t at =
          mc_scale_place(0, queue.open.q.n, (uint64_t)threadIdx.x * sh.blocks + sh.block,
                         (uint64_t)blockDim.x * sh.blocks);
      if (i < queue.open.q.end) look(queue.list[i]);
      if (at < queue.open.q.n) look(queue.list[at]);
    } else { /* threads look at the run's first histories; none is taken yet */
      if (threadIdx.x < mc_ring_left(blk.run)) {
        const uint32_t v = ld_shared(
            win.ring(w) + mc_ring_slot(mc_ring_next(blk.run) + threadIdx.x, win.cap));
        if (v != MC_NOT_PUT) look(v);
      }
    }
    history_block<true, LDS_CELLS, SCORE>(a, L, off, io, queue, k, 0, refill_k);
  }
}

/* LDS bytes of a window of W cells, with its cells (and targets) or without */
constexpr size_t window_lds(size_t W, bool cells, bool score) {
  return MC_TAB_BYTES + 16 * W +
         (cells ? sizeof(mc_cell) * W + MC_PAD_BYTES + (score ? 8 * W : 0) : 0);
}

/* last: the kernel's last argument */
template <typename K, typename V>
int launch_kernel(mcgpu_context *ctx, K kern, const mc_transport_args &a, const mcgpu_options &o,
                  hipStream_t s, size_t lds, V last) {
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
  int k = o.events_per_refill > 0 ? o.events_per_refill : 0; /* 0: adaptive */
  hipLaunchKernelGGL(kern, dim3(grid), dim3(block), lds, s, a, k, per_cu, last);
  MC_HIP(ctx, hipGetLastError());
  return MCGPU_OK;
}

template <bool T, bool C, bool S>
int launch_one(mcgpu_context *ctx, const mc_transport_args &a, const mcgpu_options &o,
               hipStream_t s, size_t lds) {
  int sh = 0;
  if (C) {
    const size_t other = lds - 16 * (size_t)a.L.m;
    lds = mc_lds_with_copies(lds, a.L.m);
    sh = mc_limbs_copies(a.L.m, lds - other);
  }
  return launch_kernel(ctx, k_history<T, C, S>, a, o, s, lds, sh);
}

/* A sweep over a wide layer's windows, cells in LDS or not; ctr->left counts the
   histories that it has not finished (usually none).  Scratch from the context
   (16 bytes per history and 4 per history and window); MCGPU_ERR_NOMEM: there is
   none.  ask: the tally fits LDS, and thick cells go to k_history_if_thick. */
template <bool LDS_CELLS, bool S>
int launch_windows(mcgpu_context *ctx, const mc_transport_args &a, const mcgpu_options &o,
                   hipStream_t s, int nw, int sweep, bool ask) {
  auto kern = k_history_windows<LDS_CELLS, S>;
  const int W = (a.L.m + nw - 1) / nw;
  const size_t lds = window_lds((size_t)W, LDS_CELLS, S);
  if (lds > 65536)
    (void)hipFuncSetAttribute(reinterpret_cast<const void *>(kern),
                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  int per_cu = 0;
  int block = o.block_size;
  if (block <= 0)
    block = mc_auto_block(ctx, kern, lds, &per_cu);
  else if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kern, block, lds) != hipSuccess ||
           per_cu < 1)
    per_cu = 1;
  const int resident = per_cu * ctx->num_cus, grid = o.grid_blocks > 0 ? o.grid_blocks : resident;
  const int k = o.events_per_refill > 0 ? o.events_per_refill : 0;

  /* ev[n], at[n], list[n], parked (the rings), queue counters, counts, cursors,
     and put, got, blocks a line apart */
  const size_t n = (size_t)a.n;
  const size_t cap = n * (size_t)nw <= MC_RING_WORDS ? mc_ring_cap((uint32_t)n) : 0; /* 0: no ring */
  const size_t rings = cap ? (cap + MC_RING_PAD) * (size_t)nw : 0;
  const size_t words = (16 * n + 4 * rings + 255) / 256 * 256;
  int rc = mc_ensure(ctx, &ctx->work, &ctx->work_bytes,
                     words + (16 + 12 * MC_WINDOW_STEP) * MC_MAX_WINDOWS + 4);
  if (rc) return rc;
  unsigned char *base = (unsigned char *)ctx->work;
  mc_windows win;
  win.nw = nw;
  win.W = W;
  win.cap = (uint32_t)cap;
  /* an idle block looks for parked histories for some 30 ms; at once it ends
     if there is no ring, or if blocks that have not started wait for its place */
  win.patience = cap == 0 ? 0 : (grid <= resident ? 1000 : 1);
  win.ev = (uint64_t *)base;
  win.at = (int32_t *)(base + 8 * n);
  uint32_t *list = (uint32_t *)(base + 12 * n);
  win.list = list;
  win.parked = (uint32_t *)(base + 16 * n);
  win.next = (unsigned long long *)(base + words);
  win.count = (uint32_t *)(win.next + MC_MAX_WINDOWS);
  uint32_t *cursor = win.count + MC_MAX_WINDOWS;
  win.left = &a.ctr->left;
  win.put = cursor + MC_MAX_WINDOWS;
  win.got = win.put + MC_MAX_WINDOWS * MC_WINDOW_STEP;
  win.blocks = win.got + MC_MAX_WINDOWS * MC_WINDOW_STEP;
  win.thick = ask && sweep == 0 ? win.blocks + MC_MAX_WINDOWS * MC_WINDOW_STEP : nullptr;
  const unsigned blocks = (unsigned)std::min<size_t>((n + 1023) / 1024, 4 * (size_t)ctx->num_cus);

  hipLaunchKernelGGL(k_windows_clear, dim3(1), dim3(64), 0, s, win, cursor);
  MC_HIP(ctx, hipGetLastError());
  if (sweep == 0)
    hipLaunchKernelGGL(k_windows_count<true>, dim3(blocks), dim3(1024), 0, s, a, win);
  else
    hipLaunchKernelGGL(k_windows_count<false>, dim3(blocks), dim3(1024), 0, s, a, win);
  MC_HIP(ctx, hipGetLastError());
  hipLaunchKernelGGL(k_windows_list, dim3(blocks), dim3(1024), 0, s, a.n, win, list, cursor);
  MC_HIP(ctx, hipGetLastError());
  hipLaunchKernelGGL(kern, dim3(grid), dim3(block), lds, s, a, win, k, per_cu);
  MC_HIP(ctx, hipGetLastError());
  if (win.thick)
    return launch_kernel(ctx, k_history_if_thick<S>, a, o, s, MC_TAB_BYTES + 16 * (size_t)a.L.m,
                         (const uint32_t *)win.thick);
  return MCGPU_OK;
}

/* the windows of a layer of m cells */
int windows_of(size_t m, size_t budget, bool cells, bool score) {
  const size_t fixed = window_lds(0, cells, score);
  const size_t most = (budget - fixed) / (window_lds(1, cells, score) - fixed);
  return (int)std::min<size_t>((m + most - 1) / most, 1u << 30);
}

template <bool S>
int launch_wide(mcgpu_context *ctx, const mc_transport_args &a, const mcgpu_options &o,
                hipStream_t s, size_t budget, int sweep, bool ask) {
  const int all = windows_of((size_t)a.L.m, budget, true, S);
  const int tally = windows_of((size_t)a.L.m, budget, false, S);
  const int limit = o.grid_blocks > 0 ? std::min(o.grid_blocks, MC_MAX_WINDOWS) : MC_MAX_WINDOWS;
  if (all <= limit) return launch_windows<true, S>(ctx, a, o, s, all, sweep, ask);
  if (tally > 1 && tally <= limit) return launch_windows<false, S>(ctx, a, o, s, tally, sweep, ask);
  return MCGPU_ERR_NOMEM;
}

} // namespace

int mc_launch_history(mcgpu_context *ctx, const mc_transport_args &a, const mcgpu_options &o,
                      hipStream_t s, int sweep) {
  const size_t m = (size_t)a.L.m;
  const size_t tally = 16 * m + MC_TAB_BYTES, cells = sizeof(mc_cell) * m + MC_PAD_BYTES;
  const size_t budget = ctx->lds_per_block - 256; /* the kernel's static LDS */
  const bool lds_tally = tally <= budget;
  const size_t targets = a.score ? 8 * m : 0;
  const bool lds_cells = lds_tally && tally + cells + targets <= budget;
  /* Windows, with scratch for them (not in the no-allocation entry point, whose
     context is quiet) and at least a block per window: for a layer whose tally
     does not fit (else the global tally), and for one whose tally fits but not
     its cells, if there are many histories per lane and many cells beyond
     those that fit.  Reading cells through L2 holds the long run back (37 lines
     per wave and event); windows lose to it where blocks that change windows
     run on few histories.  One window and two, in ms: 10,000 cells (4,934
     beyond) 8 M histories 234 and 161, 1 M 39.8 and 37.6, 500,000 25.5 and
     26.2; 8,500 cells 1 M 33.1 and 30.8; 7,000 cells 4 M 77 and 67, 1 M 26.9
     and 27.6; 6,000 cells 8 M 116 and 106, 4 M 62.6 and 65.5. */
  const size_t lanes = 1024 * (size_t)(o.grid_blocks > 0 ? o.grid_blocks : ctx->num_cus);
  const size_t beyond = (tally + cells + targets - std::min(budget, tally + cells + targets)) /
                        (sizeof(mc_cell) + 16 + (a.score ? 8 : 0));
  const bool long_run = !lds_cells && (double)a.n * (double)beyond >= 2e4 * (double)lanes &&
                        (size_t)a.n <= MC_RING_WORDS / 4;
  const bool block_ok = o.block_size <= 1024 && o.block_size % 64 == 0;
  if ((!lds_tally || long_run) && !ctx->quiet && a.n < (int64_t)0xFFFFFFFFu && block_ok &&
      !(a.score && !a.g)) {
    const int rc = a.score ? launch_wide<true>(ctx, a, o, s, budget, sweep, lds_tally)
                           : launch_wide<false>(ctx, a, o, s, budget, sweep, lds_tally);
    if (rc != MCGPU_ERR_NOMEM) return rc;
    ctx->err.clear();
  }
  if (a.score) { /* per-history score of a weighted tally (forward of the adjoint) */
    if (!a.g) return mc_fail(ctx, MCGPU_ERR_ARG, "score output needs target weights g");
    if (lds_cells) return launch_one<true, true, true>(ctx, a, o, s, tally + cells + targets);
    if (lds_tally) return launch_one<true, false, true>(ctx, a, o, s, tally);
    return launch_one<false, false, true>(ctx, a, o, s, MC_TAB_BYTES);
  }
  if (lds_cells) return launch_one<true, true, false>(ctx, a, o, s, tally + cells);
  if (lds_tally) return launch_one<true, false, false>(ctx, a, o, s, tally);
  const size_t most = budget / 16; /* cells of a tally in all of LDS */
  if (m <= most + MC_FULL_BEYOND)
    return launch_kernel(ctx, k_history_full, a, o, s, 16 * std::min(m, most), (int)most);
  return launch_one<false, false, false>(ctx, a, o, s, MC_TAB_BYTES);
}
