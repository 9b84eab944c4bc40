/*
 * mc_walk.h -- one transport event of Layer::particle_step
 * (src/layer.cpp:123-190) as the persistent kernels run it: a short common
 * step for the event that provably crosses its cell, and the general event
 * (mc_event_decide's operations) for everything else.
 *
 * What bounds these kernels is the number of vector instructions per event:
 * gfx950 issues one 64-bit (or three-operand) wave64 instruction per SIMD
 * every 4.25 cycles, and a wave on its own one every 8.5 whatever the
 * instruction, so the count sets both the rate of a full chip and the time of
 * a lone long history.  The common step has about half the instructions of
 * the event written out in full (mc_device.h):
 *  - the state is kept in the form the step uses: the doubled RNG state (the
 *    generator is a map mod 2^64 with no mask, and its top 32 bits are h's),
 *    1/mu as a pair, the next edge's number as a double, the cell as an
 *    offset in the layer;
 *  - the collision test needs only 20 bits of h: 1 + h (truncated) + sig_i *
 *    di_edge < 2 - 2^-18 implies 1 - h > sig_i * di_edge * (1 + 2^-40), the
 *    certificate of mc_event_decide;
 *  - the absorbed fraction is a rounding on a fixed grid (mc_absorb_thin,
 *    mc_absorb_row), with no exp to full relative accuracy;
 *  - the deposit is split into two limbs by floating-point adds and summed by
 *    two LDS adds without a returned value (mc_fx_split_limbs).
 * A lane whose event is not certified waits (`pend`) and the wave runs the
 * general event for its waiting lanes together (see mc_walk_many).
 */
#ifndef MC_WALK_H
#define MC_WALK_H

#include "internal.h"

constexpr size_t MC_TAB_BYTES = 16 * MC_ABS_N; /* the absorbed-fraction rows in LDS */

struct mc_walk {
  uint64_t s2;    /* twice the RNG state (mod 2^64) */
  double x, mu, wmc;
  double rh, rl;  /* 1/mu = rh + rl, rh = RN(1/mu); rh = NaN: no common step */
  double fe, fs;  /* number of the next edge, +-1 */
  int32_t c8, st8; /* U times the cell's offset in the layer, +-U (see below) */
};

/* U, the unit of c8 and st8.  8 where the tally is in LDS (c8 is then the byte
   offset of its words, half that of cells); 1 where it is in memory, in layers
   of any number of cells: 8 times a cell's offset needs a 32nd bit from 2^28
   cells on.  The global tally's two atomics hide the wider address. */
constexpr int MC_IN_LDS = 8, MC_IN_MEMORY = 1;

/* Edge distances are formed without range checks: with dx, x and mu in these
   bounds a = xn - x is 0 or at least 2^-752 (a difference of doubles that are
   0 or at least 2^-700), and every product of the quotient is normal.  Other
   particles take the general event until they collide. */
#define MC_WALK_X_MIN 0x1p-700
#define MC_WALK_DX_MIN 0x1p-600
#define MC_WALK_DX_MAX 0x1p600
#define MC_WALK_MU_MAX 0x1p64

template <int U>
__device__ __forceinline__ void mc_walk_turn(mc_walk &p, int32_t index) {
  const bool back = p.mu < 0;
  p.st8 = back ? -U : U;
  p.fs = back ? -1.0 : 1.0;
  p.fe = (double)index + (back ? 0.0 : 1.0);
  p.rh = 1.0 / p.mu;
  p.rl = mc_fma(-p.mu, p.rh, 1.0) * p.rh;
  const double mu = __builtin_fabs(p.mu), x = __builtin_fabs(p.x);
  if (!(mu > MC_EPS && mu <= MC_WALK_MU_MAX) || (x < MC_WALK_X_MIN && x != 0.0))
    p.rh = __builtin_nan("");
}

template <int U>
__device__ __forceinline__ void mc_walk_from(mc_walk &w, const mc_state &p, const mc_layer_k &L) {
  w.s2 = p.seed << 1;
  w.x = p.x;
  w.mu = p.mu;
  w.wmc = p.wmc;
  /* a history outside the layer ends at once; the edge's number keeps its index */
  const int64_t c = (int64_t)p.index - L.index_start;
  w.c8 = c < 0 ? -U : U * (c < L.m ? (int32_t)c : L.m);
  mc_walk_turn<U>(w, p.index);
}

__device__ __forceinline__ void mc_walk_to(mc_state &p, const mc_walk &w, const mc_layer_k &L) {
  p.seed = w.s2 >> 1;
  p.x = w.x;
  p.mu = w.mu;
  p.wmc = w.wmc;
  p.index = (int32_t)(w.fe - (w.st8 > 0 ? 1.0 : 0.0));
}

template <int U>
__device__ __forceinline__ bool mc_walk_alive(const mc_walk &w, const mc_layer_k &L) {
  return (w.wmc >= L.min_weight) && (uint32_t)w.c8 < (uint32_t)U * (uint32_t)L.m;
}

__device__ __forceinline__ void mc_walk_draw(uint64_t &s2) {
  s2 = MC_RNG_G * s2 + 2 * MC_RNG_C;
}

/* the state before the draw: the inverse of G mod 2^64 */
__device__ __forceinline__ uint64_t mc_walk_undraw(uint64_t s2) {
  return (s2 - 2 * MC_RNG_C) * 0xC097EF87329E28A5ULL;
}

/* h of the drawn state: (double)seed * 2^-63, rounded once (as mc_rnd_real) */
__device__ __forceinline__ double mc_walk_h(uint64_t s2) {
  return __builtin_fma((double)(uint32_t)(s2 >> 32), 0x1p-32, (double)(uint32_t)s2 * 0x1p-64);
}

/* wave-uniform values in scalar registers, which the compiler neither folds
   nor rebuilds from halves at each use */
struct mc_walk_k {
  mc_abs_coef A;
  double rem_max;   /* MC_ABS_REM */
  double sure_max;  /* 2 - 2^-18 */
  double three4;    /* 3/4 */
  double dx, min_weight;
  uint32_t m8, top8; /* U m, U (m - 1) */
  uint32_t one;      /* exponent field of 1.0 */
};

template <int U = MC_IN_LDS>
__device__ __forceinline__ mc_walk_k mc_walk_live(const mc_layer_k &L) {
  mc_walk_k K;
  K.A = mc_abs_coef_default();
  K.rem_max = MC_ABS_REM;
  K.sure_max = L.dx >= MC_WALK_DX_MIN && L.dx <= MC_WALK_DX_MAX ? 2.0 - 0x1p-18 : -1.0;
  K.three4 = 0.75;
  K.dx = L.dx;
  K.min_weight = L.min_weight;
  K.m8 = (uint32_t)U * (uint32_t)L.m;
  K.top8 = K.m8 - (uint32_t)U;
  K.one = 0x3FFu;
  asm volatile("" : "+v"(K.A.c7), "+s"(K.A.c6), "+s"(K.A.c5), "+s"(K.A.c4), "+s"(K.A.c3));
  asm volatile("" : "+s"(K.rem_max), "+s"(K.sure_max), "+s"(K.three4));
  asm volatile("" : "+s"(K.dx), "+s"(K.min_weight), "+s"(K.m8), "+s"(K.top8), "+s"(K.one));
  return K;
}

/* a wave-uniform value read from memory, in scalar registers */
__device__ __forceinline__ double mc_uniform(double v) {
  return mc_asf64(mc_readlane64(mc_asu64(v), 0));
}

__device__ __forceinline__ uint32_t mc_hi32(double v) { return (uint32_t)(mc_asu64(v) >> 32); }

/* Lanes of the wave as a scalar mask, and back.  Conditions are combined as
   masks (scalar ands), each ballot of one comparison. */
typedef unsigned long long mc_mask;
__device__ __forceinline__ mc_mask mc_lanes(bool b) { return __builtin_amdgcn_ballot_w64(b); }
__device__ __forceinline__ bool mc_in(mc_mask m) { return __builtin_amdgcn_inverse_ballot_w64(m); }

/* the cell of c8 (in [0, U m)).  U = 8: an unsigned 32-bit byte offset, so that
   a global load takes the uniform base in scalar registers */
template <int U>
__device__ __forceinline__ mc_cell mc_cell_at(const mc_cell *cells, uint32_t c8) {
  if (U == MC_IN_MEMORY) return cells[c8];
  return *reinterpret_cast<const mc_cell *>(reinterpret_cast<const char *>(cells) + (c8 << 1));
}

/* the cell's offset in the layer, and its word in an array of 8-byte words */
template <int U> __device__ __forceinline__ int mc_cell_of(int c8) {
  return U == MC_IN_LDS ? c8 >> 3 : c8;
}
template <int U = MC_IN_LDS, typename T> __device__ __forceinline__ T *mc_word(T *base, int c8) {
  if (U == MC_IN_MEMORY) return base + c8;
  return reinterpret_cast<T *>(reinterpret_cast<char *>(base) + c8);
}
template <int U = MC_IN_LDS, typename T>
__device__ __forceinline__ const T *mc_word(const T *base, int c8) {
  if (U == MC_IN_MEMORY) return base + c8;
  return reinterpret_cast<const T *>(reinterpret_cast<const char *>(base) + c8);
}

/* The common step on cell `cell`, for every lane of the wave: the draw, then
   the crossing's next edge xn, flight q and absorbed fraction u.  Returns
   the lanes whose event certainly is that crossing, u certified; for the
   others mc_walk_general finishes the event.  run: the lanes that matter.
   tab: the rows of mc_abs_tab (LDS).
   A quotient from rh = NaN fails every test.  A negative quotient (a particle
   beyond its edge) fails the range of y: a negative y, and -0 where sig_a is 0,
   have the sign bit set. */
__device__ __forceinline__ mc_mask mc_walk_cross(mc_walk &p, mc_mask run, const mc_cell cell,
                                                 const double2 *tab, const mc_walk_k &K,
                                                 double &xn, double &q, double &u) {
  mc_walk_draw(p.s2);
  xn = p.fe * K.dx;
  const double a = xn - p.x;
  q = mc_div_by_pair(a, p.mu, p.rh, p.rl);
  /* 1 + h with h's top 20 bits (h itself is less than 2^-20 above); the fma
     written out, as the compiler's form copies the addend first */
  const uint32_t sh = (uint32_t)(p.s2 >> 32);
  const double h1 = mc_asf64((uint64_t)__builtin_amdgcn_alignbit(K.one, sh, 12) << 32);
  double t;
  asm("v_fma_f64 %0, %1, %2, %3" : "=v"(t) : "v"(cell.sig_i), "v"(q), "v"(h1));
  const double y = cell.sig_a * q;
  mc_mask ok = run & mc_lanes(t < K.sure_max);
  double rem;
  /* y in [0, MC_ABS_THIN) by its high word (negative and NaN fail) */
  const mc_mask thin = mc_lanes(mc_hi32(y) < (uint32_t)((1023 - 8) << 20));
  if (__builtin_expect((run & ~thin) == 0, 1)) { /* wave-uniform: every live lane is thin */
    u = mc_absorb_thin(y, K.three4, &K.A, &rem);
  } else {
    ok &= mc_lanes(mc_hi32(y) < 0x3FE60000u); /* [0, MC_ABS_YMAX) */
    const unsigned k = mc_abs_index(y);
    const double2 row = tab[k < MC_ABS_N ? k : MC_ABS_N - 1u];
    u = mc_absorb_row(y, row.x, row.y, &K.A, &rem);
  }
  return ok & mc_lanes(__builtin_fabs(rem) < K.rem_max);
}

/* The general event, after mc_walk_cross has drawn: mc_event_decide's
   operations and the absorption.  Returns the deposit; coll: whether it
   collided, di: the flight.  THICK: for mc_walk_thick, which divides by rh alone
   (after a collision |mu| is below 1, and mc_div_by_rcp tests the rest). */
template <int U, bool THICK = false>
__device__ __forceinline__ double mc_walk_general(mc_walk &p, const mc_cell cell, const double dx,
                                                  const mc_coef &K, bool &coll, double &di) {
  const double h = mc_walk_h(p.s2);
  const double xn = p.fe * dx;
  const bool flat = !(p.mu < -MC_EPS || MC_EPS < p.mu);
  const double di_edge = flat ? MC_MAXREAL : mc_div_by_rcp(xn - p.x, p.mu, p.rh);
  const double reach = cell.sig_i * di_edge;
  const int sure_cross =
      (int)!(cell.sig_i > MC_EPS) | (int)((1.0 - h) > mc_fma(reach, 0x1p-40, reach));
  di = di_edge;
  coll = false;
  if (!sure_cross) {
    const double dq = -mc_log_k(h, &K) / cell.sig_i;
    coll = dq < di_edge;
    if (coll) di = dq;
  }
  const double dw = (1 - mc_exp_k(-cell.sig_a * di, &K)) * p.wmc;
  p.wmc -= dw;
  if (coll) {
    p.x += di * p.mu;
    mc_walk_draw(p.s2);
    p.mu = 2 * mc_walk_h(p.s2) - 1;
    if (THICK) {
      const bool back = p.mu < 0;
      const double fs = back ? -1.0 : 1.0;
      p.st8 = back ? -U : U;
      p.fe = mc_fma(0.5, fs - p.fs, p.fe); /* the same cell's other edge, or this one */
      p.fs = fs;
      p.rh = 1.0 / p.mu;
    } else { /* the index from the edge ahead: fe is index + 1 moving up, index moving down */
      mc_walk_turn<U>(p, (int32_t)p.fe - (p.st8 > 0 ? 1 : 0));
    }
  } else {
    p.x = xn;
    p.fe += p.fs;
    p.c8 += p.st8;
  }
  return dw;
}

/* The waiting lanes (per 64 live ones) at which the wave runs the general
   event.  Running it for one lane costs the wave about three common steps;
   letting w lanes wait leaves w/2 of 64 idle on average.  With a chance p per
   event the sum is least at w = sqrt(128 * 64 * 3 p), which is 400 times the
   general events per iteration (64 p / w) at that w: move towards it. */
__device__ __forceinline__ int mc_walk_wait(int wait, int general, int iterations) {
  const int want = 400 * general;
  if (want > wait * iterations) return wait < 16 ? wait + 1 : 16;
  return wait > 1 ? wait - 1 : 1;
}

/* Where the waiting lanes start: w = sqrt(128 * 64 * 3 p) for the mean chance p
   of a collision in 64 cells spread over the layer, at the mean cosine of 1/2.
   In short layers most histories collide all the way; below 6 the walk finds w
   by itself in time.  Starting from 1 everywhere, w grew by one an interval and
   histories of a hundred events ended before it had: 200,000 on 10,180 cells
   0.74 -> 0.58 ms, 64 slabs of 2,000 cells 0.96 -> 0.81, forward 0.94 -> 0.81,
   gradient 1.07 -> 0.91. */
template <int U>
__device__ __forceinline__ int mc_walk_first_wait(const mc_cell *cells, const mc_layer_k &L) {
  if (L.m < 128) return L.m < 64 ? 12 : 4;
  const int c = (int)(((int64_t)__lane_id() * L.m) >> 6);
  const double p = 2.0 * cells[c].sig_i * L.dx;
  const uint32_t sum = mc_wave_sum_u32((uint32_t)(p > 0.0 ? (p < 1.0 ? p : 1.0) * 0x1p20 : 0.0));
  const int w = (int)__builtin_sqrtf((float)sum * (24576.0f * 0x1p-26f));
  return w < 6 ? 1 : (w < 16 ? w : 16);
}

/* Histories that set out together from one cell in one direction stay in the
   same cell as long as none collides (an event moves each by one cell), and a
   wave's adds to one LDS word follow one another.  So such lanes set out one
   event apart: their cells, and the words they add to, then lie side by side.
   The window kernel lets two or more wait (they start at a window's edge),
   the others four or more, in layers of 256 cells on: in shorter ones the
   events spent waiting cost more than the adds (100,000 histories through
   host buffers on 100 cells 1.63 ms against 1.67 with it).
   Measured without and with: 2 M histories into both faces of a 1,000-cell
   layer 10.4 -> 4.9 ms, forward and gradient of 1,000 cells and 1 M histories
   11.6 -> 10.2 ms, 512 slabs 46.9 -> 43.1 ms, 2 M histories in windows of
   20,000 cells 176 -> 123 ms.  With each event of a start a call of
   mc_walk_many, short histories lost: the cycle loop 12.9 -> 14.1 ms, now
   13.0. */
constexpr int MC_APART_CELLS = 256;

/* the next lane to set out (fresh may be empty) */
__device__ __forceinline__ mc_mask mc_sets_out(mc_mask &fresh) {
  const mc_mask one = fresh & (0 - fresh);
  fresh ^= one;
  return one;
}

/* Up to ki events of every lane in `run` (lanes whose history goes on; `pend`:
   lanes whose drawn event waits for the general form; `fresh`: lanes that set
   out one after the other, one per event; all wave-uniform masks, disjoint).
   on_event(lanes, c8, cell, coll, di, dw, wmc) is called by the whole wave for
   an event of `lanes` in cell c8 / U (wmc: the weight after it).  ei counts a
   lane's events, col its collisions.  Returns how often the general event ran.
   Every lane computes the common step (lanes not in `run` on whatever they
   hold); only the lanes of a certified crossing commit it.  A history's end
   shows at its next step, whose draw is taken back: the step's own tests and
   the weight's are then the only ones, and an iteration in which no lane
   stops or waits costs one scalar comparison.  PAD: cells[-1] and cells[m]
   exist and hold NaN, so that a lane that left the layer fails the step's
   tests; without them the cell index is clamped and tested.  The next cell is
   loaded before the tally's adds, so that its latency passes under them and
   the next draw.
   Measured with the history kernel, against testing every lane's index and
   weight and the quotient's range at each step, and reading the cell as two
   words: 40 M histories on 100 cells 19.5 -> 17.0 ms, 20 M on 1,000 cells
   58.9 -> 48.2 ms, 8 M on 4,000 cells (bound by LDS: the counter of its active
   cycles stood at 90 % of the time) 81.0 -> 64.6 ms; 1,000 on 1,000 cells,
   where the longest history's events follow one another, 1.09 -> 0.92 ms. */
template <bool PAD, int U, typename F>
__device__ __forceinline__ int mc_walk_many(mc_walk &p, mc_mask &run, mc_mask &pend,
                                            mc_mask &fresh, int ki, int wait,
                                            const mc_cell *cells, const double2 *tab,
                                            const mc_walk_k &K, uint32_t &ei, uint32_t &col,
                                            F on_event) {
  static_assert(!PAD || U == MC_IN_LDS, "cells in LDS, tally in LDS");
  int general = 0;
  auto cell_of = [&](int c8) {
    if (PAD) /* c8 >= -8 */
      return *reinterpret_cast<const mc_cell *>(reinterpret_cast<const char *>(cells) + 2 * c8);
    return mc_cell_at<U>(cells, (uint32_t)c8 < K.top8 ? (uint32_t)c8 : K.top8);
  };
  for (;;) {
    const int live = __popcll(run | pend | fresh);
    if (live == 0) break;
    const int nwait = ki > 0 ? (wait * live + 63) >> 6 : 1;
    if ((run | fresh) != 0 && ki > 0 && __popcll(pend) < nwait) {
      const int k0 = ki;
      run |= mc_sets_out(fresh);
      mc_mask all = run | fresh;
      uint64_t s2 = p.s2; /* the state of the lanes not in run: the draw below is for all */
      mc_cell cell;
      if (mc_in(all)) cell = cell_of(p.c8);
      for (;;) {
        double xn, q, u;
        mc_mask ok = mc_walk_cross(p, run, cell, tab, K, xn, q, u);
        ok &= mc_lanes(p.wmc >= K.min_weight);
        if (!PAD) ok &= mc_lanes((uint32_t)p.c8 < K.m8);
        const mc_cell here = cell;
        const int c8 = p.c8;
        const double dw = u * p.wmc;
        if (mc_in(ok)) {
          p.wmc -= dw;
          p.x = xn;
          p.fe += p.fs;
          p.c8 += p.st8;
          cell = cell_of(p.c8);
        }
        on_event(ok, c8, here, false, q, dw, p.wmc);
        --ki;
        if (__builtin_expect(ok != all, 0)) { /* wave-uniform: a lane stopped, waits or sets out */
          const mc_mask out = run & ~ok;
          const mc_mask waits = out & mc_lanes(p.wmc >= K.min_weight) &
                                mc_lanes((uint32_t)p.c8 < K.m8);
          if (mc_in(out)) {
            s2 = mc_in(waits) ? p.s2 : mc_walk_undraw(p.s2);
            ei += (uint32_t)(k0 - ki - 1);
          }
          pend |= waits;
          run = ok;
          if (fresh != 0) {
            const mc_mask sets_out = mc_sets_out(fresh);
            if (mc_in(sets_out)) {
              p.s2 = s2;
              ei -= (uint32_t)(k0 - ki);
            }
            run |= sets_out;
          }
          all = run | fresh;
          if (run == 0 || __popcll(pend) >= nwait) break;
        }
        if (ki == 0) break;
      }
      if (mc_in(run))
        ei += (uint32_t)(k0 - ki);
      else
        p.s2 = s2;
    }
    if (pend != 0 && ((run | fresh) == 0 || __popcll(pend) >= nwait)) {
      ++general;
      const int c8 = p.c8;
      mc_cell cell;
      cell.sig_a = cell.sig_i = 0.0;
      bool coll = false;
      double di = 0.0, dw = 0.0;
      if (mc_in(pend)) {
        cell = mc_cell_at<U>(cells, (uint32_t)c8);
        dw = mc_walk_general<U>(p, cell, K.dx, mc_coef_default(), coll, di);
        ++ei;
        col += coll ? 1u : 0u;
      }
      on_event(pend, c8, cell, coll, di, dw, p.wmc);
      run |= pend;
      pend = 0;
    }
    run &= mc_lanes(p.wmc >= K.min_weight) & mc_lanes((uint32_t)p.c8 < K.m8);
    if (ki == 0) break;
  }
  return general;
}

/* mc_walk_many for thick cells, where most events are general ones: no common
   step before them, every lane's event a general one.  Bound by the general
   event's instructions, some 300 of them.  (Within mc_walk_many, as a mode of
   its own, this made the common loop 5 to 10 % slower.)  Its coefficients and
   dx stay in registers; with dx among the scalar ones the kernels' arguments
   came back from their spills at each event.  Histories of 2,300 events, all
   collisions, on 100 cells, by the history kernel with mc_walk_many and so: one
   2.86 and 1.70 ms, 20,000 of them 3.91 and 2.34, 2 M of 340 events 42.3 and
   25.7. */
template <int U, typename F>
__device__ __forceinline__ void mc_walk_thick(mc_walk &p, mc_mask &run, mc_mask &fresh, int ki,
                                              const mc_cell *cells, const mc_walk_k &K,
                                              uint32_t &ei, uint32_t &col, F on_event) {
  mc_coef C = mc_coef_default();
  double dx = K.dx;
  asm volatile("" : "+v"(C.l8), "+v"(C.l7), "+v"(C.l6), "+v"(C.l5), "+v"(C.l4), "+v"(C.l3));
  asm volatile("" : "+s"(C.e5), "+s"(C.e4), "+s"(C.e3), "+s"(C.ziv), "+v"(dx));
  run |= fresh;
  fresh = 0;
  for (; ki > 0 && run != 0; --ki) { /* wave-uniform */
    const int c8 = p.c8;
    mc_cell cell;
    cell.sig_a = cell.sig_i = 0.0;
    bool coll = false;
    double di = 0.0, dw = 0.0;
    if (mc_in(run)) {
      cell = mc_cell_at<U>(cells, (uint32_t)c8);
      mc_walk_draw(p.s2);
      dw = mc_walk_general<U, true>(p, cell, dx, C, coll, di);
      ++ei;
      col += coll ? 1u : 0u;
    }
    on_event(run, c8, cell, coll, di, dw, p.wmc);
    run &= mc_lanes(p.wmc >= K.min_weight) & mc_lanes((uint32_t)p.c8 < K.m8);
  }
}

/* exit code of a history that ends in state p (2: alive, stopped by the cap) */
__device__ __forceinline__ int mc_end_code(const mc_state &p, bool at_cap, const mc_layer_k &L) {
  return at_cap && mc_alive(p, L) ? 2 : mc_exit_code(p, L);
}

/* -------------------------------------------------------------- work queue */

/* The histories 0 .. n-1 of a call, taken by waves in runs: the first run of
   each wave is its own by position (no atomic), later ones come from the
   call's counter, a quarter of what is left per wave at a time.  With one
   atomic per refill instead, short histories wait for the counter: one
   address takes about one atomic every 7 ns from a full chip.
   First runs go to wave 0 of every block, then to wave 1 of every block, ...:
   few histories spread over all CUs and SIMDs.  A SIMD runs two waves as fast
   as one (each issues at most every 8.5 cycles, the SIMD every 4.25), four
   at half speed, and a wave's lanes wait for each other's general events; so
   up to 64 histories for each of the first eight waves of a CU are dealt out
   evenly among those waves. */
struct mc_queue {
  uint64_t n, next, end; /* the wave's run [next, end) */
  uint64_t first, seen;  /* where the counter's zero stands; the last place seen */
  uint32_t waves;
  bool dry;              /* no run left to take */
};

__device__ __forceinline__ uint64_t mc_run_size(uint64_t left, uint32_t waves) {
  const uint64_t s = left / (4u * (uint64_t)waves);
  return s < 64 ? 64 : (s > 4096 ? 4096 : s);
}

/* per_cu: blocks on a CU; this is block `block` of `blocks` that share the queue */
__device__ __forceinline__ mc_queue mc_queue_open(int64_t n, int per_cu, uint32_t block,
                                                  uint32_t blocks) {
  mc_queue q;
  const uint32_t per_block = blockDim.x >> 6;
  const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const uint32_t pos = wave * blocks + block;
  q.n = (uint64_t)n;
  q.waves = blocks * per_block;
  const uint32_t few = (per_block * (uint32_t)per_cu > 8u ? (8u + per_cu - 1) / per_cu : per_block) *
                       blocks;
  const uint64_t size = q.n <= 64ull * few ? (q.n + few - 1) / few : mc_run_size(q.n, q.waves);
  q.next = pos * size;
  q.end = q.next + size;
  q.first = q.seen = q.waves * size;
  if (q.end > q.n) q.end = q.n;
  if (q.next > q.n) q.next = q.n;
  q.dry = q.first >= q.n;
  return q;
}

__device__ __forceinline__ bool mc_queue_more(const mc_queue &q) {
  return !q.dry || q.next < q.end;
}

__device__ __forceinline__ int64_t mc_queue_take(mc_queue &q, mc_mask need,
                                                 unsigned long long *counter) {
  const uint64_t cnt = (uint64_t)__popcll(need), have = q.end - q.next;
  const uint64_t rank = (uint64_t)mc_mbcnt64(need);
  uint64_t i = q.next + rank;
  if (cnt <= have || q.dry) {
    if (rank >= have) i = ~0ull;
    q.next = cnt < have ? q.next + cnt : q.end;
  } else { /* wave-uniform */
    const uint64_t size = mc_run_size(q.n - q.seen, q.waves); /* seen < n: not dry */
    unsigned long long base = 0;
    if (__lane_id() == 0) base = atomicAdd(counter, (unsigned long long)size);
    base = mc_readlane64(base, 0) + q.first;
    uint64_t end = base + size;
    if (end >= q.n) {
      q.dry = true;
      end = q.n;
    }
    if (base > q.n) base = q.n;
    q.seen = base;
    if (rank >= have) i = base + (rank - have) < end ? base + (rank - have) : ~0ull;
    const uint64_t used = cnt - have;
    q.next = base + used < end ? base + used : end;
    q.end = end;
  }
  return (int64_t)i;
}

/* whether the wave can still take histories; a history for each lane of `need`
   or -1 (called by the whole wave) */
struct mc_call_queue {
  mc_queue q;
  unsigned long long *counter;
  __device__ __forceinline__ bool more() const { return mc_queue_more(q); }
  static constexpr bool LEAVES = false;
  __device__ __forceinline__ int least() const { return 8; }
  __device__ __forceinline__ int64_t take(mc_mask need) { return mc_queue_take(q, need, counter); }
};

/* the histories [.., end) of a block's tile, from its LDS counter */
struct mc_tile_queue {
  unsigned long long *counter; /* LDS */
  uint64_t end;
  bool dry;
  __device__ __forceinline__ bool more() const { return !dry; }
  static constexpr bool LEAVES = false;
  __device__ __forceinline__ int least() const { return 8; }
  __device__ __forceinline__ int64_t take(mc_mask need) {
    const uint64_t cnt = (uint64_t)__popcll(need);
    unsigned long long base = 0;
    if (__lane_id() == 0) base = atomicAdd(counter, (unsigned long long)cnt);
    base = mc_readlane64(base, 0);
    dry = base + cnt >= end;
    const uint64_t i = base + (uint64_t)mc_mbcnt64(need);
    return i < end ? (int64_t)i : -1;
  }
};

/* The block's totals, LDS words zeroed by the block: events, collisions, left,
   right, killed; then whether a history hit the cap.  One global atomic per
   block and nonzero total (mc_totals_out): with one per wave the five
   addresses of a full chip's 4,096 waves alone took 0.14 ms. */
constexpr int MC_TOTALS = 6;

/* by one thread of the block, after a barrier; copy: of the totals */
__device__ __forceinline__ void mc_totals_out(const unsigned long long *s_tot, mc_counters *ctr,
                                              unsigned copy) {
  unsigned long long *to = mc_counter_word(ctr, copy, 1);
  if (s_tot[0]) atomicAdd(&to[0], s_tot[0]);
  if (s_tot[1]) atomicAdd(&to[1], s_tot[1]);
  if (s_tot[2]) atomicAdd(&to[2], s_tot[2]);
  if (s_tot[3]) atomicAdd(&to[3], s_tot[3]);
  if (s_tot[4]) atomicAdd(&to[4], s_tot[4]);
  if (s_tot[5]) atomicOr(&ctr->status, 1u);
}

/* A wave's histories, one per lane, until its queue is empty.
   io.load(i, state) reads history i (and resets what the caller keeps per
   lane) and returns the events it has had before; io.store(i, state, code, ev,
   col) takes a finished one (ev with those before, col without) and returns
   whether the lane goes on, from no events, with the state it leaves in
   `state` (a replay); io.code(state, at_cap, L) is its exit code (3: none to
   count);
   on_event as in mc_walk_many; moves(k) is called before every (at most) k
   events per lane, k <= k_max.
   refill_k: events between refills; 0: adapted per wave, from a quarter of the
   layer's cells (8 to 128), by the lanes
   found idle at each refill (many idle: the histories are short against the
   interval, halve it; almost none: double it, since each refill costs a pass
   through this loop). */
template <bool PAD, int U = MC_IN_LDS, bool THICK = false, typename IO, typename Queue, typename Event, typename Moves>
__device__ __forceinline__ void mc_walk_bank(IO &io, Queue &queue, const mc_layer_k &L,
                                             const mc_walk_k &K, const mc_cell *cells,
                                             const double2 *tab, int refill_k, int k_max,
                                             uint64_t max_events, unsigned long long *s_tot,
                                             Event on_event, Moves moves) {
  mc_walk p;
  p.s2 = 0;
  p.x = p.mu = p.wmc = p.rh = p.rl = p.fe = p.fs = 0.0;
  p.c8 = p.st8 = 0;
  int64_t idx = 0;
  bool has = false;
  mc_mask run = 0, pend = 0; /* lanes whose history goes on / waits for the general event */
  mc_mask fresh = 0;         /* lanes whose history has not set out yet */
  const int apart = Queue::LEAVES ? 2 : (L.m >= MC_APART_CELLS ? 4 : 65);
  uint64_t ev = 0, before = 0; /* events of the lane's history; those before this call */
  uint32_t col = 0;
  const bool adapt = refill_k <= 0;
  int kk = adapt ? 128 : refill_k;
  int wait = 1;
  const int first_wait = Queue::LEAVES ? mc_walk_first_wait<U>(cells, L) : 0;
  bool first = true; /* no histories taken yet */
  /* wave-uniform bound on every lane's event count (a waiting event counted);
     recomputed exactly (the largest in the wave) when an interval could reach
     the cap, which then shortens the interval: no history passes the cap */
  uint64_t ev_bound = 0;
  for (;;) {
    if (queue.more()) { /* wave-uniform */
      const mc_mask need = mc_lanes(!has);
      if (adapt) {
        const int idle = __popcll(need);
        kk = idle > 16 ? kk >> 1 : (idle < 4 ? kk << 1 : kk);
        kk = kk < queue.least() ? queue.least() : (kk < 256 ? kk : 256);
      }
      if (need) {
        const int64_t i = queue.take(need);
        if (!queue.more()) {
          if (adapt) kk = 256; /* no refill to come */
        } else if (first) {
          /* from the layer's cells: a history crosses about as many as there
             are */
          if (adapt && L.m < 512) kk = L.m > 32 ? L.m >> 2 : 8;
          wait = Queue::LEAVES ? first_wait : mc_walk_first_wait<U>(cells, L);
        }
        first = false;
        bool on = false;
        if (!has && i >= 0) {
          mc_state in;
          ev = io.load(i, in);
          mc_walk_from<U>(p, in, L);
          idx = i;
          has = true;
          on = mc_walk_alive<U>(p, L) && ev < max_events;
          if (IO::RESUMES) before = ev;
          col = 0;
        }
        mc_mask out = mc_lanes(on);
        if (!Queue::LEAVES && out) { /* of other cells: at once */
          const int c8 = __builtin_amdgcn_readlane(p.c8, __builtin_ctzll(out));
          const mc_mask here = out & mc_lanes(p.c8 == c8);
          run |= out & ~here;
          out = here;
        }
        const int up = __popcll(out & mc_lanes(p.st8 > 0)), down = __popcll(out) - up;
        mc_mask &to = (up > down ? up : down) >= apart ? fresh : run;
        to |= out;
        if (IO::RESUMES) ev_bound = max_events; /* recomputed below */
      }
    }
    if constexpr (Queue::LEAVES) {
      const bool leaves = queue.leave(__popcll(mc_lanes(has)));
      if (leaves) { /* wave-uniform: the histories are stored as they stand */
        if (mc_in(pend)) p.s2 = mc_walk_undraw(p.s2);
        pend = run = fresh = 0;
      } else if (mc_lanes(has) == 0 && queue.wait()) {
        continue;
      }
    }
    if (mc_lanes(has) == 0) break; /* wave-uniform */
    int ki = kk < k_max ? kk : k_max - 1; /* a waiting lane may add one */
    if (ev_bound + (uint64_t)ki >= max_events) {
      ev_bound = mc_wave_max_u64(has ? ev + (mc_in(pend) ? 1u : 0u) : 0ull);
      if (ev_bound + (uint64_t)ki >= max_events)
        ki = ev_bound < max_events ? (int)(max_events - ev_bound) : 0;
    }
    ev_bound += (uint64_t)ki;
    moves(ki + 1);
    uint32_t ei = 0; /* events of this interval */
    if (THICK) {
      mc_walk_thick<U>(p, run, fresh, ki, cells, K, ei, col, on_event);
    } else {
      const int general =
          mc_walk_many<PAD, U>(p, run, pend, fresh, ki, wait, cells, tab, K, ei, col, on_event);
      wait = mc_walk_wait(wait, general, ki);
    }
    ev += ei;
    const bool on = mc_in(run | fresh), waits = mc_in(pend);
    const bool ends = has && !waits && (!on || ev >= max_events);
    if (mc_lanes(ends) == 0) continue; /* wave-uniform */
    bool again = false;
    int code = 3;
    uint32_t n_ev = 0, n_col = 0; /* for the totals */
    if (ends) {
      mc_state out;
      mc_walk_to(out, p, L);
      /* at the cap and alive: a runaway history stopped by the guard */
      code = io.code(out, ev >= max_events, L);
      n_ev = (uint32_t)(ev - before);
      n_col = col;
      if ((ev - before) >> 25) { /* 64 of them could pass 2^32 */
        atomicAdd(&s_tot[0], (unsigned long long)(ev - before));
        atomicAdd(&s_tot[1], (unsigned long long)col);
        n_ev = n_col = 0;
      }
      has = io.store(idx, out, code, ev, col);
      if (has) {
        mc_walk_from<U>(p, out, L);
        again = mc_walk_alive<U>(p, L);
        ev = before = 0;
        col = 0;
      }
    }
    /* The totals: each in a lane of its own, added at once.  (Atomic adds of all
       lanes to one word become a loop over the lanes, some 18 instructions for
       each: 300 slabs of 32 thick cells, whose histories have 7 events, 1.40
       ms with two of them, now 1.28.) */
    uint32_t total = mc_wave_sum_u32(n_ev);
    const uint32_t cols = mc_wave_sum_u32(n_col);
    const uint32_t nl = (uint32_t)__popcll(mc_lanes(code == -1));
    const uint32_t nr = (uint32_t)__popcll(mc_lanes(code == 1));
    const uint32_t nk = (uint32_t)__popcll(mc_lanes(code == 0));
    const unsigned lane = (unsigned)__lane_id();
    total = lane == 1 ? cols : (lane == 2 ? nl : (lane == 3 ? nr : (lane == 4 ? nk : total)));
    if (lane < 5 && total != 0) atomicAdd(&s_tot[lane], (unsigned long long)total);
    if (mc_lanes(code == 2) != 0 && lane == 0) atomicOr(&s_tot[5], 1ull);
    run = (run & mc_lanes(has)) | mc_lanes(again);
  }
}

/* ------------------------------------------------------------- block tally */

/* How a block's LDS tally takes terms.  Limbs (mc_fx_split) when the weights
   allow a useful interval between moves, else 128-bit adds with carry. */
struct mc_block_tally {
  mc_fx_split S;
  int every;  /* events per lane between two moves of the limbs (per wave) */
  int limbs;  /* 0: words (lo, hi) with carry */
};

/* smallest k with 2^k >= v (v >= 0, not subnormal); large for inf and NaN */
__device__ __forceinline__ int mc_ceil_log2(double v) {
  const uint64_t b = mc_asu64(v) & 0x7FFFFFFFFFFFFFFFULL;
  return (int)(b >> 52) - 1023 + ((b & 0x000FFFFFFFFFFFFFULL) ? 1 : 0);
}

/* What a block expects of its terms, in LDS: binary exponents of the largest
   weight, of the largest sig_a dx, and (gradients) of the largest target
   weight and sig_i.  A guess that sets the split; larger terms go to the
   global tally, where a full chip's adds to one word follow one another at
   about 7 ns each, so they have to stay rare. */
struct mc_scale {
  int w, thick, g, b;
};

/* by one thread, before a barrier */
__device__ __forceinline__ void mc_scale_clear(mc_scale *s) { *s = {-1023, -1023, -1023, -1023}; }

__device__ __forceinline__ bool mc_thick(const mc_cell k, double dx) {
  return (k.sig_i > k.sig_a ? k.sig_i : k.sig_a) * dx > 0.5;
}

/* Adds to *count (LDS, cleared before a barrier) the cells with sig_i dx or sig_a
   dx above 1/2, by all threads of a block.
   mc_walk_thick serves where they are more than half: at the mean cosine of 1/2
   two events in three collide there.  Batches of thick slabs without it and
   with, in ms: 300 slabs of 32 cells 1.24 and 0.90, 200 smaller ones 0.395 and
   0.298. */
__device__ __forceinline__ void mc_count_thick(uint32_t *count, const mc_cell *cells, int m,
                                               double dx) {
  uint32_t n = 0;
  for (int c = threadIdx.x; c < m; c += blockDim.x) n += mc_thick(cells[c], dx) ? 1u : 0u;
  n = mc_wave_sum_u32(n);
  if (__lane_id() == 0 && n != 0) atomicAdd(count, n);
}

/* the weights of histories first .. end - 1, as one history per thread of
   `threads` finds them, spread over all; pos: this thread's place */
__device__ __forceinline__ uint64_t mc_scale_place(uint64_t first, uint64_t end, uint64_t pos,
                                                   uint64_t threads) {
  const uint64_t n = end - first;
  if (n <= threads) return first + pos; /* may be end or beyond */
  const uint64_t i = (uint64_t)((double)pos * ((double)n / (double)threads));
  return first + (i < n ? i : n - 1);
}

/* the cells of a block's layer, by all its threads */
__device__ __forceinline__ void mc_scale_cells(mc_scale *s, const mc_cell *cells, int m,
                                               double dx) {
  double most = 0.0;
  for (int c = threadIdx.x; c < m; c += blockDim.x) {
    const double a = cells[c].sig_a;
    most = a > most ? a : most;
  }
  atomicMax(&s->thick, mc_ceil_log2(most * dx));
}

/* V: terms up to the largest weight in a layer of few cells.  In one of many
   cells a smaller V (a cell absorbs a small part of the weight) means rarer
   moves: the largest weight times 16 sig_a dx of the thickest cell (terms
   above need |mu| < 1/16 there, one crossing in 256), but no less than 2^-4
   or 2^-6 of the weight, where moves are rare enough.  With V from the number
   of cells alone, 2 M histories into the face of a layer of 10,000 cells with
   a mean sig_a dx of 0.011 took 67 ms, nearly every term in the global tally;
   now 2.0.  Largest weights seen by one history per thread, over the whole
   bank: a bank sorted by weight is seen whole. */
constexpr int MC_THICK_CELLS = 1024;
__device__ __forceinline__ mc_block_tally mc_block_tally_for(int m, const mc_scale &s, int waves) {
  mc_block_tally B;
  const int k = __builtin_amdgcn_readfirstlane(s.w);
  int less = 0;
  if (m >= MC_THICK_CELLS) {
    const int most = m < 4096 ? 4 : 6, thin = -4 - __builtin_amdgcn_readfirstlane(s.thick);
    less = thin < 0 ? 0 : (thin < most ? thin : most);
  }
  const int V = k - less;
  const int Vc = V < -30 ? -30 : (V > 2 ? 2 : V);
  B.limbs = V <= 2; /* an interval of at least 512 events per lane */
  B.S = mc_fx_split_for(Vc);
  const int lg = mc_fx_split_log2_terms(Vc);
  B.every = (int)((1u << (lg < 30 ? lg : 30)) / (64u * (unsigned)waves));
  return B;
}

/* A term that neither limb conversion takes: rounded to the resolution if it
   lies below, else to the global tally.  Returns what is left for the limbs.
   (Out of line: with the rounding inline the cycle loop, whose light particles
   often take mc_fx_split_small, went from 21.1 to 22.6 ms.) */
__device__ __noinline__ static double mc_tally_rest(unsigned long long *fx_lo,
                                                    unsigned long long *fx_hi, uint32_t *flags,
                                                    unsigned int *status, int c, double dw) {
  if (mc_fx_split_signed_tiny(&dw)) return dw;
  const mc_fx_flagged g = mc_fx_from_double_general(dw);
  if (g.flags) {
    atomicOr(&flags[c], g.flags);
    if (g.flags & 8u) atomicOr(status, 2u);
  }
  mc_fx_atomic_add(&fx_lo[c], &fx_hi[c], g.v);
  return 0.0;
}

/* A block's limb tally of m cells: 2^sh copies of every word, those of a cell
   side by side, first all of limb 0, then all of limb 1.  A lane adds to copy
   lane mod 2^sh: histories that enter a short layer together stay in the same
   cell all the way through (setting out apart would cost as many events as
   they have), and the adds of a wave to one word follow one another.  As many
   copies as fit a quarter of a CU's LDS, where four blocks of 256 run: larger
   blocks wait longer for their last histories.  Measured with one copy and
   with these: 2 M histories into both faces of a layer of 100 cells 1.32 ->
   0.90 ms, of 150 1.84 -> 1.11, of 250 2.91 -> 1.53, of 300 (where they set out
   apart) 1.94 both; the cycle loop on eight ranks of 125 cells 24.0 -> 20.9
   ms. */
struct mc_limbs {
  unsigned long long *t0, *t1; /* the words of cell 0 */
  int sh;
};

__device__ __forceinline__ mc_limbs mc_limbs_at(unsigned long long *t, int m, int sh) {
  return {t, t + ((size_t)m << sh), sh};
}

constexpr size_t MC_COPIES_LDS = 40960 - 256; /* static LDS */

/* log2 of the copies for m cells in `room` bytes */
__host__ __device__ __forceinline__ int mc_limbs_copies(int m, size_t room) {
  int sh = 0;
  while (sh < 5 && (32 * (size_t)m << sh) <= room) ++sh;
  return sh;
}

/* dynamic LDS with copies, for a block that needs `lds` bytes with one */
inline size_t mc_lds_with_copies(size_t lds, int m) {
  if (lds >= MC_COPIES_LDS) return lds;
  const int sh = mc_limbs_copies(m, MC_COPIES_LDS - lds + 16 * (size_t)m);
  return lds + (16 * (size_t)m << sh) - 16 * (size_t)m;
}

/* this lane's copy */
__device__ __forceinline__ mc_limbs mc_limbs_mine(const mc_limbs &T) {
  const int c = (int)(threadIdx.x & ((1u << T.sh) - 1u));
  return {T.t0 + c, T.t1 + c, T.sh};
}

/* add dw of `lanes` to cell c8 / 8 of the limb tally (T: this lane's copy),
   called by the whole wave; fx_lo, fx_hi: global tally */
__device__ __forceinline__ void mc_tally_limbs(const mc_limbs &T, const mc_fx_split &S,
                                               unsigned long long *fx_lo,
                                               unsigned long long *fx_hi, uint32_t *flags,
                                               unsigned int *status, mc_mask lanes, int c8,
                                               double dw) {
  const mc_mask take = lanes & mc_lanes(mc_fx_split_direct(dw, &S));
  if (__builtin_expect(take != lanes, 0)) { /* wave-uniform: small, large or special terms */
    if (mc_in(lanes & ~take) && !mc_fx_split_small(&dw))
      dw = mc_tally_rest(fx_lo, fx_hi, flags, status, c8 >> 3, dw);
  }
  if (mc_in(lanes)) {
    uint64_t n0, n1;
    mc_fx_split_limbs(dw, &S, &n0, &n1);
    atomicAdd(mc_word(T.t0, c8 << T.sh), (unsigned long long)n0);
    atomicAdd(mc_word(T.t1, c8 << T.sh), (unsigned long long)n1);
  }
}

/* move the limbs of cells first, first + step, ... to the global tally; any
   wave may do it while others add (each limb is exchanged with zero).  A
   lane takes the copies of its cell in an order of its own: the lanes' words
   lie in different banks.  (The copies' sums stay in 64 bits: the bound on
   the terms between two moves is for all copies together.) */
__device__ __forceinline__ void mc_limbs_move(const mc_limbs &T, int L, int m, int first, int step,
                                              unsigned long long *fx_lo,
                                              unsigned long long *fx_hi) {
  const int copies = 1 << T.sh;
  for (int c = first; c < m; c += step) {
    uint64_t n0 = 0, n1 = 0;
    for (int j = 0; j < copies; ++j) {
      const int at = (c << T.sh) + ((j + c) & (copies - 1));
      n0 += atomicExch(&T.t0[at], 0ull);
      n1 += atomicExch(&T.t1[at], 0ull);
    }
    if (n0 | n1) mc_fx_atomic_add(&fx_lo[c], &fx_hi[c], mc_fx_limbs(n0, n1, L));
  }
}

/* the rows of mc_abs_tab into LDS (all threads of the block; then a barrier) */
__device__ __forceinline__ void mc_tab_fill(double2 *tab) {
  for (int j = threadIdx.x; j < MC_ABS_N; j += blockDim.x)
    tab[j] = make_double2(mc_abs_tab[j][0], mc_abs_tab[j][1]);
}

/* The moves(k) of a limb tally: whole tables of m cells, by this wave. */
struct mc_mover {
  mc_limbs T;
  unsigned long long *fx_lo, *fx_hi;
  int m, L, every, left;
  __device__ __forceinline__ void operator()(int k) {
    if (left < k) { /* wave-uniform */
      mc_limbs_move(T, L, m, __lane_id(), 64, fx_lo, fx_hi);
      left = every;
    }
    left -= k;
  }
};

/* A tally that takes all of a block's LDS: the layer's first m cells, as limbs
   or as words with carry, the rows of mc_abs_tab read from memory; terms of the
   few cells beyond go to the global tally.  For layers whose tally fits LDS but
   not beside the rows (10,136 to 10,240 cells) where they cannot go in windows:
   with every term in the global tally 200,000 histories on 10,180 cells take
   176 ms, 2 M on thick ones 150; so 17.6 and 1.1 (10,240 cells, 16 of them
   beyond: 22.3; 10,100, beside the rows: 16.1). */
constexpr int MC_FULL_BEYOND = 16;

struct mc_full_tally {
  unsigned long long *t; /* LDS */
  int m;
  mc_block_tally B;
  unsigned long long *fx_lo, *fx_hi;
  uint32_t *flags;
  unsigned int *status;
  int left;
  __device__ __forceinline__ mc_limbs limbs() const { return mc_limbs_at(t, m, 0); }
  /* events between two calls of moves */
  __device__ __forceinline__ int every() const { return B.limbs ? B.every : 1 << 30; }
  __device__ __forceinline__ void moves(int k) {
    if (!B.limbs) return;
    if (left < k) { /* wave-uniform */
      mc_limbs_move(limbs(), B.S.L, m, __lane_id(), 64, fx_lo, fx_hi);
      left = B.every;
    }
    left -= k;
  }
  __device__ __forceinline__ void add(mc_mask lanes, int c8, double dw) const {
    const mc_mask beyond = lanes & mc_lanes(c8 >= 8 * m);
    if (beyond != 0) { /* wave-uniform */
      if (mc_in(beyond)) mc_tally(fx_lo, fx_hi, flags, status, c8 >> 3, dw);
      lanes &= ~beyond;
    }
    if (B.limbs)
      mc_tally_limbs(limbs(), B.S, fx_lo, fx_hi, flags, status, lanes, c8, dw);
    else if (mc_in(lanes))
      mc_tally(t, t + m, flags, status, c8 >> 3, dw);
  }
  /* to the global tally, by all threads after a barrier */
  __device__ __forceinline__ void out() const {
    if (B.limbs)
      mc_limbs_move(limbs(), B.S.L, m, threadIdx.x, blockDim.x, fx_lo, fx_hi);
    else
      for (int c = threadIdx.x; c < m; c += blockDim.x)
        mc_fx_atomic_add(&fx_lo[c], &fx_hi[c], mc_fx{t[c], t[m + c]});
  }
};

/* the m cells at `from` into LDS at `to`, with the pads of mc_walk_many's PAD
   (MC_PAD_BYTES more than the cells); returns the first cell's address */
constexpr size_t MC_PAD_BYTES = 2 * sizeof(mc_cell);
__device__ __forceinline__ mc_cell *mc_cells_fill(mc_cell *to, const mc_cell *from, int m) {
  for (int c = threadIdx.x; c < m; c += blockDim.x) to[c + 1] = from[c];
  if (threadIdx.x < 2) {
    mc_cell nan;
    nan.sig_a = nan.sig_i = __builtin_nan("");
    to[threadIdx.x ? m + 1 : 0] = nan;
  }
  return to + 1;
}

#endif /* MC_WALK_H */
