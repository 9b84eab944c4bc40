/*
 * mc_adjoint.h -- the gradient terms of a replayed event and their block
 * tallies, shared by the single-slab and the batched adjoint kernels.
 */
#ifndef MC_ADJOINT_H
#define MC_ADJOINT_H

#include "mc_walk.h"

/* Two signed limb tallies (sig_a, sig_i) of m cells in LDS: t[0..m) and
   t[m..2m) hold sig_a's limbs, t[2m..4m) sig_i's; the global accumulators'
   words lie `stride` apart: ga lo, ga hi, gi lo, gi hi. */
struct mc_grad_tally {
  unsigned long long *t; /* LDS limbs, or null: straight into fx */
  unsigned long long *fx;
  int64_t stride;
  uint32_t *flags_a, *flags_i;
  unsigned int *status;
  int m;
  mc_fx_split S;
  int every;
};

/* the largest sig_i of a block's cells, by all its threads */
__device__ __forceinline__ void mc_scale_scatter(mc_scale *s, const mc_cell *cells, int m) {
  double most = 0.0;
  for (int c = threadIdx.x; c < m; c += blockDim.x) {
    const double b = cells[c].sig_i;
    most = b > most ? b : most;
  }
  atomicMax(&s->b, mc_ceil_log2(most));
}

/* V: a term is at most about the largest target weight times the particle
   weight times a flight, or, where the history collides, 1 / sig_i: 1, 64
   cells (terms above need |mu| < 1/64, one crossing in 4,096) or 1 over the
   largest sig_i, whichever is most.  Larger terms go to fx.  Returns whether
   limbs serve (an interval of at least 64 events per lane between moves, with 16
   waves and k = 5); if not, t holds words with carry. */
__device__ __forceinline__ bool mc_grad_split(mc_grad_tally &G, const mc_scale &s, double dx,
                                              int waves) {
  const int flight = mc_ceil_log2(dx) + 6, b = __builtin_amdgcn_readfirstlane(s.b);
  const int free_path = b < -13 ? 0 : 1 - b; /* none: nothing scatters (MC_EPS < 2^-13) */
  const int longest = flight > free_path ? flight : free_path;
  const int k = __builtin_amdgcn_readfirstlane(s.w + s.g) + (longest > 0 ? longest : 0);
  const int V = k < -30 ? -30 : (k > 5 ? 5 : k);
  G.S = mc_fx_split_for(V);
  const int lg = mc_fx_split_signed_log2_terms(V);
  G.every = (int)((1u << (lg < 30 ? lg : 30)) / (64u * (unsigned)waves));
  return k <= 5;
}

enum { MC_GRAD_GLOBAL, MC_GRAD_LIMBS, MC_GRAD_CARRY }; /* fx; t as limbs; t with carry */

/* which: 0 sig_a, 1 sig_i; called by the whole wave */
template <int MODE>
__device__ __forceinline__ void mc_grad_add(const mc_grad_tally &G, int which, mc_mask lanes, int c8,
                                            double v) {
  lanes &= mc_lanes(v != 0.0); /* (NaN differs from 0) */
  unsigned long long *fx = G.fx + 2 * which * G.stride;
  uint32_t *flags = which ? G.flags_i : G.flags_a;
  if (MODE == MC_GRAD_GLOBAL) { /* c8 in units of MC_IN_MEMORY */
    if (mc_in(lanes)) mc_tally<true>(fx, fx + G.stride, flags, G.status, c8, v);
    return;
  }
  if (MODE == MC_GRAD_CARRY) {
    unsigned long long *t = G.t + 2 * which * G.m;
    if (mc_in(lanes)) mc_tally<true>(t, t + G.m, flags, G.status, c8 >> 3, v);
    return;
  }
  const mc_mask take = lanes & mc_lanes(mc_fx_split_signed_direct(v, &G.S));
  if (__builtin_expect(take != lanes, 0)) {
    if (mc_in(lanes & ~take) && !mc_fx_split_signed_small(&v))
      v = mc_tally_rest(fx, fx + G.stride, flags, G.status, c8 >> 3, v);
  }
  if (mc_in(lanes)) {
    uint64_t n0, n1;
    mc_fx_split_limbs(v, &G.S, &n0, &n1);
    unsigned long long *t = mc_word(G.t + 2 * which * G.m, c8);
    atomicAdd(t, (unsigned long long)n0);
    atomicAdd(t + G.m, (unsigned long long)n1);
  }
}

/* both tallies' limbs (or words) of cells first, first + step, ... to fx */
__device__ __forceinline__ void mc_grad_move(const mc_grad_tally &G, int first, int step,
                                             bool limbs = true) {
  for (int c = first; c < G.m; c += step)
    for (int w = 0; w < 2; ++w) {
      unsigned long long *t = G.t + 2 * w * G.m + c;
      const uint64_t n0 = atomicExch(t, 0ull), n1 = atomicExch(t + G.m, 0ull);
      unsigned long long *fx = G.fx + 2 * w * G.stride + c;
      if (n0 | n1)
        mc_fx_atomic_add(fx, fx + G.stride,
                         limbs ? mc_fx_signed_limbs(n0, n1, G.S.L) : mc_fx{n0, n1});
    }
}

struct mc_grad_mover {
  const mc_grad_tally &G;
  int left;
  __device__ __forceinline__ void operator()(int k) {
    if (left < k) { /* wave-uniform */
      mc_grad_move(G, __lane_id(), 64);
      left = G.every;
    }
    left -= k;
  }
};

/* A lane's replay: from the initial bank, with the history's score T known
   (HAVE_SCORE) or summed in a first replay (phase 0). */
template <bool HAVE_SCORE> struct mc_grad_io {
  const mcgpu_bank &init;
  const double *score;
  double T, P;
  int phase; /* 0: score replay, 1: gradient replay */
  __device__ __forceinline__ void read(int64_t i, mc_state &p) {
    p.seed = init.seed[i];
    p.x = init.x[i];
    p.mu = init.mu[i];
    p.wmc = init.wmc[i];
    p.index = init.index[i];
    P = 0.0;
  }
  static constexpr bool RESUMES = false;
  __device__ __forceinline__ int code(const mc_state &p, bool at_cap, const mc_layer_k &L) {
    return mc_end_code(p, at_cap, L);
  }
  __device__ __forceinline__ uint64_t load(int64_t i, mc_state &p) {
    read(i, p);
    T = HAVE_SCORE ? score[i] : 0.0;
    phase = HAVE_SCORE ? 1 : 0;
    return 0;
  }
  __device__ __forceinline__ bool store(int64_t i, mc_state &p, int code, uint64_t, uint32_t) {
    if (HAVE_SCORE || phase == 1 || code == 2) return false;
    read(i, p); /* score known: the same history again for the gradient */
    phase = 1;
    return true;
  }
};

/* one event of `lanes` (mc_walk_many's on_event) */
template <int MODE, bool HAVE_SCORE>
__device__ __forceinline__ void mc_grad_event(mc_grad_io<HAVE_SCORE> &io, const mc_grad_tally &G,
                                              const double *g, mc_mask lanes, int c8,
                                              const mc_cell &cell, bool coll, double di, double dw,
                                              double wmc) {
  double gc = 0.0;
  if (mc_in(lanes)) gc = *mc_word<MODE == MC_GRAD_GLOBAL ? MC_IN_MEMORY : MC_IN_LDS>(g, c8);
  if (!HAVE_SCORE) {
    const mc_mask first = lanes & mc_lanes(io.phase == 0);
    if (mc_in(first)) io.T = io.T + gc * dw;
    lanes &= ~first;
  }
  double term_a, term_i;
  mc_adjoint_terms(cell, coll, di, dw, gc, wmc, io.T, io.P, term_a, term_i);
  mc_grad_add<MODE>(G, 0, lanes, c8, term_a);
  mc_grad_add<MODE>(G, 1, lanes & mc_lanes(cell.sig_i > MC_EPS), c8, term_i);
  if (mc_in(lanes)) io.P = io.P + gc * dw;
}

#endif /* MC_ADJOINT_H */
