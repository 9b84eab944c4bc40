/*
 * mc_ring.h -- positions in the rings of histories parked at a window's edge
 * (history.hip).  Integer code only, so it compiles as HIP device code and as
 * plain host C (gcc) for CPU-side tests; the device kernels use this source.
 *
 * put[] and got[] count positions in 32 bits and wrap: a history may be parked
 * many times, and a ring takes more than 2^32 of them in a long call.  So a
 * ring's slots are a power of two: the slot of a position, its low bits, goes
 * on evenly over the wrap.  A block holds a run of claimed positions as one
 * 64-bit word, next below end, from which its waves take by adding to it;
 * next starts below 2^31, so that neither the run (2^29 at most) nor what
 * waves take past its end (64 each) can carry into end.
 */
#ifndef MC_RING_H
#define MC_RING_H

#include <stdint.h>

#include "mc_fx.h" /* MC_FN_HD */

/* The count at which the positions of a call start: every call passes the wrap. */
#define MC_RING_START 0xFFFFFFC0u

/* slots for n histories (n <= 2^29) */
MC_FN_HD uint32_t mc_ring_cap(uint32_t n) {
  uint32_t cap = 1;
  while (cap < n) cap <<= 1;
  return cap;
}

MC_FN_HD uint32_t mc_ring_slot(uint32_t position, uint32_t cap) { return position & (cap - 1u); }

/* the run of `size` positions from `at` on */
MC_FN_HD unsigned long long mc_ring_run(uint32_t at, uint32_t size) {
  const uint32_t next = at & 0x7FFFFFFFu;
  return (unsigned long long)next | (unsigned long long)(next + size) << 32;
}

MC_FN_HD uint32_t mc_ring_next(unsigned long long run) { return (uint32_t)run; }

/* positions left in a run */
MC_FN_HD uint32_t mc_ring_left(unsigned long long run) {
  const int32_t left = (int32_t)((uint32_t)(run >> 32) - (uint32_t)run);
  return left > 0 ? (uint32_t)left : 0u;
}

#endif /* MC_RING_H */
