"""The ring positions of histories parked at a window's edge (mc-mpi_amd/csrc/
mc_ring.h), compiled for the host with gcc: runs and slots over the wrap of the
32-bit positions, which a call reaches after 2^32 parked histories."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SHIM = r"""
#include "mc_ring.h"
uint32_t rg_cap(uint32_t n) { return mc_ring_cap(n); }
uint32_t rg_slot(uint32_t p, uint32_t cap) { return mc_ring_slot(p, cap); }
/* planted: a run of the positions themselves */
static unsigned long long naive(uint32_t at, uint32_t size) {
  return (unsigned long long)at | (unsigned long long)(at + size) << 32;
}
/* waves take 64 at a time until the run is used up, then `late` more at once
   (waves that saw the run before it was); the slots handed out */
long rg_take(uint32_t at, uint32_t size, uint32_t cap, int planted, int late, uint32_t *slots,
             long room) {
  unsigned long long run = planted ? naive(at, size) : mc_ring_run(at, size);
  long n = 0;
  while (mc_ring_left(run) != 0 || late-- > 0) {
    const unsigned long long was = run;
    run += 64;
    uint32_t have = mc_ring_left(was);
    if (have > 64) have = 64;
    for (uint32_t r = 0; r < have; ++r) {
      if (n < room) slots[n] = mc_ring_slot(mc_ring_next(was) + r, cap);
      ++n;
    }
  }
  return n;
}
"""


@pytest.fixture(scope="module")
def rg(tmp_path_factory):
    d = tmp_path_factory.mktemp("rg")
    src, so = d / "rg.c", d / "librg.so"
    src.write_text(SHIM)
    subprocess.run(["gcc", "-O2", "-std=gnu11", "-fPIC", "-shared", "-ffp-contract=off",
                    "-I", os.path.join(ROOT, "mc-mpi_amd", "csrc"), "-o", str(so), str(src), "-lm"],
                   check=True)
    L = C.CDLL(str(so))
    L.rg_cap.restype = L.rg_slot.restype = C.c_uint32
    L.rg_cap.argtypes, L.rg_slot.argtypes = [C.c_uint32], [C.c_uint32, C.c_uint32]
    L.rg_take.restype = C.c_long
    L.rg_take.argtypes = [C.c_uint32, C.c_uint32, C.c_uint32, C.c_int, C.c_int, C.c_void_p,
                          C.c_long]
    return L


def _taken(rg, at, size, cap, planted=0):
    slots = np.zeros(size + 4096, np.uint32)
    n = rg.rg_take(at, size, cap, planted, 16, slots.ctypes.data, len(slots))
    return n, slots[:n] if n <= len(slots) else None


@pytest.mark.parametrize("n", [1, 2, 3, 1000, 8_000_000, (1 << 28) - 1, 1 << 28, 1 << 29])
def test_capacity(rg, n):
    cap = rg.rg_cap(n)
    assert cap >= n and cap & (cap - 1) == 0 and cap < 2 * n


@pytest.mark.parametrize("n", [1, 100, 4097, 200_000])
@pytest.mark.parametrize("at", [0, 64, (1 << 31) - 5, 1 << 31, (1 << 32) - 64, (1 << 32) - 1])
def test_a_run_hands_out_its_positions_and_no_other(rg, n, at):
    cap = rg.rg_cap(n)
    got, slots = _taken(rg, at, n, cap)
    assert got == n
    want = (at + np.arange(n, dtype=np.uint64)) % np.uint64(1 << 32) % np.uint64(cap)
    assert np.array_equal(slots, want)
    # positions claimed one after the other lie in different slots, over the wrap too
    assert len(np.unique(slots)) == n


def test_planted_run_of_whole_positions_is_caught(rg):
    """Whole positions carry from next into end at the wrap."""
    n = 100
    got, slots = _taken(rg, (1 << 32) - 10, n, rg.rg_cap(n), planted=1)
    assert got != n
