"""Tally terms below 2^-36 (mc-mpi_amd/csrc/mc_fx.h), compiled for the host with
gcc: every one that is not negative has limbs, equal to the oracle's 128-bit
fixed-point conversion, down to subnormal numbers and zero."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SHIM = r"""
#include "mc_fx.h"
void tt_limbs(const double *v, long n, int V, int is_signed, uint64_t *out, int8_t *taken) {
  const mc_fx_split S = mc_fx_split_for(V);
  for (long i = 0; i < n; ++i) {
    double x = v[i];
    uint64_t n0, n1;
    taken[i] = is_signed ? mc_fx_split_signed_small(&x) || mc_fx_split_signed_tiny(&x)
                         : mc_fx_split_small(&x) || mc_fx_split_tiny(&x);
    if (!taken[i]) continue;
    mc_fx_split_limbs(x, &S, &n0, &n1);
    const mc_fx r = is_signed ? mc_fx_signed_limbs(n0, n1, S.L) : mc_fx_limbs(n0, n1, S.L);
    out[2 * i] = r.lo;
    out[2 * i + 1] = r.hi;
  }
}
"""


@pytest.mark.parametrize("V", [-30, 0, 2])
@pytest.mark.parametrize("signed", [0, 1])
def test_tiny_terms_have_limbs(tmp_path, oracle, V, signed):
    src, so = tmp_path / "tt.c", tmp_path / "libtt.so"
    src.write_text(SHIM)
    subprocess.run(["gcc", "-O2", "-std=gnu11", "-fPIC", "-shared", "-ffp-contract=off",
                    "-I", os.path.join(ROOT, "mc-mpi_amd", "csrc"), "-o", str(so), str(src), "-lm"],
                   check=True)
    L = C.CDLL(str(so))
    L.tt_limbs.argtypes = [C.c_void_p, C.c_long, C.c_int, C.c_int, C.c_void_p, C.c_void_p]
    rng = np.random.default_rng(31)
    p2 = np.ldexp(1.0, np.arange(-1074, -30))
    near = np.ldexp(1.0, -89) * (1 + rng.integers(-8, 9, 4000) * 2.0 ** -53)  # about the tie
    v = np.concatenate([p2, np.nextafter(p2, 0), np.nextafter(p2, 1), 1.5 * p2, near,
                        np.ldexp(rng.uniform(1, 2, 300_000), rng.integers(-110, -30, 300_000)),
                        [0.0, 5e-324, 1e-310]])
    v = np.concatenate([v, -v])
    out, taken = np.zeros(2 * len(v), np.uint64), np.zeros(len(v), np.int8)
    L.tt_limbs(v.ctypes.data, len(v), V, signed, out.ctypes.data, taken.ctypes.data)
    t = taken != 0
    small = np.abs(v) < 2.0 ** -36
    assert np.array_equal(t, small if signed else small & ~np.signbit(v))
    want, flags = oracle.fx_convert(v)
    assert not flags[t].any()
    assert np.array_equal(out.reshape(-1, 2)[t], want.reshape(-1, 2)[t])
