"""The arithmetic of the transport kernels' common step (mc-mpi_amd/csrc/
mc_math.h, mc_fx.h), compiled for the host with gcc: the absorbed fraction
1 - RN(exp(-y)) against the oracle's correctly rounded exp, and the two-limb
form of a tally term against the oracle's 128-bit fixed-point conversion."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SHIM = r"""
#include <stdint.h>
#include "mc_fx.h"
void pw_absorb(const double *y, long n, int row, double *u, int8_t *ok) {
  const mc_abs_coef K = mc_abs_coef_default();
  for (long i = 0; i < n; ++i) {
    double rem;
    if (row) {
      const unsigned k = mc_abs_index(y[i]);
      u[i] = k < MC_ABS_N ? mc_absorb_row(y[i], mc_abs_tab[k][0], mc_abs_tab[k][1], &K, &rem)
                          : (rem = 1.0);
    } else {
      u[i] = mc_absorb_thin(y[i], 0.75, &K, &rem);
    }
    ok[i] = __builtin_fabs(rem) < MC_ABS_REM;
  }
}
/* taken: 1 directly, 2 as a small term, 0 not by the limbs */
void pw_limbs(const double *v, long n, int V, uint64_t *out, int8_t *taken, uint64_t *n0s,
              uint64_t *n1s) {
  const mc_fx_split S = mc_fx_split_for(V);
  for (long i = 0; i < n; ++i) {
    double x = v[i];
    taken[i] = mc_fx_split_direct(x, &S) ? 1 : (mc_fx_split_small(&x) ? 2 : 0);
    out[2 * i] = out[2 * i + 1] = n0s[i] = n1s[i] = 0;
    if (!taken[i]) continue;
    mc_fx_split_limbs(x, &S, &n0s[i], &n1s[i]);
    const mc_fx r = mc_fx_limbs(n0s[i], n1s[i], S.L);
    out[2 * i] = r.lo;
    out[2 * i + 1] = r.hi;
  }
}
void pw_signed_limbs(const double *v, long n, int V, uint64_t *out, int8_t *taken, uint64_t *n0s,
                     uint64_t *n1s) {
  const mc_fx_split S = mc_fx_split_for(V);
  for (long i = 0; i < n; ++i) {
    double x = v[i];
    taken[i] = mc_fx_split_signed_direct(x, &S) ? 1 : (mc_fx_split_signed_small(&x) ? 2 : 0);
    out[2 * i] = out[2 * i + 1] = n0s[i] = n1s[i] = 0;
    if (!taken[i]) continue;
    mc_fx_split_limbs(x, &S, &n0s[i], &n1s[i]);
    const mc_fx r = mc_fx_signed_limbs(n0s[i], n1s[i], S.L);
    out[2 * i] = r.lo;
    out[2 * i + 1] = r.hi;
  }
}
void pw_quotient(const double *a, const double *b, long n, double *q) {
  for (long i = 0; i < n; ++i) {
    const double rh = 1.0 / b[i], rl = mc_fma(-b[i], rh, 1.0) * rh;
    q[i] = mc_div_by_pair(a[i], b[i], rh, rl);
  }
}
/* 1 + (the top 20 of h's 32 high bits) + sig_i di < 2 - 2^-18 */
void pw_crosses(const uint32_t *sh, const double *sig_i, const double *di, long n, int8_t *sure) {
  for (long i = 0; i < n; ++i) {
    const double h1 = mc_asf64((uint64_t)(0x3FF00000u | (sh[i] >> 12)) << 32);
    sure[i] = mc_fma(sig_i[i], di[i], h1) < 2.0 - 0x1p-18;
  }
}
int pw_signed_log2_terms(int V) { return mc_fx_split_signed_log2_terms(V); }
int pw_L(int V) { return mc_fx_split_for(V).L; }
int pw_log2_terms(int V) { return mc_fx_split_log2_terms(V); }
void pw_join(const uint64_t *n0, const uint64_t *n1, long n, int L, uint64_t *out) {
  for (long i = 0; i < n; ++i) {
    const mc_fx r = mc_fx_limbs(n0[i], n1[i], L);
    out[2 * i] = r.lo;
    out[2 * i + 1] = r.hi;
  }
}
"""


@pytest.fixture(scope="module")
def pw(tmp_path_factory):
    d = tmp_path_factory.mktemp("pw")
    src = d / "pw.c"
    src.write_text(SHIM)
    so = d / "libpw.so"
    subprocess.run(["gcc", "-O2", "-std=gnu11", "-fPIC", "-shared", "-ffp-contract=off",
                    "-I", os.path.join(ROOT, "mc-mpi_amd", "csrc"), "-o", str(so), str(src), "-lm"],
                   check=True)
    L = C.CDLL(str(so))
    p, n, i = C.c_void_p, C.c_long, C.c_int
    L.pw_absorb.argtypes = [p, n, i, p, p]
    L.pw_limbs.argtypes = L.pw_signed_limbs.argtypes = [p, n, i, p, p, p, p]
    L.pw_join.argtypes = [p, p, n, i, p]
    L.pw_quotient.argtypes = [p, p, n, p]
    L.pw_crosses.argtypes = [p, p, p, n, p]
    return L


def _fractions(lo, hi):
    """y in [2^lo, 2^hi), next to the rows' ends and to the grid's midpoints."""
    rng = np.random.default_rng(21)
    y = 2.0 ** rng.uniform(lo, hi, 1_500_000)
    k = np.arange(1, 89)
    ends = (k + 0.5) / 128.0
    ends = np.concatenate([np.nextafter(ends, 0), ends, np.nextafter(ends, 1), k / 128.0])
    mids = (np.arange(1, 200_001) - 0.5) * 2.0 ** -53 * 2.0 ** rng.integers(0, 44, 200_000)
    return np.concatenate([y, ends, mids, np.nextafter(mids, 0), np.nextafter(mids, 1),
                           [0.0, 5e-324, 2.0 ** -54, 2.0 ** -53, 2.0 ** -1000]])


@pytest.mark.parametrize("row", [0, 1])
def test_absorbed_fraction_is_certified_exactly(pw, oracle, row):
    """Where the rounding is certified, u equals 1 - RN(exp(-y)) bit for bit;
    about one argument in 8,000 is not (in a random sample: at most 1 in 4,000)."""
    top = 0.6875 if row else 2.0 ** -8
    for lo, hi in ((-40, -0.54), (-14, -6)):
        y = _fractions(lo, hi)
        y = y[(y <= top) if row else (y < top)]
        u, ok = np.empty_like(y), np.empty(len(y), np.int8)
        pw.pw_absorb(y.ctypes.data, len(y), row, u.ctypes.data, ok.ctypes.data)
        want = 1 - oracle.math_eval("exp", -y)
        bad = (ok != 0) & (u.view(np.uint64) != want.view(np.uint64))
        assert not bad.any(), y[bad][:5]
        rnd = 2.0 ** np.random.default_rng(22).uniform(-16, np.log2(top), 400_000)
        pw.pw_absorb(rnd.ctypes.data, len(rnd), row, u.ctypes.data, ok.ctypes.data)
        assert (ok[:len(rnd)] == 0).mean() < 1 / 4000


def test_absorbed_fraction_catches_a_loose_certificate(pw, oracle):
    """With the certificate's margin dropped (every u accepted), arguments whose
    exponential lies next to a midpoint come out wrong: the sample above holds
    such arguments."""
    y = _fractions(-8, -0.55)
    y = y[(y > 2.0 ** -8) & (y <= 0.6875)]
    u, ok = np.empty_like(y), np.empty(len(y), np.int8)
    pw.pw_absorb(y.ctypes.data, len(y), 1, u.ctypes.data, ok.ctypes.data)
    want = 1 - oracle.math_eval("exp", -y)
    assert (u != want).any()


@pytest.mark.parametrize("V", [-30, -7, -6, -1, 0, 1, 2])
def test_limbs_equal_the_fixed_point_term(pw, oracle, V):
    """n1 2^L + n0 is the oracle's integer for every term that the limbs take;
    every non-negative term below 2^V (down to 2^-88, and zero) is taken, no
    term of 2^V or more, negative or not finite; |n0| <= 2^(L-1) and
    n1 <= 2^(V+88-L), as the interval between two moves assumes."""
    rng = np.random.default_rng(23)
    e = np.arange(-1074, 42)
    p2 = np.ldexp(1.0, e)
    v = np.concatenate([p2, np.nextafter(p2, 0), np.nextafter(p2, np.inf), p2 * 1.5, -p2,
                        rng.uniform(1, 2, 600_000) * np.ldexp(1.0, rng.integers(-95, V + 2, 600_000)),
                        (2 * rng.integers(0, 2 ** 51, 200_000) + 1) * np.ldexp(
                            0.5 ** 88, -rng.integers(0, 52, 200_000)) * 0.5,  # ties and near ties
                        [0.0, -0.0, np.inf, -np.inf, np.nan]])
    v = np.ascontiguousarray(v)
    n = len(v)
    out, n0, n1 = np.zeros(2 * n, np.uint64), np.zeros(n, np.uint64), np.zeros(n, np.uint64)
    taken = np.zeros(n, np.int8)
    pw.pw_limbs(v.ctypes.data, n, V, out.ctypes.data, taken.ctypes.data, n0.ctypes.data,
                n1.ctypes.data)
    should = ((v == 0) & ~np.signbit(v)) | ((v >= 2.0 ** -88) & (v < max(2.0 ** V, 2.0 ** -36)))
    assert np.array_equal(taken != 0, should)
    want, fl = oracle.fx_convert(v)
    t = taken != 0
    assert not fl[t].any()
    assert np.array_equal(out.reshape(-1, 2)[t], want.reshape(-1, 2)[t])
    L = pw.pw_L(V)
    assert np.abs(n0[t].view(np.int64)).max() <= 2 ** (L - 1)
    assert n1[t].max() <= 2 ** max(V + 88 - L, 52 - L)
    lg = pw.pw_log2_terms(V)
    assert lg + L - 1 <= 63 and lg + V + 88 - L <= 64


@pytest.mark.parametrize("V", [-35, 5, 13, 14])
def test_limbs_to_the_ends_of_the_stated_range(pw, oracle, V):
    """mc_fx_split_for's range; one further, terms next to 2^V come out wrong."""
    test_limbs_equal_the_fixed_point_term(pw, oracle, V)
    if V == 14:
        with pytest.raises(AssertionError):
            test_limbs_equal_the_fixed_point_term(pw, oracle, V + 1)


@pytest.mark.parametrize("V", [-30, -3, 0, 2, 5])
def test_signed_limbs_equal_the_fixed_point_term(pw, oracle, V):
    """The same for terms of either sign (the gradients')."""
    rng = np.random.default_rng(25)
    p2 = np.ldexp(1.0, np.arange(-1074, 42))
    v = np.concatenate([p2, np.nextafter(p2, 0), np.nextafter(p2, np.inf), p2 * 1.5,
                        rng.uniform(1, 2, 400_000) * np.ldexp(1.0, rng.integers(-95, V + 2, 400_000)),
                        (2 * rng.integers(0, 2 ** 51, 200_000) + 1) * np.ldexp(
                            0.5 ** 88, -rng.integers(0, 52, 200_000)) * 0.5, [np.inf, np.nan]])
    v = np.concatenate([v, -v])
    n = len(v)
    out, n0, n1 = np.zeros(2 * n, np.uint64), np.zeros(n, np.uint64), np.zeros(n, np.uint64)
    taken = np.zeros(n, np.int8)
    pw.pw_signed_limbs(v.ctypes.data, n, V, out.ctypes.data, taken.ctypes.data, n0.ctypes.data,
                       n1.ctypes.data)
    a = np.abs(v)
    t = taken != 0
    assert np.array_equal(t, (a == 0) | ((a >= 2.0 ** -88) & (a < max(2.0 ** V, 2.0 ** -36))))
    want, fl = oracle.fx_convert(v)
    assert not fl[t].any()
    assert np.array_equal(out.reshape(-1, 2)[t], want.reshape(-1, 2)[t])
    L, lg = pw.pw_L(V), pw.pw_signed_log2_terms(V)
    assert np.abs(n0[t].view(np.int64)).max() <= 2 ** (L - 1)
    assert np.abs(n1[t].view(np.int64)).max() <= 2 ** max(V + 88 - L, 52 - L)
    assert lg + L - 1 <= 63 and lg + V + 88 - L <= 63


def test_limb_sums_join_with_borrow_and_carry(pw):
    """The joined sum of many terms: limb 0 of either sign, limb 1 up to 2^64 - 1."""
    rng = np.random.default_rng(24)
    n0 = rng.integers(-2 ** 62, 2 ** 62, 5000).astype(np.int64)
    n0[:4] = [0, -1, 2 ** 62, -2 ** 62]
    n1 = rng.integers(0, 2 ** 63, 5000, dtype=np.uint64) * np.uint64(2) + np.uint64(1)
    n1[:3] = [0, 1, 2 ** 64 - 1]
    n0 = np.where((n1 < 2 ** 30) & (n0 < 0), -n0, n0)
    for L in (29, 40, 41, 44, 45):
        out = np.zeros(10_000, np.uint64)
        u0 = n0.view(np.uint64).copy()
        pw.pw_join(u0.ctypes.data, n1.ctypes.data, 5000, L, out.ctypes.data)
        for i in range(5000):
            s = (int(n1[i]) << L) + int(n0[i])
            assert (int(out[2 * i + 1]) << 64 | int(out[2 * i])) == s % (1 << 128)


def test_edge_quotient_is_the_ieee_division(pw):
    """a / b by the pair equals the division over the stated ranges: random,
    next to a representable or halfway quotient, powers of two, and zero."""
    rng = np.random.default_rng(26)
    n = 3_000_000
    b = rng.uniform(1, 2, n) * np.ldexp(1.0, rng.integers(-60, 64, n)) * rng.choice([-1.0, 1.0], n)
    b[: n // 2] = rng.uniform(-1, 1, n // 2)
    b[np.abs(b) < 1e-12] = 1.0
    a = rng.uniform(1, 2, n) * np.ldexp(1.0, rng.integers(-752, 700, n)) * rng.choice([-1.0, 1.0], n)
    k = slice(0, n // 2, 2)
    q = rng.uniform(1, 2, a[k].size)
    a[k] = q * b[k]  # quotients next to a double
    a[k] = np.nextafter(a[k], rng.choice([-np.inf, 0, np.inf], a[k].size))
    k = slice(1, n // 2, 2)
    a[k] = rng.integers(0, 1000, a[k].size) * 1e-3 - rng.uniform(0, 1, a[k].size)
    p2 = np.ldexp(1.0, np.arange(-60, 65))
    b = np.concatenate([b, p2, np.nextafter(p2[1:-1], 0), np.nextafter(p2[:-1], np.inf), [1.0, -3.0]])
    a = np.concatenate([a, rng.uniform(-1, 1, b.size - n)])
    a[-2:] = 0.0
    got = np.empty_like(a)
    pw.pw_quotient(a.ctypes.data, b.ctypes.data, a.size, got.ctypes.data)
    assert np.array_equal(got, a / b)


def test_crossing_by_20_bits_never_takes_a_collision(pw, oracle):
    """Where the 20-bit sum certifies a crossing, the sampled flight
    -log(h) / sig_i is not below the way to the edge; cells whose sum lies next
    to the limit are in the sample, and both answers occur."""
    rng = np.random.default_rng(27)
    n = 1_000_000
    sh = rng.integers(0, 2 ** 32, n, dtype=np.uint64).astype(np.uint32)
    h = sh * 2.0 ** -32 + rng.integers(0, 2 ** 31, n) * 2.0 ** -63
    sig = 2.0 ** rng.uniform(-30, 12, n)
    reach = 2.0 ** rng.uniform(-30, 0.1, n)
    reach[::2] = np.maximum(1 - h[::2], 2.0 ** -30) * (1 + rng.normal(0, 1, n // 2) * 2.0 ** -17)
    reach[::8] = 0.0
    di = reach / sig
    sure = np.empty(n, np.int8)
    pw.pw_crosses(sh.ctypes.data, sig.ctypes.data, di.ctypes.data, n, sure.ctypes.data)
    sure = sure != 0
    assert 0.1 < sure.mean() < 0.9
    h = np.maximum(h, 2.0 ** -63)
    flight = -oracle.math_eval("log", h) / sig
    assert not (flight[sure] < di[sure]).any()
    near = sure & (1 - h < reach * (1 + 2.0 ** -14)) & (reach > 2.0 ** -3)
    assert near.any()
