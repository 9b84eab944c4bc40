"""GPU: layers of more cells than 28 or 30 bits count, every kernel, against
the oracle on the few thousand cells at either end where the histories run."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
FIELDS = ("seed", "x", "mu", "wmc", "index")
DX, MIN_W, SPAN = 1.0, 5e-2, 4000


def _say(msg):
    print(msg, flush=True)


class _Huge:
    """m cells of width 1; histories in the first and the last SPAN / 2 cells
    and around cell 2^28, whose flights are some tens of cells."""

    def __init__(self, m):
        import torch
        from mcgpu import PARTICLE, configs
        self.m, n = m, 90
        rng = np.random.default_rng(m)
        self.parts = [(0, 0), (2 ** 28 - SPAN // 2, 1), (m - SPAN, 2)]
        self.bank = np.zeros(3 * n, dtype=PARTICLE)
        self.bank["seed"] = configs.seed_chain(3 * n)
        self.bank["mu"] = rng.uniform(-1, 1, 3 * n)
        self.bank["wmc"] = 1.0
        self.sig_a = torch.full((m,), 0.01, dtype=torch.float64, device="cuda")
        self.sig_i = torch.full((m,), 0.02, dtype=torch.float64, device="cuda")
        for lo, k in self.parts:
            first = (0, SPAN // 4, SPAN // 2)[k]
            at = lo + first + rng.integers(0, SPAN // 2, n)
            at[0] = (0, 2 ** 28, m - 1)[k]
            self.bank["index"][k * n:(k + 1) * n] = at
            self.bank["x"][k * n:(k + 1) * n] = at + rng.uniform(0.1, 0.9, n)
            sa, ss = rng.uniform(0.005, 0.02, SPAN), rng.uniform(0.01, 0.05, SPAN)
            self.sig_a[lo:lo + SPAN] = torch.from_numpy(sa).cuda()
            self.sig_i[lo:lo + SPAN] = torch.from_numpy(ss).cuda()
        self.n = n

    def part(self, k):
        lo, _ = self.parts[k]
        cut = slice(k * self.n, (k + 1) * self.n)
        return lo, cut, *(t[lo:lo + SPAN].cpu().numpy() for t in (self.sig_a, self.sig_i))


def _sum_over_parts(h, per_part):
    """per-part arrays of SPAN cells added up where parts overlap: {cell: value}"""
    import torch
    out = {}
    for (lo, _), v in zip(h.parts, per_part):
        for c in np.flatnonzero(v):
            out[lo + int(c)] = out.get(lo + int(c), 0.0) + v[c]
    idx = np.array(sorted(out), dtype=np.int64)
    return torch.from_numpy(idx).cuda(), np.array([out[int(i)] for i in idx])


def _check_cells(h, got, per_part):
    import torch
    idx, want = _sum_over_parts(h, per_part)
    assert torch.count_nonzero(got).item() == len(want)
    assert np.allclose(got[idx].cpu().numpy(), want, rtol=1e-14, atol=0)


@pytest.mark.parametrize("kernel,m", [("history", 2 ** 28 + 3000), ("event", 2 ** 28 + 3000),
                                      ("batch", 2 ** 28 + 3000), ("history", 2 ** 30 + 3000)])
def test_layers_of_more_than_2_28_cells(oracle, kernel, m):
    import mcgpu
    import torch
    _say(f"{kernel} m={m}")
    h = _Huge(m)
    # sigs = 1 cell rate, ar = its absorbed part, as the entry point takes them
    sigs = h.sig_a + h.sig_i
    ar = h.sig_a / sigs
    ref = []
    for k in range(3):
        lo, cut, sa, ss = h.part(k)
        s_, a_ = (t[lo:lo + SPAN].cpu().numpy() for t in (sigs, ar))
        o = oracle.simulate_bank(64, lo, SPAN, DX, MIN_W, s_, a_, h.bank[cut], nthread=8)
        ends = o["bank"]["index"]
        assert np.all((ends >= lo) | (lo == 0)) and np.all((ends < lo + SPAN) | (lo + SPAN == m))
        ref.append(o)
    with mcgpu.Context(0) as ctx:
        b = mcgpu.bank_to_device(h.bank)
        w = torch.zeros(m, dtype=torch.float64, device="cuda")
        r = torch.zeros(len(h.bank), dtype=torch.int8, device="cuda")
        if kernel == "batch":
            plan = mcgpu.Batch(ctx, [(0, m, DX, MIN_W, 0, 0, len(h.bank))], sigs, ar, w, b, r)
            st = plan.run()
            plan.close()
        else:
            st, _ = ctx.simulate_device(b, sigs, ar, w, 0, m, DX, MIN_W, result=r,
                                        options=mcgpu.make_options(kernel))
    got = mcgpu.bank_from_device(b)
    for f in FIELDS:
        assert np.array_equal(got[f], np.concatenate([o["bank"][f] for o in ref])), f
    assert np.array_equal(r.cpu().numpy().astype(np.int32),
                          np.concatenate([o["result"] for o in ref]))
    assert st["events"] == sum(int(o["events"].sum()) for o in ref)
    _check_cells(h, w, [o["tally_exact"] for o in ref])
    del sigs, ar, w, h
    torch.cuda.empty_cache()


@pytest.mark.parametrize("batched", [False, True])
def test_gradient_of_more_than_2_28_cells(oracle, batched):
    import mcgpu
    import torch
    m = 2 ** 28 + 3000
    _say(f"gradient m={m} batched={batched}")
    h = _Huge(m)
    g = torch.zeros(m, dtype=torch.float64, device="cuda")
    rng = np.random.default_rng(4)
    for k in range(3):
        lo = h.parts[k][0]
        g[lo:lo + SPAN] = torch.from_numpy(rng.uniform(-1, 1, SPAN)).cuda()
    score, ga, gi, tally = [], [], [], []
    for k in range(3):
        lo, cut, sa, ss = h.part(k)
        gk = g[lo:lo + SPAN].cpu().numpy()
        o = oracle.forward_cells(lo, SPAN, DX, MIN_W, sa, ss, h.bank[cut], g=gk)
        oa, oi = oracle.adjoint_cells(lo, SPAN, DX, MIN_W, sa, ss, h.bank[cut], gk,
                                      score=o["score"])
        score.append(o["score"])
        tally.append(o["tally_exact"])
        ga.append(oa)
        gi.append(oi)
    init = mcgpu.bank_to_device(h.bank)
    work = {f: v.clone() for f, v in init.items()}
    w, da, di = (torch.zeros(m, dtype=torch.float64, device="cuda") for _ in range(3))
    sc = torch.empty(len(h.bank), dtype=torch.float64, device="cuda")
    slabs = [(0, m, DX, MIN_W, 0, 0, len(h.bank))]
    with mcgpu.Context(0) as ctx:
        if batched:
            ctx.forward_cells_batch(slabs, work, h.sig_a, h.sig_i, w, g=g, history_score=sc)
            ctx.adjoint_cells_batch(slabs, init, h.sig_a, h.sig_i, g, da, di, history_score=sc)
        else:
            ctx.forward_cells(work, h.sig_a, h.sig_i, w, 0, m, DX, MIN_W, g=g, history_score=sc)
            ctx.adjoint_cells(init, h.sig_a, h.sig_i, 0, m, DX, MIN_W, g, da, di,
                              history_score=sc)
    assert np.array_equal(sc.cpu().numpy(), np.concatenate(score))
    _check_cells(h, w, tally)
    # where two parts meet, sums of both signs: against the larger of the two
    for got, parts in ((da, ga), (di, gi)):
        idx, want = _sum_over_parts(h, parts)
        assert np.allclose(got[idx].cpu().numpy(), want, rtol=1e-13,
                           atol=1e-14 * max(np.abs(p).max() for p in parts))
        mask = torch.ones(m, dtype=torch.bool, device="cuda")
        mask[idx] = False
        assert torch.count_nonzero(got[mask]).item() == 0
        del mask
    del g, w, da, di, h
    torch.cuda.empty_cache()


def test_more_cells_than_32_bits_are_refused(ctx):
    """max_index - min_index itself beyond 31 bits: an argument error, before
    any memory is touched."""
    import mcgpu
    from mcgpu._lib import Slab
    L, one = mcgpu.lib(), np.zeros(1)
    lo, hi = -(1 << 31), (1 << 31) - 1
    p = one.ctypes.data
    rc = L.mcgpu_simulate(ctx._h, 0, None, p, p, p, lo, hi, 1.0, 0.0, None, None, None)
    assert rc == mcgpu.ERR_ARG
    bank = mcgpu._bank_struct(mcgpu.bank_to_device(np.zeros(1, mcgpu.PARTICLE)))
    rc = L.mcgpu_simulate_device(ctx._h, 1, C.byref(bank), p, p, p, lo, hi, 1.0, 0.0, None, None,
                                 None, None, None, None)
    assert rc == mcgpu.ERR_ARG
    rc = L.mcgpu_forward_cells(ctx._h, 1, C.byref(bank), p, p, p, lo, hi, 1.0, 0.0, None, None,
                               None, None, None, None)
    assert rc == mcgpu.ERR_ARG
    rc = L.mcgpu_adjoint_cells(ctx._h, 1, C.byref(bank), p, p, lo, hi, 1.0, 0.0, p, None, p, p,
                               None, None, None)
    assert rc == mcgpu.ERR_ARG
    slab = Slab(lo, hi, 1.0, 0.0, 0, 0, 1)
    h = C.c_void_p()
    rc = L.mcgpu_batch_create(ctx._h, 1, C.byref(slab), p, p, p, 1, C.byref(bank), None, None,
                              C.byref(h))
    assert rc == mcgpu.ERR_ARG and not h
    rc = L.mcgpu_forward_cells_batch(ctx._h, 1, C.byref(slab), 1, C.byref(bank), p, p, p, None,
                                     None, None, None, None, None)
    assert rc == mcgpu.ERR_ARG
