"""GPU: layers and slabs whose tally just fits a block's LDS, beside the rows of
the absorbed fraction, without them, and with a few cells beyond: bit-identical
to the oracle, and no step in time."""
import ctypes as C
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _say(msg):
    print(msg, flush=True)


def _case(m, n, wmc, thick=1.0):
    from mcgpu import PARTICLE, configs
    rng = np.random.default_rng(m + n)
    sigs, ar = thick * rng.lognormal(0.3, 0.6, m), rng.uniform(0.05, 0.95, m)
    bank = np.zeros(n, dtype=PARTICLE)
    bank["seed"] = configs.seed_chain(n)
    bank["index"] = rng.integers(0, m, n)
    bank["index"][::3] = m - 1 - rng.integers(0, 40, len(bank[::3]))  # the last cells
    bank["x"] = (bank["index"] + rng.random(n)) / m
    bank["mu"] = rng.uniform(-1, 1, n)
    bank["wmc"] = wmc
    return sigs, ar, 1.0 / m, bank


def _noalloc(bank, sigs, ar, w, m, dx, min_w, result=None):
    import torch
    import mcgpu
    from mcgpu import _bank_struct, _ptr, lib
    b, opt = _bank_struct(bank), mcgpu.make_options()
    rc = lib().mcgpu_simulate_device_noalloc(
        bank["x"].numel(), C.byref(b), _ptr(sigs), _ptr(ar), _ptr(w), 0, m, dx, min_w,
        _ptr(result), None, None, C.byref(opt), None, torch.cuda.current_stream().cuda_stream)
    assert rc == 0


def _dev(x):
    import torch
    return torch.from_numpy(np.ascontiguousarray(x)).cuda()


@pytest.mark.parametrize("wmc", [1.0, 50.0])
@pytest.mark.parametrize("m", [10_135, 10_136, 10_224, 10_225, 10_240, 10_241])
@pytest.mark.parametrize("how", ["noalloc", "one_block"])
def test_layers_whose_tally_fills_lds(ctx, oracle, how, m, wmc):
    """Without allocation, and on one block (too few for windows)."""
    import mcgpu
    _say(f"tally fills LDS {how} m={m} weights {wmc}")
    n, min_w = 600, 0.05 * wmc
    sigs, ar, dx, bank = _case(m, n, wmc, 30.0)
    o = oracle.simulate_bank(64, 0, m, dx, min_w, sigs, ar, bank, nthread=8)
    db, dw, dr = mcgpu.bank_to_device(bank), _dev(np.zeros(m)), _dev(np.zeros(n, np.int8))
    if how == "noalloc":
        _noalloc(db, _dev(sigs), _dev(ar), dw, m, dx, min_w, dr)
    else:
        ctx.simulate_device(db, _dev(sigs), _dev(ar), dw, 0, m, dx, min_w, result=dr,
                            options=mcgpu.make_options("history", grid_blocks=1))
    b = mcgpu.bank_from_device(db)
    for f in ("seed", "x", "mu", "wmc", "index"):
        assert np.array_equal(b[f], o["bank"][f]), f
    assert np.array_equal(dr.cpu().numpy().astype(np.int32), o["result"])
    assert np.array_equal(dw.cpu().numpy(), o["tally_exact"])


def _fastest(run, prepare, times=4):
    import torch
    best = 1e9
    for _ in range(times):
        prepare()
        torch.cuda.synchronize()
        t = time.perf_counter()
        run()
        torch.cuda.synchronize()
        best = min(best, time.perf_counter() - t)
    return best


def test_no_step_in_time_where_the_tally_fills_lds():
    """Thick cells, 300,000 histories from one face: with every term in the
    global tally 10,200 cells take some 77 times as long as 10,100."""
    import mcgpu
    t = {}
    for m in (10_100, 10_200):
        sigs, ar, dx, bank = _case(m, 300_000, 1.0, 1000.0)
        bank["index"], bank["x"], bank["mu"] = 0, 0.0, np.abs(bank["mu"])
        init, ds, da, w = mcgpu.bank_to_device(bank), _dev(sigs), _dev(ar), _dev(np.zeros(m))
        work = {k: v.clone() for k, v in init.items()}
        t[m] = _fastest(lambda: _noalloc(work, ds, da, w, m, dx, 1e-3),
                        lambda: [work[k].copy_(v) for k, v in init.items()])
        _say(f"no allocation, {m} thick cells: {1e3 * t[m]:.3f} ms")
    assert t[10_200] < 3 * t[10_100]


@pytest.mark.parametrize("wmc", [1.0, 50.0])
@pytest.mark.parametrize("grid", [0, 2])
def test_slabs_whose_tally_fills_lds(ctx, oracle, grid, wmc):
    """Slabs around the limits in one plan, small ones between them: on two
    blocks each takes slabs of every kind, the rows put back after each."""
    import mcgpu
    _say(f"slabs that fill LDS grid={grid} weights {wmc}")
    ms, n, min_w = [10_135, 300, 10_136, 10_224, 40, 10_225, 10_240, 2000, 10_241, 33], 250, 0.05 * wmc
    cases = [_case(m, n, wmc, 30.0 * m / 10_000) for m in ms]
    off = np.concatenate([[0], np.cumsum(ms)])
    slabs = [(0, m, 1.0 / m, min_w, int(off[s]), s * n, n) for s, m in enumerate(ms)]
    sigs, ar = (np.concatenate([c[k] for c in cases]) for k in (0, 1))
    db = mcgpu.bank_to_device(np.concatenate([c[3] for c in cases]))
    dw, dr = _dev(np.zeros(off[-1])), _dev(np.zeros(n * len(ms), np.int8))
    plan = mcgpu.Batch(ctx, slabs, _dev(sigs), _dev(ar), dw, db, dr,
                       options=mcgpu.make_options(grid_blocks=grid))
    plan.run()
    plan.close()
    b, w, r = mcgpu.bank_from_device(db), dw.cpu().numpy(), dr.cpu().numpy()
    for s, (m, (sg, a, dx, bank)) in enumerate(zip(ms, cases)):
        o = oracle.simulate_bank(64, 0, m, dx, min_w, sg, a, bank, nthread=8)
        part = slice(s * n, (s + 1) * n)
        for f in ("seed", "x", "mu", "wmc", "index"):
            assert np.array_equal(b[f][part], o["bank"][f]), (m, f)
        assert np.array_equal(r[part].astype(np.int32), o["result"]), m
        assert np.array_equal(w[off[s]:off[s + 1]], o["tally_exact"]), m


def test_no_step_in_time_where_a_slabs_tally_fills_lds(ctx):
    """As for layers: four slabs of thick cells."""
    import mcgpu
    t = {}
    for m in (10_100, 10_200):
        n = 100_000
        cases = [_case(m, n, 1.0, 1000.0) for _ in range(4)]
        for _, _, _, bank in cases:
            bank["index"], bank["x"], bank["mu"] = 0, 0.0, np.abs(bank["mu"])
        sigs, ar = (np.concatenate([c[k] for c in cases]) for k in (0, 1))
        init = mcgpu.bank_to_device(np.concatenate([c[3] for c in cases]))
        work = {k: v.clone() for k, v in init.items()}
        plan = mcgpu.Batch(ctx, [(0, m, 1.0 / m, 1e-3, s * m, s * n, n) for s in range(4)],
                           _dev(sigs), _dev(ar), _dev(np.zeros(4 * m)), work)
        t[m] = _fastest(plan.run, lambda: [work[k].copy_(v) for k, v in init.items()])
        plan.close()
        _say(f"batch, {m} thick cells: {1e3 * t[m]:.3f} ms")
    assert t[10_200] < 3 * t[10_100]


@pytest.mark.parametrize("wmc", [1.0, 50.0])
@pytest.mark.parametrize("score", [True, False])
def test_gradient_slabs_around_the_lds_limits(ctx, oracle, score, wmc):
    """Forward (with scores and without) and gradient of slabs on both sides of
    every limit: cells and tallies in LDS, the tallies alone, neither; on two
    blocks, each taking slabs of every kind."""
    import mcgpu
    import torch
    _say(f"gradient slabs score={score} weights {wmc}")
    ms, n, min_w = [2895, 2896, 300, 4053, 4054, 5066, 40, 5067, 5068, 10_135, 10_136], 60, 0.05 * wmc
    rng = np.random.default_rng(12)
    cases, g = [], []
    for m in ms:
        sigs, ar, dx, bank = _case(m, n, wmc, m / 300.0)
        cases.append((sigs * ar, sigs * (1 - ar), dx, bank))
        g.append(rng.uniform(-1, 1, m))
    off = np.concatenate([[0], np.cumsum(ms)])
    total = int(off[-1])
    slabs = [(0, m, 1.0 / m, min_w, int(off[s]), s * n, n) for s, m in enumerate(ms)]
    sa, si = (_dev(np.concatenate([c[k] for c in cases])) for k in (0, 1))
    dg = _dev(np.concatenate(g))
    init = mcgpu.bank_to_device(np.concatenate([c[3] for c in cases]))
    work = {k: v.clone() for k, v in init.items()}
    w, ga, gi = (torch.zeros(total, dtype=torch.float64, device="cuda") for _ in range(3))
    sc = torch.empty(n * len(ms), dtype=torch.float64, device="cuda")
    opt = mcgpu.make_options(grid_blocks=2)
    ctx.forward_cells_batch(slabs, work, sa, si, w, g=dg if score else None,
                            history_score=sc if score else None, options=opt)
    ctx.adjoint_cells_batch(slabs, init, sa, si, dg, ga, gi, history_score=sc if score else None,
                            options=opt)
    same = lambda t, x: np.array_equal(t.cpu().numpy().view(np.uint64), x.view(np.uint64))  # noqa: E731
    b = mcgpu.bank_from_device(work)
    for s, m in enumerate(ms):
        a_, i_, dx, bank = cases[s]
        o = oracle.forward_cells(0, m, dx, min_w, a_, i_, bank, g=g[s])
        oa, oi = oracle.adjoint_cells(0, m, dx, min_w, a_, i_, bank, g[s],
                                      score=o["score"] if score else None)
        cut, part = slice(off[s], off[s + 1]), slice(s * n, (s + 1) * n)
        for f in ("seed", "x", "mu", "wmc", "index"):
            assert np.array_equal(b[f][part], o["bank"][f]), (m, f)
        assert same(w[cut], o["tally_exact"]), m
        assert not score or same(sc[part], o["score"]), m
        assert same(ga[cut], oa) and same(gi[cut], oi), m


@pytest.mark.parametrize("what,below,above", [("forward", 5060, 5100), ("score", 4050, 4080),
                                              ("adjoint", 2890, 2910)])
def test_no_step_in_time_where_a_slabs_cells_fill_lds(ctx, what, below, above):
    """Eight slabs of thick cells, all histories from one face, where the
    global accumulators' adds to one word follow one another."""
    import mcgpu
    import torch
    t = {}
    for m in (below, above):
        n, k = 50_000, 8
        sigs, ar, dx, bank = _case(m, n, 1.0, 1000.0)
        bank["index"], bank["x"], bank["mu"] = 0, 0.0, np.abs(bank["mu"])
        sa, si = _dev(np.tile(sigs * ar, k)), _dev(np.tile(sigs * (1 - ar), k))
        g = torch.ones(k * m, dtype=torch.float64, device="cuda")
        init = mcgpu.bank_to_device(np.tile(bank, k))
        work = {f: v.clone() for f, v in init.items()}
        w, ga, gi = (torch.zeros(k * m, dtype=torch.float64, device="cuda") for _ in range(3))
        sc = torch.zeros(k * n, dtype=torch.float64, device="cuda")
        slabs = [(0, m, dx, 1e-3, s * m, s * n, n) for s in range(k)]
        with_score = {"g": g, "history_score": sc} if what != "forward" else {}
        run = lambda: ctx.forward_cells_batch(slabs, work, sa, si, w, **with_score)  # noqa: E731
        if what == "adjoint":
            run()
            run = lambda: ctx.adjoint_cells_batch(slabs, init, sa, si, g, ga, gi, history_score=sc)  # noqa: E731
        t[m] = _fastest(run, lambda: [work[f].copy_(v) for f, v in init.items()])
        _say(f"{what} of slabs of {m} thick cells: {1e3 * t[m]:.3f} ms")
    assert t[above] < 3 * t[below]
