"""GPU: single layers whose cells are thick, where every event is a general one
(half the cells and one more, exactly half, all of them; strongly absorbing,
strongly scattering; cells in LDS, through L2 and in windows): bit-identical to
the oracle, also where the event cap binds, and as fast as the same slab in a
batch."""
import time

import numpy as np
import pytest

from test_thick_slabs_gpu import _dev, _slab

pytestmark = pytest.mark.gpu

# the last ones: cells beside the tally no longer in LDS; two windows
CASES = [(1, 130, 1, "both"), (32, 400, 17, "both"), (32, 400, 16, "both"),
         (40, 300, 40, "absorbing"), (64, 1500, 64, "scattering"), (300, 900, 200, "both"),
         (1500, 700, 1500, "both"), (7000, 500, 7000, "both"), (11_000, 500, 11_000, "both")]


def _say(*a):
    print(*a, flush=True)


@pytest.mark.parametrize("m,n,thick,kind", CASES)
@pytest.mark.parametrize("cap,refill,wmc", [(0, 0, 1.0), (0, 1, 1.0), (3, 0, 1.0), (0, 0, 64.0)])
def test_layers_of_thick_cells(ctx, oracle, m, n, thick, kind, cap, refill, wmc):
    import mcgpu
    _say(f"thick layer m={m} {thick} {kind} cap {cap} refill {refill} weights {wmc}")
    sa, si, dx, bank = _slab(m, n, thick, kind, seed=m + thick)
    bank["wmc"] *= wmc
    min_w, sigs, ar = 1e-3 * wmc, sa + si, sa / (sa + si)
    o = oracle.simulate_bank(64, 0, m, dx, min_w, sigs, ar, bank, nthread=8)
    opt = mcgpu.make_options(grid_blocks=3, block_size=128, events_per_refill=refill,
                             max_events_per_history=cap)
    db, dw, dr = mcgpu.bank_to_device(bank), _dev(np.zeros(m)), _dev(np.zeros(n, np.int8))
    ctx.simulate_device(db, _dev(sigs), _dev(ar), dw, 0, m, dx, min_w, result=dr, options=opt,
                        allow=(mcgpu.ERR_EVENT_CAP,))
    b, r = mcgpu.bank_from_device(db), dr.cpu().numpy().astype(np.int32)
    same = o["events"] <= cap if cap else np.ones(n, bool)
    assert np.all(r[~same] == 2)
    for f in ("seed", "x", "mu", "wmc", "index"):
        assert np.array_equal(b[f][same], o["bank"][f][same], equal_nan=f == "x"), f
    assert np.array_equal(r[same], o["result"][same])
    if cap == 0:
        assert np.array_equal(dw.cpu().numpy(), o["tally_exact"])


@pytest.mark.parametrize("m,n,thick,kind", CASES)
@pytest.mark.parametrize("score", [True, False])
def test_gradients_of_thick_layers(ctx, oracle, m, n, thick, kind, score):
    import mcgpu
    import torch
    _say(f"thick layer, gradient, m={m} {thick} {kind} score={score}")
    sa, si, dx, bank = _slab(m, n, thick, kind, seed=3 * m + thick)
    min_w, g = 1e-3, np.random.default_rng(3).uniform(-1, 1, m)
    o = oracle.forward_cells(0, m, dx, min_w, sa, si, bank, g=g)
    oa, oi = oracle.adjoint_cells(0, m, dx, min_w, sa, si, bank, g,
                                  score=o["score"] if score else None)
    init = mcgpu.bank_to_device(bank)
    work = {k: v.clone() for k, v in init.items()}
    w, ga, gi = (torch.zeros(m, dtype=torch.float64, device="cuda") for _ in range(3))
    sc = torch.zeros(n, dtype=torch.float64, device="cuda")
    opt = mcgpu.make_options(grid_blocks=3, block_size=128)
    ctx.forward_cells(work, _dev(sa), _dev(si), w, 0, m, dx, min_w, g=_dev(g) if score else None,
                      history_score=sc if score else None, options=opt)
    ctx.adjoint_cells(init, _dev(sa), _dev(si), 0, m, dx, min_w, _dev(g), ga, gi,
                      history_score=sc if score else None, options=opt)
    assert np.array_equal(w.cpu().numpy(), o["tally_exact"])
    assert not score or np.array_equal(sc.cpu().numpy(), o["score"])
    assert np.array_equal(ga.cpu().numpy(), oa)
    assert np.array_equal(gi.cpu().numpy(), oi)


@pytest.mark.parametrize("thick", [10_000, 5001, 5000, 0])
@pytest.mark.parametrize("cap,score", [(0, False), (0, True), (3, False)])
def test_long_runs_of_thick_cells(ctx, oracle, thick, cap, score):
    """10,000 cells fit LDS without the cross sections; long runs (here on two
    blocks) go in two windows, those of thick cells in one."""
    import mcgpu
    m, n, min_w = 10_000, 9000, 0.05
    _say(f"long run, {thick} of {m} cells thick, cap {cap} score {score}")
    sa, si, dx, bank = _slab(m, n, thick, "both", seed=thick)
    o = oracle.forward_cells(0, m, dx, min_w, sa, si, bank, g=np.linspace(-1, 1, m))
    opt = mcgpu.make_options(grid_blocks=2, max_events_per_history=cap)
    for _ in range(2):
        db, dw, dr = mcgpu.bank_to_device(bank), _dev(np.zeros(m)), _dev(np.zeros(n, np.int8))
        if score:
            sc = _dev(np.zeros(n))
            st = ctx.forward_cells(db, _dev(sa), _dev(si), dw, 0, m, dx, min_w,
                                   g=_dev(np.linspace(-1, 1, m)), history_score=sc, result=dr,
                                   options=opt)
            assert np.array_equal(sc.cpu().numpy(), o["score"])
            assert np.array_equal(dw.cpu().numpy(), o["tally_exact"])
            continue
        sigs, ar = sa + si, sa / (sa + si)
        q = oracle.simulate_bank(64, 0, m, dx, min_w, sigs, ar, bank, nthread=8)
        ev, col = _dev(np.zeros(n, np.int64)), _dev(np.zeros(n, np.int64))
        st, _ = ctx.simulate_device(db, _dev(sigs), _dev(ar), dw, 0, m, dx, min_w, result=dr,
                                    events=ev, collisions=col, options=opt,
                                    allow=(mcgpu.ERR_EVENT_CAP,))
        same = q["events"] <= cap if cap else np.ones(n, bool)
        b, r = mcgpu.bank_from_device(db), dr.cpu().numpy().astype(np.int32)
        assert np.all(r[~same] == 2) and np.array_equal(r[same], q["result"][same])
        for f in ("seed", "x", "mu", "wmc", "index"):
            assert np.array_equal(b[f][same], q["bank"][f][same], equal_nan=f == "x"), f
        assert np.array_equal(ev.cpu().numpy()[same], q["events"][same].astype(np.int64))
        assert st["events"] == int(ev.sum()) and st["collisions"] == int(col.sum())
        if cap == 0:
            assert np.array_equal(dw.cpu().numpy(), q["tally_exact"])


def test_a_thick_layer_is_as_fast_as_a_thick_slab(ctx):
    """One history of some 2,300 collisions, by itself and as a batch of one slab:
    with the common step before every general event a layer takes half as long
    again."""
    import mcgpu
    import torch
    m = 100
    sa, si = _dev(np.full(m, 300.0)), _dev(np.full(m, 1e5))
    sigs, ar = sa + si, sa / (sa + si)
    bank = np.zeros(1, dtype=mcgpu.PARTICLE)
    bank["seed"], bank["index"], bank["x"], bank["mu"], bank["wmc"] = 5127801, 50, 0.505, 0.5, 1.0
    init = mcgpu.bank_to_device(bank)
    work = {k: v.clone() for k, v in init.items()}
    w = torch.zeros(m, dtype=torch.float64, device="cuda")
    plan = mcgpu.Batch(ctx, [(0, m, 1.0 / m, 1e-3, 0, 0, 1)], sigs, ar, w, work)

    def best(run):
        t = []
        for _ in range(12):
            for k, v in init.items():
                work[k].copy_(v)
            torch.cuda.synchronize()
            t0 = time.perf_counter()
            run()
            torch.cuda.synchronize()
            t.append(time.perf_counter() - t0)
        return min(t)
    slab = best(plan.run)
    layer = best(lambda: ctx.simulate_device(work, sigs, ar, w, 0, m, 1.0 / m, 1e-3))
    plan.close()
    _say(f"a thick layer {1e3 * layer:.3f} ms, a slab {1e3 * slab:.3f} ms")
    assert layer < 1.25 * slab
