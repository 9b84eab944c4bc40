"""GPU: weights, cross sections and targets that are infinite, NaN or beyond the
tally's range, through the block tallies of the batches and the gradients:
every cell they do not touch keeps the oracle's bits, those they touch are
infinite or NaN as the oracle's."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
M, N, MIN_W = 60, 800, 1e-3


def _dev(x):
    import torch
    return torch.from_numpy(np.ascontiguousarray(x)).cuda()


def _inputs(seed, thick):
    from mcgpu import PARTICLE, configs
    rng = np.random.default_rng(seed)
    dx = 1.0 / M
    sa, si = thick * rng.lognormal(0, 0.5, M), thick * rng.lognormal(0, 0.5, M)
    bank = np.zeros(N, dtype=PARTICLE)
    bank["seed"] = configs.seed_chain(N)
    bank["index"] = rng.integers(0, M - 20, N)  # the last cells are reached from these
    bank["x"] = (bank["index"] + rng.random(N)) * dx
    bank["mu"] = rng.uniform(-1, 1, N)
    bank["wmc"] = 1.0
    return sa, si, dx, bank


def _plant(what, sa, si, bank, g):
    if what == "inf_weight":
        bank["wmc"][5] = np.inf
    elif what == "nan_weight":
        bank["wmc"][5::100] = np.nan
    elif what == "heavy":
        bank["wmc"][5] = 1e13
    elif what == "nan_absorption":
        sa[7] = np.nan
    elif what == "inf_absorption":
        sa[7] = np.inf
    elif what == "nan_scattering":
        si[7] = np.nan
    elif what == "inf_scattering":
        si[7] = np.inf
    elif what == "nan_target":
        g[30] = np.nan
    elif what == "inf_target":
        g[30], g[31] = np.inf, -np.inf


@pytest.mark.parametrize("thick", [1.0, 60.0])
@pytest.mark.parametrize("what", ["inf_weight", "nan_weight", "heavy", "nan_absorption",
                                  "inf_absorption", "nan_scattering", "inf_scattering"])
def test_batched_transport(ctx, oracle, what, thick):
    import mcgpu
    print(f"batch, {what}, thick {thick}", flush=True)
    cases = [_inputs(1, thick), _inputs(2, thick)]
    _plant(what, cases[0][0], cases[0][1], cases[0][3], None)
    with np.errstate(invalid="ignore"):
        sigs = [c[0] + c[1] for c in cases]
        ar = [c[0] / s for c, s in zip(cases, sigs)]
    db = mcgpu.bank_to_device(np.concatenate([c[3] for c in cases]))
    dw, dr = _dev(np.zeros(2 * M)), _dev(np.zeros(2 * N, np.int8))
    plan = mcgpu.Batch(ctx, [(0, M, 1.0 / M, MIN_W, s * M, s * N, N) for s in range(2)],
                       _dev(np.concatenate(sigs)), _dev(np.concatenate(ar)), dw, db, dr)
    plan.run(allow=(mcgpu.ERR_RANGE,) if what == "heavy" else ())
    plan.close()
    b, w = mcgpu.bank_from_device(db), dw.cpu().numpy()
    for s, (_, _, dx, bank) in enumerate(cases):
        o = oracle.simulate_bank(64, 0, M, dx, MIN_W, sigs[s], ar[s], bank, nthread=8)
        of = slice(s * N, (s + 1) * N)
        for f in ("seed", "x", "mu", "wmc", "index"):
            assert np.array_equal(b[f][of], o["bank"][f], equal_nan=f[0] != "s" and f != "index"), f
        assert np.array_equal(dr.cpu().numpy()[of].astype(np.int32), o["result"])
        assert np.array_equal(w[s * M:(s + 1) * M], o["tally_exact"], equal_nan=True)
        assert s == 1 or what == "nan_weight" or not np.isfinite(o["tally_exact"]).all()


@pytest.mark.parametrize("batched", [False, True])
@pytest.mark.parametrize("what", ["inf_weight", "nan_weight", "nan_absorption", "inf_absorption",
                                  "nan_scattering", "nan_target", "inf_target"])
def test_gradients(ctx, oracle, what, batched):
    """(With infinite sig_i a history collides where it stands, without end.)
    The oracle keeps one word of flags for both gradients of a cell, the
    library one each: where it is set, either may be what is not finite."""
    import mcgpu
    import torch
    print(f"gradient, {what}, batched={batched}", flush=True)
    sa, si, dx, bank = _inputs(3, 1.0)
    g = np.random.default_rng(4).uniform(-1, 1, M)
    _plant(what, sa, si, bank, g)
    o = oracle.forward_cells(0, M, dx, MIN_W, sa, si, bank, g=g)
    oa, oi = oracle.adjoint_cells(0, M, dx, MIN_W, sa, si, bank, g, score=o["score"])
    init = mcgpu.bank_to_device(bank)
    work = {k: v.clone() for k, v in init.items()}
    w, ga, gi = (torch.zeros(M, dtype=torch.float64, device="cuda") for _ in range(3))
    sc = torch.zeros(N, dtype=torch.float64, device="cuda")
    if batched:
        slabs = [(0, M, dx, MIN_W, 0, 0, N)]
        ctx.forward_cells_batch(slabs, work, _dev(sa), _dev(si), w, g=_dev(g), history_score=sc)
        ctx.adjoint_cells_batch(slabs, init, _dev(sa), _dev(si), _dev(g), ga, gi, history_score=sc)
    else:
        ctx.forward_cells(work, _dev(sa), _dev(si), w, 0, M, dx, MIN_W, g=_dev(g), history_score=sc)
        ctx.adjoint_cells(init, _dev(sa), _dev(si), 0, M, dx, MIN_W, _dev(g), ga, gi,
                          history_score=sc)
    w, ga, gi, sc = (t.cpu().numpy() for t in (w, ga, gi, sc))
    assert np.array_equal(sc, o["score"], equal_nan=True)
    assert np.array_equal(w, o["tally_exact"], equal_nan=True)
    plain = np.isfinite(oa) & np.isfinite(oi)
    assert np.array_equal(ga[plain], oa[plain]) and np.array_equal(gi[plain], oi[plain])
    assert not (np.isfinite(ga) & np.isfinite(gi))[~plain].any()
    assert not plain.all() or what in ("nan_weight", "inf_absorption", "nan_scattering")
