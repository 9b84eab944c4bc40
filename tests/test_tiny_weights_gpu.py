"""GPU: particle weights so small that most deposits lie below the tally's
resolution of 2^-88: the oracle's tallies, and no step in time (such terms used
to go to the global tally one after the other)."""
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _bank(m, n, wmc, seed):
    from mcgpu import PARTICLE, configs
    rng = np.random.default_rng(seed)
    bank = np.zeros(n, dtype=PARTICLE)
    bank["seed"] = configs.seed_chain(n)
    bank["mu"] = np.sqrt(rng.random(n))
    bank["wmc"] = wmc * rng.uniform(0.5, 1.0, n)
    return rng.lognormal(0.3, 0.6, m), rng.uniform(0.05, 0.95, m), bank


@pytest.mark.parametrize("log2", [-74, -80, -86, -90])
@pytest.mark.parametrize("how", ["history", "event", "gradient"])
def test_weights_about_the_resolution(ctx, oracle, how, log2):
    import mcgpu
    import torch
    print(f"tiny weights 2^{log2} {how}", flush=True)
    m, n, wmc = 60, 3000, 2.0 ** log2
    sigs, ar, bank = _bank(m, n, wmc, 5)
    dx, min_w = 1.0 / m, 1e-3 * wmc
    d = lambda v: torch.from_numpy(np.ascontiguousarray(v)).cuda()  # noqa: E731
    db, w = mcgpu.bank_to_device(bank), d(np.zeros(m))
    if how == "gradient":
        sa, si, g = sigs * ar, sigs * (1 - ar), np.linspace(-1, 1, m)
        o = oracle.forward_cells(0, m, dx, min_w, sa, si, bank, g=g)
        oa, oi = oracle.adjoint_cells(0, m, dx, min_w, sa, si, bank, g, score=o["score"])
        ga, gi, sc = d(np.zeros(m)), d(np.zeros(m)), d(np.zeros(n))
        init = {k: v.clone() for k, v in db.items()}
        ctx.forward_cells(db, d(sa), d(si), w, 0, m, dx, min_w, g=d(g), history_score=sc)
        ctx.adjoint_cells(init, d(sa), d(si), 0, m, dx, min_w, d(g), ga, gi, history_score=sc)
        assert np.array_equal(ga.cpu().numpy(), oa) and np.array_equal(gi.cpu().numpy(), oi)
    else:
        o = oracle.simulate_bank(64, 0, m, dx, min_w, sigs, ar, bank, nthread=8)
        ctx.simulate_device(db, d(sigs), d(ar), w, 0, m, dx, min_w,
                            options=mcgpu.make_options(how))
    assert np.array_equal(w.cpu().numpy(), o["tally_exact"])
    assert np.array_equal(mcgpu.bank_from_device(db)["wmc"], o["bank"]["wmc"])


def test_no_step_in_time_for_tiny_weights(ctx):
    import mcgpu
    import torch
    m, n, t = 1000, 200_000, {}
    d = lambda v: torch.from_numpy(np.ascontiguousarray(v)).cuda()  # noqa: E731
    for wmc in (1.0, 2.0 ** -80):
        sigs, ar, bank = _bank(m, n, wmc, 6)
        init, ds, da, w = mcgpu.bank_to_device(bank), d(sigs), d(ar), d(np.zeros(m))
        t[wmc] = 1e9
        for _ in range(4):
            work = {k: v.clone() for k, v in init.items()}
            torch.cuda.synchronize()
            t0 = time.perf_counter()
            ctx.simulate_device(work, ds, da, w, 0, m, 1.0 / m, 1e-3 * wmc)
            t[wmc] = min(t[wmc], time.perf_counter() - t0)
        print(f"weights {wmc:g}: {1e3 * t[wmc]:.3f} ms", flush=True)
    assert t[2.0 ** -80] < 4 * t[1.0]
