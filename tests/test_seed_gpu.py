"""GPU: seeds with bit 63 set.  The generator's state has 63 bits, so a history
draws the same numbers with the bit and without; one that has no event leaves
with its seed as it came, in every kernel, as the oracle's does."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", [40, 10_200])
@pytest.mark.parametrize("how", ["host", "history", "event", "batch", "forward", "forward_batch"])
def test_seeds_of_64_bits(ctx, oracle, how, m):
    import mcgpu
    import torch
    from mcgpu import PARTICLE
    print(f"seeds of 64 bits {how} m={m}", flush=True)
    rng = np.random.default_rng(m)
    n, dx, min_w = 200, 1.0 / m, 5e-2
    bank = np.zeros(n, dtype=PARTICLE)
    bank["seed"] = rng.integers(0, 1 << 64, n, dtype=np.uint64)
    bank["seed"][::2] |= np.uint64(1 << 63)
    bank["index"] = rng.integers(0, m, n)
    bank["x"] = (bank["index"] + rng.random(n)) * dx
    bank["mu"] = rng.uniform(-1, 1, n)
    bank["wmc"] = 1.0
    bank["wmc"][::5] = 1e-2                                  # below the least weight
    bank["index"][::7] = rng.choice([-1, m, m + 50], len(bank[::7]))  # outside
    sigs, ar = np.full(m, 0.1 / dx), rng.uniform(0.3, 0.9, m)
    sa, si = sigs * ar, sigs * (1.0 - ar)
    o = oracle.simulate_bank(64, 0, m, dx, min_w, sigs, ar, bank, nthread=8)
    idle = o["events"] == 0
    assert np.any(idle & (bank["seed"] >> np.uint64(63) == 1)) and not idle.all()
    if how == "host":
        b, w = bank.copy(), np.zeros(m)
        result, _, _ = ctx.simulate(b, sigs, ar, w, 0, m, dx, min_w)
    else:
        d = lambda v: torch.from_numpy(np.ascontiguousarray(v)).cuda()  # noqa: E731
        db, dw, dr = mcgpu.bank_to_device(bank), d(np.zeros(m)), d(np.zeros(n, np.int8))
        slabs = [(0, m, dx, min_w, 0, 0, n)]
        if how == "batch":
            plan = mcgpu.Batch(ctx, slabs, d(sigs), d(ar), dw, db, dr)
            plan.run()
            plan.close()
        elif how == "forward":
            ctx.forward_cells(db, d(sa), d(si), dw, 0, m, dx, min_w, result=dr)
        elif how == "forward_batch":
            ctx.forward_cells_batch(slabs, db, d(sa), d(si), dw, result=dr)
        else:
            ctx.simulate_device(db, d(sigs), d(ar), dw, 0, m, dx, min_w, result=dr,
                                options=mcgpu.make_options(how))
        b, w, result = mcgpu.bank_from_device(db), dw.cpu().numpy(), dr.cpu().numpy()
    for f in ("seed", "x", "mu", "wmc", "index"):
        assert np.array_equal(b[f], o["bank"][f]), f
    assert np.array_equal(result.astype(np.int32), o["result"])
    assert np.array_equal(w, o["tally_exact"])
