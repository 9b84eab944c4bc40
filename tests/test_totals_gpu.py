"""GPU: a call's totals (events, collisions, ends) are those of its histories, on
grids of one block to a full chip and in repeated calls; and the ends of a full
grid's blocks do not wait for each other."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _case(m, n, mult, seed=11):
    from mcgpu import PARTICLE, configs
    rng = np.random.default_rng(seed)
    dx = 1.0 / m
    sa, si = (np.exp(0.5 * rng.standard_normal(m)) * mult for _ in range(2))
    bank = np.zeros(n, dtype=PARTICLE)
    bank["seed"] = configs.seed_chain(n)
    bank["index"] = rng.integers(0, m, n)
    bank["x"] = (bank["index"] + rng.random(n)) * dx
    bank["mu"] = rng.uniform(-1, 1, n)
    bank["wmc"] = 1.0
    return sa, si, dx, bank


def _dev(x):
    import torch
    return torch.from_numpy(np.ascontiguousarray(x)).cuda()


def _ends(result):
    return [int(np.count_nonzero(result == c)) for c in (-1, 1, 0)]


@pytest.mark.parametrize("kernel", ["history", "event"])
@pytest.mark.parametrize("m,n", [(1, 3000), (40, 5000), (11_000, 600)])
@pytest.mark.parametrize("grid", [0, 1, 9])
def test_totals_of_a_call(ctx, oracle, kernel, m, n, grid):
    import mcgpu
    print(f"totals {kernel} m={m} n={n} grid={grid}", flush=True)
    sa, si, dx, bank = _case(m, n, 3.0)
    o = oracle.simulate_bank(64, 0, m, dx, 1e-2, sa + si, sa / (sa + si), bank, nthread=8)
    opt = mcgpu.make_options(kernel, grid_blocks=grid)
    for _ in range(2):
        st, _ = ctx.simulate_device(mcgpu.bank_to_device(bank), _dev(sa + si), _dev(sa / (sa + si)),
                                    _dev(np.zeros(m)), 0, m, dx, 1e-2, options=opt)
        assert st["events"] == o["events"].sum()
        assert [st["n_left"], st["n_right"], st["n_killed"]] == _ends(o["result"])
        assert 0 < st["collisions"] < st["events"]
    if kernel == "history":
        col = _dev(np.zeros(n, np.int64))
        ev = _dev(np.zeros(n, np.int64))
        st, _ = ctx.simulate_device(mcgpu.bank_to_device(bank), _dev(sa + si), _dev(sa / (sa + si)),
                                    _dev(np.zeros(m)), 0, m, dx, 1e-2, events=ev, collisions=col,
                                    options=opt)
        assert st["collisions"] == int(col.sum()) and st["events"] == int(ev.sum())


def test_totals_of_batches_and_gradients(ctx, oracle):
    import mcgpu
    import torch
    m, n, S = 30, 700, 12
    parts = [_case(m, n, 3.0, seed=s) for s in range(S)]
    dx, min_w = 1.0 / m, 1e-2
    slabs = [(0, m, dx, min_w, s * m, s * n, n) for s in range(S)]
    sa, si = (np.concatenate([p[k] for p in parts]) for k in (0, 1))
    bank = np.concatenate([p[3] for p in parts])
    o = [oracle.simulate_bank(64, 0, m, dx, min_w, p[0] + p[1], p[0] / (p[0] + p[1]), p[3],
                              nthread=8) for p in parts]
    events = sum(int(q["events"].sum()) for q in o)
    ends = list(np.sum([_ends(q["result"]) for q in o], axis=0))
    w, ga, gi = (torch.zeros(S * m, dtype=torch.float64, device="cuda") for _ in range(3))
    work = mcgpu.bank_to_device(bank)
    plan = mcgpu.Batch(ctx, slabs, _dev(sa + si), _dev(sa / (sa + si)), w, work)
    fresh = mcgpu.bank_to_device(bank)
    for _ in range(3):
        for k, v in fresh.items():
            work[k].copy_(v)
        torch.cuda.synchronize()
        st = plan.run()
        st = st[0] if isinstance(st, tuple) else st
        assert st["events"] == events
        assert [st["n_left"], st["n_right"], st["n_killed"]] == ends
    plan.close()
    e1 = o[0]["events"].sum()
    for _ in range(2):
        for k, v in fresh.items():
            work[k].copy_(v)
        st = ctx.forward_cells_batch(slabs, work, _dev(sa), _dev(si), w)
        assert st["events"] > 0.99 * events
        st = ctx.adjoint_cells_batch(slabs, fresh, _dev(sa), _dev(si), _dev(np.ones(S * m)), ga, gi)
        assert st["events"] > 0.99 * events
        one = mcgpu.bank_to_device(parts[0][3])
        args = _dev(parts[0][0]), _dev(parts[0][1])
        st = ctx.adjoint_cells(one, *args, 0, m, dx, min_w, _dev(np.ones(m)), ga[:m], gi[:m])
        assert st["events"] > 0.99 * e1
        st = ctx.forward_cells(one, *args, w[:m], 0, m, dx, min_w)
        assert st["events"] > 0.99 * e1


def test_blocks_do_not_wait_at_their_ends(ctx):
    """20,000 histories of a dozen events, on 256 blocks and on a full grid of
    1,024: with all totals in one line the adds of 768 more blocks took 46 us."""
    import mcgpu
    sa, si, dx, bank = _case(10, 20_000, 5.0)
    init = mcgpu.bank_to_device(bank)
    work = {k: v.clone() for k, v in init.items()}
    sigs, ar, w = _dev(sa + si), _dev(sa / (sa + si)), _dev(np.zeros(10))

    def kernel_ms(grid):
        import torch
        t = []
        for _ in range(40):
            for k, v in init.items():
                work[k].copy_(v)
            torch.cuda.synchronize()
            t.append(ctx.simulate_device(work, sigs, ar, w, 0, 10, dx, 1e-3,
                                         options=mcgpu.make_options(grid_blocks=grid))[0]["kernel_ms"])
        return sorted(t)[10]
    few, full = kernel_ms(256), kernel_ms(0)
    print(f"256 blocks {1e3 * few:.1f} us, a full grid {1e3 * full:.1f} us", flush=True)
    assert full - few < 0.032


def test_blocks_of_few_cells(ctx):
    """Gradients of 1,000 histories of one event on one cell, with the blocks that
    the call takes and on 256: on a full grid they take 2.3 times as long."""
    import mcgpu
    import torch
    sa, si, dx, bank = _case(1, 1000, 0.1)
    init, g = mcgpu.bank_to_device(bank), _dev(np.ones(1))
    ga, gi = (torch.zeros(1, dtype=torch.float64, device="cuda") for _ in range(2))

    def kernel_ms(grid):
        t = [ctx.adjoint_cells(init, _dev(sa), _dev(si), 0, 1, dx, 1e-3, g, ga, gi,
                               options=mcgpu.make_options(grid_blocks=grid))["kernel_ms"]
             for _ in range(40)]
        return sorted(t)[10]
    few, own = kernel_ms(256), kernel_ms(0)
    print(f"256 blocks {1e3 * few:.1f} us, by itself {1e3 * own:.1f} us", flush=True)
    assert own < 1.4 * few


@pytest.mark.parametrize("m,n", [(8, 65_536), (8, 65_537), (9, 65_536), (1, 255)])
def test_around_the_limits_of_few_cells(ctx, oracle, m, n):
    import mcgpu
    print(f"few cells m={m} n={n}", flush=True)
    sa, si, dx, bank = _case(m, n, 2.0)
    o = oracle.simulate_bank(64, 0, m, dx, 1e-2, sa + si, sa / (sa + si), bank, nthread=8)
    db, dw = mcgpu.bank_to_device(bank), _dev(np.zeros(m))
    st, _ = ctx.simulate_device(db, _dev(sa + si), _dev(sa / (sa + si)), dw, 0, m, dx, 1e-2)
    assert st["events"] == o["events"].sum()
    assert np.array_equal(dw.cpu().numpy(), o["tally_exact"])
    b = mcgpu.bank_from_device(db)
    for f in ("seed", "x", "mu", "wmc", "index"):
        assert np.array_equal(b[f], o["bank"][f]), f
