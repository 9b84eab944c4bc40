"""GPU: batches of slabs whose cells are thick, where every event is a general
one (half the cells and one more, exactly half, all of them; strongly absorbing,
strongly scattering): bit-identical to the oracle, also where the event cap binds."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _slab(m, n, thick, kind, seed):
    from mcgpu import PARTICLE, configs
    rng = np.random.default_rng(seed)
    dx = 1.0 / m
    sa, si = rng.uniform(0.01, 0.1, m) / dx, rng.uniform(0.01, 0.1, m) / dx
    k = rng.permutation(m)[:thick]
    if kind != "scattering":
        sa[k] = rng.uniform(0.6, 40.0, thick) / dx
    if kind != "absorbing":
        si[k] = rng.uniform(0.6, 40.0, thick) / dx
    si[::9] = 5e-5  # no flight is sampled there
    bank = np.zeros(n, dtype=PARTICLE)
    bank["seed"] = configs.seed_chain(n)
    bank["index"] = rng.integers(-1, m + 1, n)
    bank["x"] = (bank["index"] + rng.random(n)) * dx
    bank["mu"] = rng.uniform(-1, 1, n)
    bank["mu"][::13] = rng.choice([0.0, 1e-4, -1e-5], len(bank[::13]))
    bank["wmc"] = rng.uniform(0.2, 1.0, n)
    return sa, si, dx, bank


CASES = [(32, 400, 17, "both"), (32, 400, 16, "both"), (40, 300, 40, "absorbing"),
         (64, 700, 64, "scattering"), (300, 900, 200, "both"), (1, 130, 1, "both"),
         (1500, 300, 1500, "both")]


def _dev(x):
    import torch
    return torch.from_numpy(np.ascontiguousarray(x)).cuda()


@pytest.mark.parametrize("cap,refill", [(0, 0), (0, 1), (3, 0)])
def test_batches_of_thick_slabs(ctx, oracle, cap, refill):
    import mcgpu
    print(f"thick slabs, cap {cap} refill {refill}", flush=True)
    parts = [_slab(*c, seed=7 + i) for i, c in enumerate(CASES)]
    cells = np.concatenate([[0], np.cumsum([c[0] for c in CASES])])
    first = np.concatenate([[0], np.cumsum([c[1] for c in CASES])])
    min_w = 1e-3
    slabs = [(0, c[0], p[2], min_w, int(cells[s]), int(first[s]), c[1])
             for s, (c, p) in enumerate(zip(CASES, parts))]
    sigs = np.concatenate([p[0] + p[1] for p in parts])
    ar = np.concatenate([p[0] / (p[0] + p[1]) for p in parts])
    db = mcgpu.bank_to_device(np.concatenate([p[3] for p in parts]))
    dw, dr = _dev(np.zeros(int(cells[-1]))), _dev(np.zeros(int(first[-1]), np.int8))
    plan = mcgpu.Batch(ctx, slabs, _dev(sigs), _dev(ar), dw, db, dr,
                       options=mcgpu.make_options(grid_blocks=3, block_size=128,
                                                  events_per_refill=refill,
                                                  max_events_per_history=cap))
    plan.run(allow=(mcgpu.ERR_EVENT_CAP,))
    plan.close()
    b, w, r = mcgpu.bank_from_device(db), dw.cpu().numpy(), dr.cpu().numpy()
    for s, (c, p) in enumerate(zip(CASES, parts)):
        cut, of = slice(cells[s], cells[s + 1]), slice(first[s], first[s + 1])
        o = oracle.simulate_bank(64, 0, c[0], p[2], min_w, sigs[cut], ar[cut], p[3], nthread=8)
        same = o["events"] <= cap if cap else np.ones(c[1], bool)
        assert cap == 0 or np.all(r[of][~same] == 2)
        for f in ("seed", "x", "mu", "wmc", "index"):
            assert np.array_equal(b[f][of][same], o["bank"][f][same], equal_nan=f == "x"), (c, f)
        assert np.array_equal(r[of][same].astype(np.int32), o["result"][same]), c
        if cap == 0:
            assert np.array_equal(w[cut], o["tally_exact"]), c


@pytest.mark.parametrize("score", [True, False])
def test_gradients_of_thick_slabs(ctx, oracle, score):
    import mcgpu
    import torch
    print(f"thick slabs, gradient, score={score}", flush=True)
    parts = [_slab(*c, seed=70 + i) for i, c in enumerate(CASES)]
    cells = np.concatenate([[0], np.cumsum([c[0] for c in CASES])])
    first = np.concatenate([[0], np.cumsum([c[1] for c in CASES])])
    min_w = 1e-3
    slabs = [(0, c[0], p[2], min_w, int(cells[s]), int(first[s]), c[1])
             for s, (c, p) in enumerate(zip(CASES, parts))]
    sa, si = (_dev(np.concatenate([p[k] for p in parts])) for k in (0, 1))
    g = np.random.default_rng(3).uniform(-1, 1, int(cells[-1]))
    init = mcgpu.bank_to_device(np.concatenate([p[3] for p in parts]))
    work = {k: v.clone() for k, v in init.items()}
    w, ga, gi = (torch.zeros(int(cells[-1]), dtype=torch.float64, device="cuda") for _ in range(3))
    sc = torch.zeros(int(first[-1]), dtype=torch.float64, device="cuda")
    opt = mcgpu.make_options(grid_blocks=3, block_size=128)
    ctx.forward_cells_batch(slabs, work, sa, si, w, g=_dev(g) if score else None,
                            history_score=sc if score else None, options=opt)
    ctx.adjoint_cells_batch(slabs, init, sa, si, _dev(g), ga, gi,
                            history_score=sc if score else None, options=opt)
    for s, (c, p) in enumerate(zip(CASES, parts)):
        cut, of = slice(cells[s], cells[s + 1]), slice(first[s], first[s + 1])
        o = oracle.forward_cells(0, c[0], p[2], min_w, p[0], p[1], p[3], g=g[cut])
        oa, oi = oracle.adjoint_cells(0, c[0], p[2], min_w, p[0], p[1], p[3], g[cut],
                                      score=o["score"] if score else None)
        assert np.array_equal(w[cut].cpu().numpy(), o["tally_exact"]), c
        assert not score or np.array_equal(sc[of].cpu().numpy(), o["score"]), c
        assert np.array_equal(ga[cut].cpu().numpy(), oa), c
        assert np.array_equal(gi[cut].cpu().numpy(), oi), c
