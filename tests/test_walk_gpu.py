"""GPU: the history kernel's block tally and work queue at their edges, every
history and the exact tally bit-identical to the oracle: particle weights of
every scale (which set the two-limb tally's split, or choose the tally with
carry), weights that differ from the block's first histories by twelve orders
of magnitude, and history counts around the sizes at which the queue deals
them out differently."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _say(msg):
    print(msg, flush=True)


def _case(m, n, seed, wmc):
    from mcgpu import PARTICLE, configs
    rng = np.random.default_rng(seed)
    sigs, ar = rng.lognormal(0.3, 0.6, m), rng.uniform(0.05, 0.95, m)
    bank = np.zeros(n, dtype=PARTICLE)
    bank["seed"] = configs.seed_chain(n)
    bank["index"] = rng.integers(0, m, n)
    bank["x"] = (bank["index"] + rng.random(n)) / m
    bank["mu"] = rng.uniform(-1, 1, n)
    bank["wmc"] = wmc
    return sigs, ar, 1.0 / m, bank


def _check(ctx, oracle, m, n, seed, wmc, min_w, kernel="history", **opts):
    import mcgpu
    sigs, ar, dx, bank = _case(m, n, seed, wmc)
    o = oracle.simulate_bank(64, 0, m, dx, min_w, sigs, ar, bank, nthread=8)
    b, w = bank.copy(), np.zeros(m)
    result, st, rc = ctx.simulate(b, sigs, ar, w, 0, m, dx, min_w,
                                  options=mcgpu.make_options(kernel, **opts))
    assert rc == 0
    for f in ("seed", "x", "mu", "wmc", "index"):
        assert np.array_equal(b[f], o["bank"][f]), f
    assert np.array_equal(result, o["result"])
    assert st["events"] == int(o["events"].sum())
    assert np.array_equal(w, o["tally_exact"])


@pytest.mark.parametrize("m", [40, 1500, 4200])
@pytest.mark.parametrize("scale", [1e-14, 1e-8, 1e-3, 1.0, 3.9, 5.0, 1e3, 1e9])
def test_weights_of_every_scale(ctx, oracle, m, scale):
    _say(f"weights {scale} m={m}")
    rng = np.random.default_rng(m)
    _check(ctx, oracle, m, 700, m, scale * rng.uniform(0.5, 1.0, 700), 1e-3 * scale)


@pytest.mark.parametrize("first", [1e-9, 1.0, 1e6])
def test_later_weights_unlike_the_first(ctx, oracle, first):
    """The first histories of every wave weigh `first`; the others anything
    from 1e-7 to 1e5, so that many deposits lie outside the block's split."""
    _say(f"first weights {first}")
    rng = np.random.default_rng(5)
    n = 9000
    wmc = 10.0 ** rng.uniform(-7, 5, n)
    wmc[:2048] = first
    _check(ctx, oracle, 60, n, 6, wmc, 1e-10, grid_blocks=2, block_size=256)


@pytest.mark.parametrize("events_per_refill", [0, 1, 5000])
@pytest.mark.parametrize("n", [1, 2, 255, 256, 257, 2047, 2049, 4100])
def test_history_counts_around_the_queue_sizes(ctx, oracle, n, events_per_refill):
    _say(f"n={n} events_per_refill={events_per_refill}")
    _check(ctx, oracle, 30, n, n, 1.0, 1e-2, events_per_refill=events_per_refill)


@pytest.mark.parametrize("n", [3000, 70_000])
def test_runs_from_the_counter(ctx, oracle, n):
    """More histories than the first runs hold: few blocks, many later runs."""
    _say(f"n={n}, later runs")
    _check(ctx, oracle, 25, n, n, 1.0, 1e-2, grid_blocks=3, block_size=64)


@pytest.mark.parametrize("compaction_interval", [1, 3, 64])
@pytest.mark.parametrize("scale", [1e-8, 1.0, 1e3])
@pytest.mark.parametrize("n", [50, 700, 5000])
def test_event_kernel_passes_then_drain(ctx, oracle, n, scale, compaction_interval):
    """Two waves of 256 pool slots each: banks that never leave the drain, that
    just fill the pools, and that pass through them many times, with on-edge
    and dead slots at the switch and every form of tally."""
    _say(f"event n={n} weights {scale} ci={compaction_interval}")
    rng = np.random.default_rng(n)
    _check(ctx, oracle, 45, n, n, scale * rng.uniform(0.5, 1.0, n), 1e-2 * scale, kernel="event",
           grid_blocks=1, block_size=128, particles_per_lane=4,
           compaction_interval=compaction_interval)


def _gradient(ctx, oracle, m, n, seed, wscale, gscale, with_score, batched):
    """Forward with scores and adjoint against the oracle, one slab (or the
    slab twice in a batch): scores, tally and both gradients, bit for bit."""
    import mcgpu
    import torch
    rng = np.random.default_rng(seed)
    sa, ss = rng.lognormal(0, 0.5, m), rng.lognormal(0, 0.5, m)
    ss[::7] = 5e-5  # not sampled there: no sig_i term
    _, _, dx, bank = _case(m, n, seed, wscale * rng.uniform(0.5, 1.0, n))
    g = gscale * rng.uniform(-1, 1, m) * (rng.random(m) < 0.3)
    dev = lambda x: torch.from_numpy(np.ascontiguousarray(x)).cuda()  # noqa: E731
    zeros = lambda k: torch.zeros(k, dtype=torch.float64, device="cuda")  # noqa: E731
    min_w = 1e-3 * wscale
    o = oracle.forward_cells(0, m, dx, min_w, sa, ss, bank, g=g)
    oa, oi = oracle.adjoint_cells(0, m, dx, min_w, sa, ss, bank, g,
                                  score=o["score"] if with_score else None)
    k = 2 if batched else 1
    rep = lambda x: dev(np.tile(x, k))  # noqa: E731
    init = mcgpu.bank_to_device(np.tile(bank, k))
    work = {f: v.clone() for f, v in init.items()}
    w, ga, gi = zeros(k * m), zeros(k * m), zeros(k * m)
    score = torch.empty(k * n, dtype=torch.float64, device="cuda")
    if batched:
        slabs = [(0, m, dx, min_w, s * m, s * n, n) for s in range(k)]
        ctx.forward_cells_batch(slabs, work, rep(sa), rep(ss), w, g=rep(g), history_score=score)
        ctx.adjoint_cells_batch(slabs, init, rep(sa), rep(ss), rep(g), ga, gi,
                                history_score=score if with_score else None)
    else:
        ctx.forward_cells(work, dev(sa), dev(ss), w, 0, m, dx, min_w, g=dev(g),
                          history_score=score)
        ctx.adjoint_cells(init, dev(sa), dev(ss), 0, m, dx, min_w, dev(g), ga, gi,
                          history_score=score if with_score else None)
    same = lambda t, x: np.array_equal(t.cpu().numpy().view(np.uint64),  # noqa: E731
                                       np.tile(x, k).view(np.uint64))
    assert same(score, o["score"])
    assert same(w, o["tally_exact"])
    assert same(ga, oa) and same(gi, oi)
    assert oa.any() and oi.any()


@pytest.mark.parametrize("batched", [False, True])
@pytest.mark.parametrize("wscale,gscale", [(1.0, 1e-9), (1.0, 20.0), (1.0, 1e4), (1e-8, 1.0),
                                           (1e3, 1.0)])
def test_gradient_terms_of_every_scale(ctx, oracle, wscale, gscale, batched):
    _say(f"gradient, weights {wscale} targets {gscale} batched={batched}")
    _gradient(ctx, oracle, 90, 500, 3, wscale, gscale, True, batched)


@pytest.mark.parametrize("with_score", [True, False])
@pytest.mark.parametrize("m,batched", [(2890, False), (2900, False), (5100, False), (2880, True),
                                       (4100, True)])
def test_gradient_layers_around_the_lds_limits(ctx, oracle, m, batched, with_score):
    """Cells, targets and tallies in LDS (56 B a cell); the tallies alone
    (32 B, one slab); neither."""
    _say(f"gradient, m={m} batched={batched} with_score={with_score}")
    _gradient(ctx, oracle, m, 120, m, 1.0, 1.0, with_score, batched)


@pytest.mark.parametrize("m,n,opts", [(10_136, 900, {}), (20_500, 400, {}), (20_500, 3000, {}),
                                      (31_000, 64, {"grid_blocks": 5, "block_size": 128}),
                                      (31_000, 64, {"grid_blocks": 2})])
@pytest.mark.parametrize("host", [True, False])
def test_wide_layers_in_windows(ctx, oracle, m, n, opts, host):
    """Layers of more cells than a block's LDS tally holds: two windows just
    above the limit, three and four of them, and too few blocks for them (the
    global tally).  Histories cross the windows' edges both ways; counts add up
    over the sweeps."""
    import mcgpu
    import torch
    _say(f"windows m={m} n={n} {opts} host={host}")
    sigs, ar, dx, bank = _case(m, n, m + n, 1.0)
    sigs *= 3.0
    lo = 700
    bank["index"] += lo
    bank["x"] = (bank["index"] + 0.25) * dx
    min_w = 1e-2
    bank["wmc"][::50] = 1e-3  # finished as they come
    o = oracle.simulate_bank(64, lo, m, dx, min_w, sigs, ar, bank, nthread=8)
    options = mcgpu.make_options("history", **opts)
    if host:
        b, w = bank.copy(), np.zeros(m)
        result, st, rc = ctx.simulate(b, sigs, ar, w, lo, lo + m, dx, min_w, options=options)
    else:
        db = mcgpu.bank_to_device(bank)
        dev = lambda x: torch.from_numpy(np.ascontiguousarray(x)).cuda()  # noqa: E731
        dw, dr = dev(np.zeros(m)), dev(np.zeros(n, np.int8))
        ev, co = dev(np.zeros(n, np.int64)), dev(np.full(n, 5))
        st, rc = ctx.simulate_device(db, dev(sigs), dev(ar), dw, lo, lo + m, dx, min_w, result=dr,
                                     events=ev, collisions=co, options=options)
        b, w, result = mcgpu.bank_from_device(db), dw.cpu().numpy(), dr.cpu().numpy()
        assert np.array_equal(ev.cpu().numpy(), o["events"])
        assert np.array_equal(co.cpu().numpy(), o["collisions"])
    for f in ("seed", "x", "mu", "wmc", "index"):
        assert np.array_equal(b[f], o["bank"][f]), f
    assert np.array_equal(result.astype(np.int32), o["result"])
    assert st["events"] == int(o["events"].sum())
    assert st["collisions"] == int(o["collisions"].sum())
    assert st["n_left"] + st["n_right"] + st["n_killed"] == n
    assert np.array_equal(w, o["tally_exact"])


def test_wide_layer_event_cap_counts_over_sweeps(ctx, oracle):
    """A cap that histories reach after several sweeps ends them at exactly
    that count; shorter ones are the oracle's."""
    import mcgpu
    import torch
    m, n, cap = 10_400, 300, 9000
    sigs, ar, dx, bank = _case(m, n, 9, 1.0)
    _say("windows, event cap")
    o = oracle.simulate_bank(64, 0, m, dx, 1e-3, sigs, ar, bank, nthread=8)
    db = mcgpu.bank_to_device(bank)
    dev = lambda x: torch.from_numpy(np.ascontiguousarray(x)).cuda()  # noqa: E731
    dr, ev = dev(np.zeros(n, np.int8)), dev(np.zeros(n, np.int64))
    st, rc = ctx.simulate_device(db, dev(sigs), dev(ar), dev(np.zeros(m)), 0, m, dx, 1e-3,
                                 result=dr, events=ev, allow=(mcgpu.ERR_EVENT_CAP,),
                                 options=mcgpu.make_options("history", max_events_per_history=cap))
    longer = o["events"] > cap
    assert longer.any() and not longer.all() and rc == mcgpu.ERR_EVENT_CAP
    e, r, b = ev.cpu().numpy(), dr.cpu().numpy(), mcgpu.bank_from_device(db)
    assert np.all(e[longer] == cap) and np.all(r[longer] == 2)
    assert np.array_equal(e[~longer], o["events"][~longer])
    assert np.array_equal(r[~longer], o["result"][~longer])
    for f in ("seed", "x", "mu", "wmc", "index"):
        assert np.array_equal(b[f][~longer], o["bank"][f][~longer]), f
    assert st["events"] == int(np.minimum(o["events"], cap).sum())


def test_wide_layer_scores(ctx, oracle):
    """forward_cells with per-history scores over windows: the same sums in
    event order."""
    import mcgpu
    import torch
    m, n = 12_000, 200
    rng = np.random.default_rng(8)
    sa, ss, g = rng.lognormal(0, 0.5, m), rng.lognormal(0, 0.5, m), rng.uniform(-1, 1, m)
    _, _, dx, bank = _case(m, n, 8, 1.0)
    _say("windows, scores")
    o = oracle.forward_cells(0, m, dx, 1e-3, sa, ss, bank, g=g)
    db = mcgpu.bank_to_device(bank)
    dev = lambda x: torch.from_numpy(np.ascontiguousarray(x)).cuda()  # noqa: E731
    w, sc = dev(np.zeros(m)), dev(np.full(n, 7.0))
    ctx.forward_cells(db, dev(sa), dev(ss), w, 0, m, dx, 1e-3, g=dev(g), history_score=sc)
    assert np.array_equal(w.cpu().numpy(), o["tally_exact"])
    assert np.array_equal(sc.cpu().numpy().view(np.uint64), o["score"].view(np.uint64))


@pytest.mark.parametrize("kernel", ["history", "event"])
@pytest.mark.parametrize("dx", [1e-190, 1e-3, 1.0, 1e190])
def test_particles_at_the_bounds_of_the_common_step(ctx, oracle, dx, kernel):
    """Directions from grazing to far above 1, positions of 0, tiny, on and
    beyond an edge, and cell widths for which the common step is not used."""
    import mcgpu
    _say(f"bounds of the common step dx={dx} {kernel}")
    m = 24
    sigs, ar, _, bank = _case(m, 2000, 61, 1.0)
    sigs = sigs * 0.2 / dx
    rng = np.random.default_rng(62)
    bank["x"] = (bank["index"] + rng.random(2000)) * dx
    edge = rng.integers(0, 2000, 500)
    bank["x"][edge] = (bank["index"][edge] + rng.integers(0, 2, 500)) * dx
    bank["x"][::97] += 0.5 * dx
    first = bank["index"] == 0
    bank["x"][first] = rng.choice([0.0, 5e-324, 2.0 ** -701, 2.0 ** -700, 1e-150], first.sum()) * dx
    eps = 1e-4
    mus = np.array([0.0, eps, np.nextafter(eps, 1), 1e-9, 1.0, 3.0, 2.0 ** 64, 2.0 ** 65, 1e150])
    bank["mu"][::3] = (mus[rng.integers(0, mus.size, 667)] * rng.choice([-1.0, 1.0], 667))
    o = oracle.simulate_bank(64, 0, m, dx, 1e-2, sigs, ar, bank, nthread=8)
    b, w = bank.copy(), np.zeros(m)
    result, st, rc = ctx.simulate(b, sigs, ar, w, 0, m, dx, 1e-2,
                                  options=mcgpu.make_options(kernel))
    assert rc == 0
    for f in ("seed", "x", "mu", "wmc", "index"):
        assert np.array_equal(b[f], o["bank"][f], equal_nan=f not in ("seed", "index")), f
    assert np.array_equal(result, o["result"])
    assert st["events"] == int(o["events"].sum())
    assert np.array_equal(w, o["tally_exact"])


@pytest.mark.parametrize("m,n,opts", [(10_200, 12_000, {"grid_blocks": 8, "block_size": 256}),
                                      (16_000, 6000, {}), (10_200, 3000, {"grid_blocks": 700})])
def test_wide_layer_histories_from_one_edge(ctx, oracle, m, n, opts):
    """All histories start in the first window: every block begins there, and
    blocks change windows as histories are parked, several times over."""
    import mcgpu
    _say(f"windows from one edge m={m} n={n} {opts}")
    sigs, ar, dx, bank = _case(m, n, m + n, 1.0)
    bank["index"] = 0
    bank["x"] = 0.0
    bank["mu"] = np.abs(bank["mu"])
    o = oracle.simulate_bank(64, 0, m, dx, 5e-2, sigs, ar, bank, nthread=8)
    b, w = bank.copy(), np.zeros(m)
    result, st, rc = ctx.simulate(b, sigs, ar, w, 0, m, dx, 5e-2,
                                  options=mcgpu.make_options("history", **opts))
    assert rc == 0
    for f in ("seed", "x", "mu", "wmc", "index"):
        assert np.array_equal(b[f], o["bank"][f]), f
    assert np.array_equal(result, o["result"])
    assert st["events"] == int(o["events"].sum())
    assert np.array_equal(w, o["tally_exact"])


@pytest.mark.parametrize("events_per_refill", [0, 1, 3])
@pytest.mark.parametrize("m,n", [(255, 500), (256, 3), (256, 4), (256, 65), (700, 1300)])
def test_histories_that_set_out_apart(ctx, oracle, m, n, events_per_refill):
    """Histories from one cell, most of them in one direction, some that end at
    once, in layers around the size from which they set out one event apart."""
    import mcgpu
    _say(f"one cell m={m} n={n} events_per_refill={events_per_refill}")
    sigs, ar, dx, bank = _case(m, n, m + n, 1.0)
    bank["index"] = m // 3
    bank["x"] = bank["index"] * dx
    bank["mu"] = np.where(np.arange(n) % 5 == 4, -1.0, 1.0) * np.abs(bank["mu"])
    bank["wmc"][::7] = 1e-3
    bank["index"][3::11] = m
    o = oracle.simulate_bank(64, 0, m, dx, 1e-2, sigs, ar, bank, nthread=8)
    b, w = bank.copy(), np.zeros(m)
    result, st, rc = ctx.simulate(
        b, sigs, ar, w, 0, m, dx, 1e-2,
        options=mcgpu.make_options("history", events_per_refill=events_per_refill, block_size=64,
                                   grid_blocks=1 + n // 200))
    assert rc == 0
    for f in ("seed", "x", "mu", "wmc", "index"):
        assert np.array_equal(b[f], o["bank"][f]), f
    assert np.array_equal(result, o["result"])
    assert st["events"] == int(o["events"].sum())
    assert np.array_equal(w, o["tally_exact"])


@pytest.mark.parametrize("n", [8290, 8320])
def test_long_run_of_a_layer_whose_cells_do_not_fit(ctx, oracle, n):
    """10,000 cells on two blocks, around the number of histories from which the
    layer goes in two windows."""
    _say(f"cells that do not fit, n={n}")
    _check(ctx, oracle, 10_000, n, 71, 1.0, 5e-2, grid_blocks=2)


@pytest.mark.parametrize("kernel", ["history", "event"])
@pytest.mark.parametrize("thick", [0.03, 1.0, 30.0])
@pytest.mark.parametrize("m", [1023, 1024, 4096])
def test_thick_cells_and_sorted_weights(ctx, oracle, m, thick, kernel):
    """Cells that absorb much of the weight, where the split follows the
    thickest one, and weights that rise through the bank."""
    import mcgpu
    n = 3000
    _say(f"thick cells m={m} {thick} {kernel}")
    sigs, ar, dx, bank = _case(m, n, m, np.geomspace(1e-6, 1.0, 3000))
    sigs = sigs * thick * m
    bank["index"][::2] = 0
    bank["x"][::2] = 0.0
    bank["mu"][::2] = np.abs(bank["mu"][::2])
    o = oracle.simulate_bank(64, 0, m, dx, 1e-8, sigs, ar, bank, nthread=8)
    b, w = bank.copy(), np.zeros(m)
    result, st, rc = ctx.simulate(b, sigs, ar, w, 0, m, dx, 1e-8,
                                  options=mcgpu.make_options(kernel))
    assert rc == 0
    for f in ("seed", "x", "mu", "wmc", "index"):
        assert np.array_equal(b[f], o["bank"][f]), f
    assert np.array_equal(result, o["result"])
    assert st["events"] == int(o["events"].sum())
    assert np.array_equal(w, o["tally_exact"])


@pytest.mark.parametrize("m", [1, 2, 74, 75, 144, 145, 273, 491, 817, 818])
def test_tally_copies(ctx, oracle, m):
    """Layers around the sizes at which the block keeps fewer copies of its
    tally, histories all from one face and from anywhere."""
    import mcgpu
    n = 1500
    _say(f"tally copies m={m}")
    sigs, ar, dx, bank = _case(m, n, m + 5, 1.0)
    bank["index"][::2] = 0
    bank["x"][::2] = 0.0
    bank["mu"][::2] = np.abs(bank["mu"][::2])
    o = oracle.simulate_bank(64, 0, m, dx, 1e-2, sigs, ar, bank, nthread=8)
    for grid in (0, 1):
        b, w = bank.copy(), np.zeros(m)
        result, st, rc = ctx.simulate(b, sigs, ar, w, 0, m, dx, 1e-2,
                                      options=mcgpu.make_options("history", grid_blocks=grid))
        assert rc == 0
        for f in ("seed", "x", "mu", "wmc", "index"):
            assert np.array_equal(b[f], o["bank"][f]), f
        assert np.array_equal(result, o["result"])
        assert st["events"] == int(o["events"].sum())
        assert np.array_equal(w, o["tally_exact"])


@pytest.mark.parametrize("kernel", ["history", "event"])
@pytest.mark.parametrize("lo", [0, 700, -5000])
def test_particles_outside_the_layer(ctx, oracle, lo, kernel):
    """Indices next to the layer and as far as 32 bits go: such a history ends
    at once, with its index as it was."""
    import mcgpu
    m, n = 40, 400
    _say(f"outside the layer lo={lo} {kernel}")
    sigs, ar, dx, bank = _case(m, n, 17, 1.0)
    far = np.array([-1, m, 1 << 28, 1 << 29, (1 << 29) + 5, 3 << 29, -(1 << 29), -(1 << 29) + 7,
                    (1 << 31) - 1, -(1 << 31)])
    bank["index"] += lo
    bank["x"] = (bank["index"] + 0.25) * dx
    bank["index"][::3] = np.clip(far[np.arange(134) % 10] + lo, -(1 << 31), (1 << 31) - 1)
    o = oracle.simulate_bank(64, lo, m, dx, 1e-2, sigs, ar, bank, nthread=8)
    b, w = bank.copy(), np.zeros(m)
    result, st, rc = ctx.simulate(b, sigs, ar, w, lo, lo + m, dx, 1e-2,
                                  options=mcgpu.make_options(kernel))
    assert rc == 0
    for f in ("seed", "x", "mu", "wmc", "index"):
        assert np.array_equal(b[f], o["bank"][f]), f
    assert np.array_equal(result, o["result"])
    assert st["events"] == int(o["events"].sum())
    assert np.array_equal(w, o["tally_exact"])


def test_long_run_with_scores(ctx, oracle):
    """The same for a device bank with counts and per-history scores, whose
    targets take LDS too: 9,000 cells in three windows."""
    import mcgpu
    import torch
    m, n = 9000, 9000
    rng = np.random.default_rng(81)
    sa, ss, g = rng.lognormal(0.5, 0.5, m), rng.lognormal(0, 0.5, m), rng.uniform(-1, 1, m)
    _, _, dx, bank = _case(m, n, 82, 1.0)
    _say("cells that do not fit, scores")
    o = oracle.forward_cells(0, m, dx, 1e-1, sa, ss, bank, g=g)
    db = mcgpu.bank_to_device(bank)
    dev = lambda x: torch.from_numpy(np.ascontiguousarray(x)).cuda()  # noqa: E731
    w, sc, dr = dev(np.zeros(m)), dev(np.full(n, 7.0)), dev(np.zeros(n, np.int8))
    ctx.forward_cells(db, dev(sa), dev(ss), w, 0, m, dx, 1e-1, g=dev(g), history_score=sc,
                      result=dr, options=mcgpu.make_options("history", grid_blocks=2))
    b = mcgpu.bank_from_device(db)
    for f in ("seed", "x", "mu", "wmc", "index"):
        assert np.array_equal(b[f], o["bank"][f]), f
    assert np.array_equal(dr.cpu().numpy().astype(np.int32), o["result"])
    assert np.array_equal(w.cpu().numpy(), o["tally_exact"])
    assert np.array_equal(sc.cpu().numpy().view(np.uint64), o["score"].view(np.uint64))
