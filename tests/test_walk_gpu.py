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


def _check(ctx, oracle, m, n, seed, wmc, min_w, **opts):
    import mcgpu
    sigs, ar, dx, bank = _case(m, n, seed, wmc)
    o = oracle.simulate_bank(64, 0, m, dx, min_w, sigs, ar, bank, nthread=8)
    b, w = bank.copy(), np.zeros(m)
    result, st, rc = ctx.simulate(b, sigs, ar, w, 0, m, dx, min_w,
                                  options=mcgpu.make_options("history", **opts))
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
