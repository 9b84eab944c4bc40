"""Performance cases: what a user of mcgpu has it do, through its public entry points.

A case is a dict of plain values.  `prepare` makes what a program holds before
the call (source banks, cross sections, plans), `run` makes one pass, `work`
states the least bytes and floating-point operations of a pass, and `exact`
repeats small and middle cases in plain torch binary64 arithmetic.

Every transport pass starts from the source bank again: the calls advance the
bank in place, so a program that keeps its source copies it (or draws it anew
with create_particles) before each call.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "mc-mpi_amd"))

import mcgpu  # noqa: E402
from mcgpu.autograd import SlabProblem, slab_tally  # noqa: E402

DEV = "cuda"
EPS = 1e-4
MAXREAL = 1.7976931348623157e308
X_INI = 0.7071067690849304  # the cycle loop's source (mc-mpi_amd/reference_job.yaml)


def listed():
    return [
        # a short probe of 1,000 histories on the 100-cell slab, source drawn on
        # the device: the time of one history and of the launches
        {"name": "source100_1k", "kind": "source", "m": 100, "n": 1000, "kernel": "history"},
        # the drop-in call on host buffers, the 100-cell slab at its own size
        {"name": "host100_100k", "kind": "host", "m": 100, "n": 100_000},
        # one rank's interior layer of a decomposed slab, flux from both faces,
        # an odd number of particles
        {"name": "inflow1000_2m", "kind": "bank", "law": "inflow", "m": 1000, "n": 1_999_999,
         "kernel": "history"},
        # the 10,000-cell slab: the main workload, thin cells, long histories
        {"name": "slab10k_8m", "kind": "bank", "law": "lognormal", "m": 10_000, "n": 8_000_000,
         "kernel": "history"},
        # the same slab with the event kernel
        {"name": "slab10k_event_1m", "kind": "bank", "law": "lognormal", "m": 10_000,
         "n": 1_000_000, "kernel": "event"},
        # a layer of more cells than a tally in LDS holds
        {"name": "slab20k_200k", "kind": "bank", "law": "lognormal", "m": 20_000, "n": 200_000,
         "kernel": "history"},
        # many slabs of 32 to 8,192 cells and 100 to 100,000 particles in one plan
        {"name": "batch512", "kind": "batch", "slabs": 512, "scale": 0.1},
        # forward and gradient of the 1,000-cell slab through autograd
        {"name": "grad1000_1m", "kind": "grad", "m": 1000, "n": 1_000_000, "hint": True},
        # a small ragged one whose target is known only in the backward
        {"name": "grad313_20k", "kind": "grad", "m": 313, "n": 20_011, "hint": False},
        # 64 slabs' forward and gradient, one launch each
        {"name": "gradbatch64x50k", "kind": "gradbatch", "slabs": 64, "m": 1000, "n": 50_000},
        # the synchronous cycle loop: the reference job's configuration, eight
        # ranks and one
        {"name": "cycle8_2m", "kind": "cycle", "ranks": 8, "m": 1000, "n": 2_000_000,
         "per_cycle": 100_000},
        {"name": "cycle1_2m", "kind": "cycle", "ranks": 1, "m": 1000, "n": 2_000_000,
         "per_cycle": 100_000},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["source", "host", "bank", "bank", "event", "batch", "grad", "gradbatch",
                       "cycle"])
    if kind == "source":
        return {"kind": "source", "m": _log_int(rng, 30, 400), "n": _log_int(rng, 100, 30_000),
                "kernel": rng.choice(["history", "history", "event"])}
    if kind == "host":
        return {"kind": "host", "m": _log_int(rng, 50, 1500), "n": _log_int(rng, 1000, 400_000)}
    if kind == "bank":
        if rng.random() < 0.3:
            return {"kind": "bank", "law": "inflow", "m": _log_int(rng, 200, 2000),
                    "n": _log_int(rng, 50_000, 3_000_000), "kernel": "history"}
        m = _log_int(rng, 200, 24_000)
        most = 4e10 / m if m <= 10_000 else 2e9 / m
        return {"kind": "bank", "law": "lognormal", "m": m,
                "n": _log_int(rng, min(20_000, 0.4 * most), min(3e6, most)), "kernel": "history"}
    if kind == "event":
        m = _log_int(rng, 200, 10_000)
        return {"kind": "bank", "law": "lognormal", "m": m,
                "n": _log_int(rng, 20_000, min(2e6, 1e10 / m)), "kernel": "event"}
    if kind == "batch":
        return {"kind": "batch", "slabs": _log_int(rng, 24, 700),
                "scale": round(rng.uniform(0.02, 0.1), 3)}
    if kind == "grad":
        m = _log_int(rng, 100, 3000)
        return {"kind": "grad", "m": m, "n": _log_int(rng, 5000, min(1.5e6, 1e9 / m)),
                "hint": rng.random() < 0.7}
    if kind == "gradbatch":
        return {"kind": "gradbatch", "slabs": rng.randint(5, 90), "m": _log_int(rng, 200, 1500),
                "n": _log_int(rng, 2000, 40_000)}
    return {"kind": "cycle", "ranks": rng.choice([1, 2, 3, 5, 8]), "m": _log_int(rng, 200, 1500),
            "n": _log_int(rng, 100_000, 2_000_000), "per_cycle": _log_int(rng, 20_000, 200_000)}


# ------------------------------------------------------------------ inputs


def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


def _uniform(g, n):
    return torch.rand(n, generator=g, device=DEV, dtype=torch.float64)


def _lognormal(g, n, mu, sigma):
    return torch.exp(mu + sigma * torch.randn(n, generator=g, device=DEV, dtype=torch.float64))


def _seeds(g, n):
    """63-bit RNG states, one per history."""
    return torch.randint(0, (1 << 63) - 1, (n,), generator=g, device=DEV, dtype=torch.int64)


def _bank(g, n, x=0.0, index=0, mu=None, wmc=1.0):
    full = lambda v, t: v if torch.is_tensor(v) else torch.full((n,), v, dtype=t, device=DEV)  # noqa: E731
    return {"seed": _seeds(g, n), "x": full(x, torch.float64),
            "mu": torch.sqrt(_uniform(g, n)) if mu is None else mu,
            "wmc": full(wmc, torch.float64), "index": full(index, torch.int32)}


def _chain_seed(seed):
    return (5127801 + 2654435761 * int(seed)) & ((1 << 62) - 1)


def _slab100(m):
    """sigma_a = 0.5 + 0.5 x, sigma_s = 1 - 0.5 x at the cell centres."""
    xc = (torch.arange(m, dtype=torch.float64, device=DEV) + 0.5) * (1.0 / m)
    return torch.full((m,), 1.5, dtype=torch.float64, device=DEV), (0.5 + 0.5 * xc) / 1.5


def _problem(case, seed):
    """Inputs of one case, as plain torch tensors and numbers."""
    g = _gen(seed)
    kind = case["kind"]
    m, n = case.get("m"), case.get("n")
    d = {"lo": 0, "hi": m, "dx": 1.0 / m if m else None, "min_w": 1e-3}
    if kind == "source":
        d["min_w"] = 1e-2
        d["sigs"], d["ar"] = _slab100(m)
        # a source position and a seed of its own for each seed
        d["x_ini"] = 0.25 + 0.5 * float(torch.rand(1, generator=g, device=DEV, dtype=torch.float64))
        d["chain"] = _chain_seed(seed)
    elif kind == "host":
        d["min_w"] = 1e-2
        d["sigs"], d["ar"] = _slab100(m)
        d["bank"] = _bank(g, n, mu=torch.ones(n, dtype=torch.float64, device=DEV))
    elif kind == "bank" and case["law"] == "inflow":
        # the middle fifth of a 5 m-cell slab on [0, 1], inflow through both faces
        dx_g = 1.0 / (5 * m)
        lo = 2 * m
        x0, x1 = lo * dx_g, (lo + m) * dx_g
        d.update(lo=lo, hi=lo + m, dx=(x1 - x0) / m, min_w=1e-2)
        xc = x0 + (torch.arange(m, dtype=torch.float64, device=DEV) + 0.5) * d["dx"]
        d["sigs"] = torch.full((m,), 1.5, dtype=torch.float64, device=DEV)
        d["ar"] = (0.5 + 0.5 * xc) / 1.5
        left = torch.arange(n, device=DEV) < n // 2
        mu = torch.sqrt(_uniform(g, n))
        d["bank"] = _bank(g, n, x=torch.where(left, x0, x1).to(torch.float64),
                          index=torch.where(left, lo, lo + m - 1).to(torch.int32),
                          mu=torch.where(left, mu, -mu), wmc=0.1 + 0.9 * _uniform(g, n))
    elif kind == "bank":
        sa, ss = _lognormal(g, m, 0.0, 0.5), _lognormal(g, m, 0.5, 0.5)
        d["sigs"] = sa + ss
        d["ar"] = sa / d["sigs"]
        d["bank"] = _bank(g, n)
    elif kind == "batch":
        u = _uniform(_gen(4001), 2 * case["slabs"]).tolist()  # the layout is the case's
        slabs, c0, p0 = [], 0, 0
        for s in range(case["slabs"]):
            ms = int(math.exp(math.log(32.0) + u[2 * s] * math.log(8192.0 / 32.0)))
            ns = max(1, int(case["scale"] * math.exp(math.log(1e3) + u[2 * s + 1] * math.log(1e3))))
            slabs.append((0, ms, 1.0 / ms, 1e-3, c0, p0, ns))
            c0, p0 = c0 + ms, p0 + ns
        d["slabs"] = slabs
        d["sigs"] = _lognormal(g, c0, 0.0, 1.0)
        d["ar"] = 1.0 - (0.1 + 0.89 * _uniform(g, c0))
        d["bank"] = _bank(g, p0)
    elif kind == "grad":
        d["sig_a"], d["sig_s"] = _lognormal(g, m, 0.0, 0.5), _lognormal(g, m, 0.0, 0.5)
        d["target"] = _target(m)
        d["bank"] = _bank(g, n)
    elif kind == "gradbatch":
        S = case["slabs"]
        d["slabs"] = [(0, m, 1.0 / m, 1e-3, s * m, s * n, n) for s in range(S)]
        d["sig_a"], d["sig_s"] = _lognormal(g, S * m, 0.0, 0.5), _lognormal(g, S * m, 0.0, 0.5)
        d["target"] = _target(m).repeat(S)
        d["bank"] = _bank(g, S * n)
    elif kind == "cycle":
        R = case["ranks"]
        dx_g = 1.0 / m
        per = m // R
        ranks, dxs = [], []
        for r in range(R):
            lo = r * per
            hi = m if r == R - 1 else lo + per
            x0, x1 = lo * dx_g, hi * dx_g
            dx = (x1 - x0) / (hi - lo)
            k = {"min_index": lo, "max_index": hi, "dx": dx, "particle_min_weight": 1e-12,
                 "left_border": r == 0, "right_border": r == R - 1, "cell_offset": lo}
            if x0 <= X_INI < x1:
                k.update(nb_particles_create=n, seed=_chain_seed(seed), x_ini=X_INI, wmc=1e-8)
                d["index"], d["chain"] = int(X_INI / dx), k["seed"]
            ranks.append(k)
            dxs += [dx] * (hi - lo)
        xc = (np.arange(m) + 0.5) * dx_g
        d.update(ranks=ranks, dxs=dxs, sigs=np.exp(-xc), ar=np.full(m, 0.5))
    return d


def _target(m):
    """The absorbed weight of the tenth of the cells from 0.8 m on."""
    t = torch.zeros(m, dtype=torch.float64, device=DEV)
    t[(8 * m) // 10:(9 * m) // 10] = 1.0
    return t


_ctx = None


def _context():
    """One context for the whole program, as its calls come one after the other."""
    global _ctx
    if _ctx is None:
        _ctx = mcgpu.Context(0)
    return _ctx


class _State:
    pass


def prepare(case, seed):
    s = _State()
    s.case, s.d, s.ctx = case, _problem(case, seed), _context()
    d, kind = s.d, case["kind"]
    if kind in ("source", "bank"):
        s.options = mcgpu.make_options(case["kernel"])
    if kind == "source":
        s.bank = {k: v for k, v in _bank(_gen(0), case["n"]).items()}
        s.result = torch.empty(case["n"], dtype=torch.int8, device=DEV)
    elif kind == "host":
        s.particles = np.zeros(case["n"], dtype=mcgpu.PARTICLE)
        for f, v in d["bank"].items():
            s.particles[f] = v.cpu().numpy()
        s.sigs, s.ar = d["sigs"].cpu().numpy(), d["ar"].cpu().numpy()
        del d["bank"]
    elif kind in ("bank", "gradbatch"):
        s.work = {k: v.clone() for k, v in d["bank"].items()}
        s.result = torch.empty(len(d["bank"]["x"]), dtype=torch.int8, device=DEV)
    elif kind == "batch":
        s.work = {k: v.clone() for k, v in d["bank"].items()}
        s.result = torch.empty(len(d["bank"]["x"]), dtype=torch.int8, device=DEV)
        s.weights = torch.zeros(len(d["sigs"]), dtype=torch.float64, device=DEV)
        s.plan = mcgpu.Batch(s.ctx, d["slabs"], d["sigs"], d["ar"], s.weights, s.work, s.result)
    elif kind == "grad":
        s.problem = SlabProblem(s.ctx, d["bank"], d["lo"], d["hi"], d["dx"], d["min_w"])
        s.sig_a = d["sig_a"].clone().requires_grad_(True)
        s.sig_s = d["sig_s"].clone().requires_grad_(True)
    return s


def _restore(s):
    for k, v in s.d["bank"].items():
        s.work[k].copy_(v)
    return s.work


def run(s):
    case, d, ctx = s.case, s.d, s.ctx
    kind = case["kind"]
    zeros = lambda k: torch.zeros(k, dtype=torch.float64, device=DEV)  # noqa: E731
    if kind == "source":
        ctx.create_particles(d["chain"], 0, s.bank, d["x_ini"], 1.0, d["dx"])
        w = zeros(case["m"])
        st, _ = ctx.simulate_device(s.bank, d["sigs"], d["ar"], w, d["lo"], d["hi"], d["dx"],
                                    d["min_w"], result=s.result, options=s.options)
        return {**s.bank, "weights": w, "result": s.result, "events": st["events"]}
    if kind == "host":
        p = s.particles.copy()
        w = np.zeros(case["m"])
        result, st, _ = ctx.simulate(p, s.sigs, s.ar, w, d["lo"], d["hi"], d["dx"], d["min_w"])
        return {"seed": p["seed"].view(np.int64), "x": p["x"], "mu": p["mu"], "wmc": p["wmc"],
                "index": p["index"], "weights": w, "result": result, "events": st["events"]}
    if kind == "bank":
        bank = _restore(s)
        w = zeros(case["m"])
        st, _ = ctx.simulate_device(bank, d["sigs"], d["ar"], w, d["lo"], d["hi"], d["dx"],
                                    d["min_w"], result=s.result, options=s.options)
        return {**bank, "weights": w, "result": s.result, "events": st["events"]}
    if kind == "batch":
        bank = _restore(s)
        s.weights.zero_()
        st = s.plan.run()
        return {**bank, "weights": s.weights, "result": s.result, "events": st["events"]}
    if kind == "grad":
        s.sig_a.grad = s.sig_s.grad = None
        tally = slab_tally(s.sig_a, s.sig_s, s.problem, d["target"] if case["hint"] else None)
        (tally * d["target"]).sum().backward()
        return {"tally": tally.detach(), "grad_a": s.sig_a.grad, "grad_s": s.sig_s.grad}
    if kind == "gradbatch":
        total = len(d["sig_a"])
        bank = _restore(s)
        w, ga, gs = zeros(total), zeros(total), zeros(total)
        score = torch.empty(len(bank["x"]), dtype=torch.float64, device=DEV)
        ctx.forward_cells_batch(d["slabs"], bank, d["sig_a"], d["sig_s"], w, g=d["target"],
                                history_score=score, result=s.result)
        ctx.adjoint_cells_batch(d["slabs"], d["bank"], d["sig_a"], d["sig_s"], d["target"], ga, gs,
                                history_score=score)
        return {"tally": w, "grad_a": ga, "grad_s": gs, "score": score}
    w = np.zeros(case["m"])
    out, st = ctx.sync_cycle(d["ranks"], d["sigs"], d["ar"], w, case["per_cycle"], case["n"])
    return {"weights": w, "events": st["events"], "cycles": st["cycles"],
            "left": [o["n_left"] for o in out], "right": [o["n_right"] for o in out],
            "killed": [o["n_killed"] for o in out]}


# -------------------------------------------------------------------- work

# floating-point operations one event cannot do without: the draw (4), the
# edge distance (4), the collision test (3), an exponential (10), the deposit
# and the sums (5); a replayed event adds its two gradient terms (10)
EVENT_FLOPS, GRAD_FLOPS = 26, 10
# events per history and cell, measured
PER_CELL = {"source": 0.55, "host": 1.01, "lognormal": 0.98, "inflow": 0.6, "batch": 0.7,
            "grad": 1.03, "cycle": 0.58}


def work(case):
    kind, m, n = case["kind"], case.get("m"), case.get("n")
    particle = 36  # seed, x, mu, wmc, index
    if kind == "batch":
        # mean cells (8192 - 32) / ln 256, mean particles 999,000 / ln 1000
        m = (8192 - 32) / math.log(256)
        n = case["slabs"] * case["scale"] * 999_000 / math.log(1000)
        return {"bytes": n * (2 * particle + 1) + 24 * m * case["slabs"],
                "flops": PER_CELL["batch"] * m * n * EVENT_FLOPS}
    if kind == "gradbatch":
        n *= case["slabs"]
    if kind in ("grad", "gradbatch"):
        # forward (and, the target known late, a replay for the scores), gradient replay
        replays = 3 if kind == "grad" and not case["hint"] else 2
        events = PER_CELL["grad"] * m * n
        return {"bytes": n * particle * replays + 48 * m,
                "flops": events * (replays * EVENT_FLOPS + GRAD_FLOPS)}
    per = PER_CELL[case["law"] if kind == "bank" else kind]
    return {"bytes": n * (2 * particle + 1) + 24 * m if kind != "cycle" else 24 * m + n,
            "flops": per * m * n * EVENT_FLOPS}


# ------------------------------------------------------------------- exact


def _chain(seed, n):
    """Outputs 1 .. n of the seed chain s <- (G s + C) mod 2^63."""
    G, C = 5177284530976225183, 2096348467109453893
    k = torch.arange(1, n + 1, dtype=torch.int64, device=DEV)
    A, B = G, C
    ra = torch.ones(n, dtype=torch.int64, device=DEV)
    rb = torch.zeros(n, dtype=torch.int64, device=DEV)
    wrap = lambda v: (v + (1 << 63)) % (1 << 64) - (1 << 63)  # noqa: E731
    while int(k.max()) > 0:
        odd = (k & 1).bool()
        ra, rb = torch.where(odd, wrap(A) * ra, ra), torch.where(odd, wrap(A) * rb + wrap(B), rb)
        B = (A * B + B) % (1 << 64)
        A = A * A % (1 << 64)
        k = k >> 1
    return (ra * wrap(seed) + rb) & ((1 << 63) - 1)


def _rnd(seed):
    seed = (6364136223846793005 * seed + 1442695040888963407) & ((1 << 63) - 1)
    return seed, seed.to(torch.float64) * 2.0 ** -63


def _drawn(chain, n, x_ini, wmc, index):
    seed, h = _rnd(_chain(chain, n))
    return {"seed": seed, "x": torch.full((n,), x_ini, dtype=torch.float64, device=DEV),
            "mu": 2 * h - 1, "wmc": torch.full((n,), wmc, dtype=torch.float64, device=DEV),
            "index": torch.full((n,), index, dtype=torch.int32, device=DEV)}


def _walk(bank, sa, si, dxs, off, lo, hi, min_w, g=None, T=None):
    """Every history of `bank` to its end, all of them one event at a time.
    Cell c of the concatenated arrays holds index c - off; a history lives
    while its cell is in [lo, hi) (off, lo, hi per particle) and its weight at
    least min_w.  Returns the final state, the absorbed weight per cell, the
    scores sum g dw, and with T (the scores) the two gradients."""
    n, total = len(bank["x"]), len(sa)
    out = {k: v.clone() for k, v in bank.items()}
    # copies of the sums, one per group of histories: at first every history is in one cell
    copies = max(1, min(1024, (1 << 24) // total))
    tally, ga, gs = (torch.zeros(total * copies, dtype=torch.float64, device=DEV) for _ in range(3))
    score = torch.zeros(n, dtype=torch.float64, device=DEV)
    ids = torch.arange(n, device=DEV)
    s, x, mu, w = (bank[k].clone() for k in ("seed", "x", "mu", "wmc"))
    c = bank["index"].to(torch.int64) + off
    P = torch.zeros_like(score)
    Th = T.clone() if T is not None else None
    step = 0
    while True:
        alive = (w >= min_w) & (c >= lo) & (c < hi)
        if step % 16 == 0:
            gone = ~alive
            at = ids[gone]
            for k, v in (("seed", s), ("x", x), ("mu", mu), ("wmc", w)):
                out[k][at] = v[gone]
            out["index"][at] = (c - off)[gone].to(torch.int32)
            score[at] = P[gone]
            keep = alive.nonzero().squeeze(1)
            if len(keep) == 0:
                tally, ga, gs = (v.view(total, copies).sum(1) for v in (tally, ga, gs))
                return out, tally, score, ga, gs
            if len(keep) < len(ids):
                ids, s, x, mu, w, c, P, off, lo, hi = (v[keep] for v in
                                                       (ids, s, x, mu, w, c, P, off, lo, hi))
                Th = Th[keep] if Th is not None else None
                alive = alive[keep]
        step += 1
        cc = torch.where(alive, c, lo)
        to = cc * copies + ids % copies
        a, b, dx, index = sa[cc], si[cc], dxs[cc], c - off
        s1, h = _rnd(s)
        back = mu < 0
        edge = torch.where(back, index, index + 1).to(torch.float64) * dx
        far = torch.where(mu.abs() > EPS, (edge - x) / mu, MAXREAL)
        di = torch.where(b > EPS, -torch.log(h) / b, MAXREAL)
        hit = di < far
        di = torch.minimum(di, far)
        s2, h2 = _rnd(s1)
        dw = (1 - torch.exp(-a * di)) * w
        dw = torch.where(alive, dw, 0.0)
        if g is not None:
            gc = g[cc]
            w1 = w - dw
            if Th is not None:
                left = Th - P
                ta = di * (gc * w1 - (left - gc * dw))
                ti = torch.where(b > EPS, torch.where(hit, 1.0 / b - di, -di) * left, 0.0)
                ga.index_add_(0, to, torch.where(alive, ta, 0.0))
                gs.index_add_(0, to, torch.where(alive, ti, 0.0))
            P = P + gc * dw
        tally.index_add_(0, to, dw)
        moved = torch.where(hit, x + di * mu, edge)
        x = torch.where(alive, moved, x)
        s = torch.where(alive, torch.where(hit, s2, s1), s)
        c = torch.where(alive & ~hit, torch.where(back, c - 1, c + 1), c)
        mu = torch.where(alive & hit, 2 * h2 - 1, mu)
        w = w - dw


def exact(case, seed):
    kind, m = case["kind"], case.get("m")
    if kind == "batch" or m > 2500:
        return None  # tens of thousands of steps one after the other
    d = _problem(case, seed)
    grads = kind in ("grad", "gradbatch")
    if kind == "cycle":
        bank = _drawn(d["chain"], case["n"], X_INI, 1e-8, d["index"])
        sigs, ar = (torch.from_numpy(d[k]).to(DEV) for k in ("sigs", "ar"))
        dxs, min_w = torch.tensor(d["dxs"], dtype=torch.float64, device=DEV), 1e-12
    else:
        bank = d["bank"] if "bank" in d else _drawn(d["chain"], case["n"], d["x_ini"], 1.0,
                                                    int(d["x_ini"] / d["dx"]))
        sigs, ar, min_w = d.get("sigs"), d.get("ar"), d["min_w"]
        total = len(d["sig_a"]) if grads else m
        dxs = torch.full((total,), d["dx"], dtype=torch.float64, device=DEV)
    sa, si = (d["sig_a"], d["sig_s"]) if grads else (sigs * ar, sigs * (1.0 - ar))
    n = len(bank["x"])
    first = torch.zeros(n, dtype=torch.int64, device=DEV)
    if kind == "gradbatch":
        first = torch.arange(n, device=DEV) // case["n"] * m
    off = first - (d["lo"] if kind != "cycle" else 0)
    g = d["target"] if grads else None
    end, tally, score, _, _ = _walk(bank, sa, si, dxs, off, first, first + m, min_w, g)
    if grads:
        _, _, _, ga, gs = _walk(bank, sa, si, dxs, off, first, first + m, min_w, g, score)
        out = {"tally": tally, "grad_a": ga, "grad_s": gs}
        return {**out, "score": score} if kind == "gradbatch" else out
    if kind == "cycle":
        return {"weights": tally, "events": None, "cycles": None, "left": None, "right": None,
                "killed": None}
    return {"seed": None, "x": end["x"], "mu": end["mu"], "wmc": end["wmc"], "index": None,
            "weights": tally, "result": None, "events": None}
