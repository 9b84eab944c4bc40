"""GPU: windows without rings.  With more histories x windows than rings have
words, a history that crosses a window's edge waits for the next sweep, which
the host starts when it sees that histories are left: several sweeps here."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
M, N = 250_000, 11_000_000  # 50 windows, 62 with scores: more than 2^29 / N


def _inputs():
    import torch
    g = torch.Generator(device="cuda").manual_seed(9)
    u = lambda n: torch.rand(n, generator=g, device="cuda", dtype=torch.float64)  # noqa: E731
    dx = 1.0 / M
    sa, si = (0.1 + 0.2 * u(M)) / dx, (0.1 + 0.4 * u(M)) / dx
    # near the windows' edges (every 5,000 and every 4,033 cells) and between them
    at = torch.randint(0, M, (N,), generator=g, device="cuda")
    at[::2] = (at[::2] // 5000 * 5000 + torch.randint(-3, 3, (N // 2,), generator=g,
                                                     device="cuda")).clamp(0, M - 1)
    bank = {"seed": torch.randint(0, (1 << 63) - 1, (N,), generator=g, device="cuda"),
            "x": (at + u(N)) * dx, "mu": 2 * u(N) - 1, "wmc": 0.5 + 0.5 * u(N),
            "index": at.to(torch.int32)}
    return dx, sa, si, bank


def _same(a, b):
    import torch
    return all(torch.equal(a[k].view(torch.int64) if a[k].dtype == torch.float64 else a[k],
                           b[k].view(torch.int64) if b[k].dtype == torch.float64 else b[k])
               for k in a)


def test_sweeps_equal_the_event_kernel():
    import mcgpu
    import torch
    print("windows without rings, against the event kernel", flush=True)
    dx, sa, si, bank = _inputs()
    sigs = sa + si
    out = {}
    with mcgpu.Context(0) as ctx:
        for kernel in ("history", "event"):
            b = {k: v.clone() for k, v in bank.items()}
            w = torch.zeros(M, dtype=torch.float64, device="cuda")
            r = torch.zeros(N, dtype=torch.int8, device="cuda")
            ev = torch.zeros(N, dtype=torch.int64, device="cuda")
            st, _ = ctx.simulate_device(b, sigs, sa / sigs, w, 0, M, dx, 0.05, result=r, events=ev,
                                        options=mcgpu.make_options(kernel))
            st.pop("kernel_ms")
            out[kernel] = ({**b, "w": w, "r": r, "ev": ev}, st)
    assert _same(out["history"][0], out["event"][0])
    assert out["history"][1] == out["event"][1]
    assert out["event"][0]["ev"].max() > 20


def test_sweeps_keep_the_scores():
    import mcgpu
    import torch
    print("windows without rings, scores", flush=True)
    dx, sa, si, bank = _inputs()
    g = torch.linspace(-1, 1, M, dtype=torch.float64, device="cuda")
    out = []
    with mcgpu.Context(0) as ctx:
        for batched in (False, True):
            b = {k: v.clone() for k, v in bank.items()}
            w = torch.zeros(M, dtype=torch.float64, device="cuda")
            sc = torch.zeros(N, dtype=torch.float64, device="cuda")
            if batched:
                ctx.forward_cells_batch([(0, M, dx, 0.05, 0, 0, N)], b, sa, si, w, g=g,
                                        history_score=sc)
            else:
                ctx.forward_cells(b, sa, si, w, 0, M, dx, 0.05, g=g, history_score=sc)
            out.append({**b, "w": w, "sc": sc})
    assert _same(*out)
