"""What the trained networks gain: WaveHoltz to 1e-6 on held-out problems
(64 x 64 and 128 x 128 quads, P = 4, seeds never used in training), batched,
with and without the learned warm start.  The warm-started solve must
converge to the same fixed point (the plain iteration judges the residual) in
fewer updates."""
from __future__ import annotations

import os

import numpy as np
import pytest

from wavedg_amd import warmstart

pytestmark = pytest.mark.gpu

WEIGHTS = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "wavedg_amd", "weights")


@pytest.mark.parametrize("M,count", [(64, 8), (128, 4)])
def test_warm_start_reduces_iterations(cuda, M, count):
    torch = cuda
    ws = warmstart.WarmStart.load(os.path.join(WEIGHTS, f"warmstart_m{M}_p4.npz"))
    assert ws.M == M
    print(f"warm start {M}^2: {count} held-out problems", flush=True)
    specs = warmstart.specs_for(range(warmstart.EVAL_SEED0 + 500, warmstart.EVAL_SEED0 + 500 + count))
    tol = 1e-6
    print("warm start: plain batched solve", flush=True)
    Wp, itp, _, resp, _, tp = warmstart.solve_batched(ws, specs, tol, 300, warm=False)
    print(f"plain: iterations {itp}, {tp:.1f} s", flush=True)
    Ww, itw, _, resw, t_inf, tw = warmstart.solve_batched(ws, specs, tol, 300, warm=True)
    print(f"warm: iterations {itw}, {tw:.1f} s (+{t_inf * 1e3:.1f} ms inference)", flush=True)
    assert max(resp) <= tol and max(resw) <= tol
    assert np.mean(itw) < 0.95 * np.mean(itp)
    # the same fixed point, to the accuracy the residual tolerance allows
    for a, b in zip(Ww, Wp):
        assert float(torch.linalg.norm(a - b) / torch.linalg.norm(b)) < 2e-5
    # the prediction itself is within 20 % of the converged solution
    pred = ws.predict(specs)
    err = [float(torch.linalg.norm(p - b) / torch.linalg.norm(b)) for p, b in zip(pred, Wp)]
    print(f"prediction relative errors {np.round(err, 3)}", flush=True)
    assert np.median(err) < 0.2


def test_features_walk_any_iterable(cuda):
    """Problems given one by one (an iterator) into the caller's array, with
    different numbers of sources, give each problem's own image."""
    torch = cuda
    ws = warmstart.WarmStart(16, max_batch=4)
    src = [[0.3, 0.6, 0.02, 1.0], [0.7, 0.4, 0.01, -0.5], [0.5, 0.5, 0.03, 2.0]]
    specs = [dict(omega=20.0 + 5.0 * k, sources=src[:k + 1]) for k in range(3)]
    want = torch.cat([ws.features([sp]) for sp in specs])
    shape = (3, 16, 16, warmstart.IN_LD)
    for given in (specs, tuple(specs), iter(specs)):
        out = torch.full(shape, -7.0, dtype=torch.bfloat16, device="cuda")
        assert ws.features(given, out) is out
        assert torch.equal(out, want)
    assert tuple(ws.features([]).shape) == (0, 16, 16, warmstart.IN_LD)
