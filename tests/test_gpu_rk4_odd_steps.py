"""Odd numbers of fused RK4 steps, whose stages end in the ping-pong partner:
the caller's array holds the result wherever the steps run, also on the null
stream while another stream of the process captures."""
from __future__ import annotations

import ctypes

import numpy as np
import pytest

from tests.cases import mesh_case, random_state
from wavedg_amd import capi

pytestmark = pytest.mark.gpu

BLOCKING, NON_BLOCKING = 0, 1  # hipStreamDefault, hipStreamNonBlocking


def _wave(v, e, n):
    gm = capi.Mesh(v, e)
    w = capi.Wave2D(gm, n, np.ones(gm.n_boundary, dtype=np.int32))
    return w, 0.4 * gm.min_h() / n**2


@pytest.mark.parametrize("flags", [BLOCKING, NON_BLOCKING])
@pytest.mark.parametrize("mode", [0, 1, 2])  # global, thread-local, relaxed
def test_null_stream_steps_beside_a_capture(cuda, flags, mode):
    """While a blocking stream captures, HIP refuses to say whether the null
    stream does; launches on the null stream run all the same."""
    torch = cuda
    assert torch.cuda.current_stream().cuda_stream == 0
    hip = ctypes.CDLL("libamdhip64.so")
    w, dt = _wave(*mesh_case("skewed6x5"), 4)
    u0 = torch.tensor(random_state(w.ndof, 3), device="cuda")
    ref = u0.clone()
    for _ in range(2):  # scratch in place before the capture
        ref.copy_(u0)
        w.rk4(ref, dt, 3)
    s, g = ctypes.c_void_p(), ctypes.c_void_p()
    assert hip.hipStreamCreateWithFlags(ctypes.byref(s), flags) == 0
    x = u0.clone()
    torch.cuda.synchronize()
    assert hip.hipStreamBeginCapture(s, mode) == 0
    try:
        w.rk4(x, dt, 3)
    finally:
        ended = hip.hipStreamEndCapture(s, ctypes.byref(g))
        if g:
            hip.hipGraphDestroy(g)
        hip.hipStreamDestroy(s)
        hip.hipGetLastError()
    assert ended == 0  # the steps left the capture as it was
    torch.cuda.synchronize()
    assert torch.equal(x, ref)
