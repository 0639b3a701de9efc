"""Odd numbers of fused RK4 steps, whose stages end in the ping-pong partner:
the caller's array holds the result wherever the steps run, also on the null
stream while another stream of the process captures, and what the handle
keeps for them in device memory is bounded and pays."""
from __future__ import annotations

import ctypes

import numpy as np
import pytest

from tests.cases import mesh_case, random_state
from wavedg_amd import capi, meshgen

pytestmark = pytest.mark.gpu

BLOCKING, NON_BLOCKING = 0, 1  # hipStreamDefault, hipStreamNonBlocking


def _wave(v, e, n):
    gm = capi.Mesh(v, e)
    w = capi.Wave2D(gm, n, np.ones(gm.n_boundary, dtype=np.int32))
    return w, 0.4 * gm.min_h() / n**2


@pytest.mark.parametrize("flags", [BLOCKING, NON_BLOCKING])
@pytest.mark.parametrize("mode", [0, 1, 2])  # global, thread-local, relaxed
@pytest.mark.parametrize("before", [1, 2])
def test_null_stream_steps_beside_a_capture(cuda, flags, mode, before):
    """While a blocking stream captures, HIP refuses to say whether the null
    stream does; launches on the null stream run all the same.  With one odd
    call before, this call is the one that asks for the third buffer."""
    torch = cuda
    assert torch.cuda.current_stream().cuda_stream == 0
    hip = ctypes.CDLL("libamdhip64.so")
    w, dt = _wave(*mesh_case("skewed6x5"), 4)
    u0 = torch.tensor(random_state(w.ndof, 3), device="cuda")
    ref = u0.clone()
    for _ in range(before):
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


def _free(torch):
    torch.cuda.synchronize()
    return torch.cuda.mem_get_info()[0]


def test_third_buffer_comes_with_the_second_odd_call(cuda):
    """One odd call leaves no more device memory in use than an even one; the
    calls after it at most one further state, and every call gives the bits
    that the same steps in an even call and one step give."""
    torch = cuda
    n, nx = 6, 240
    w, dt = _wave(*meshgen.perturbed_rect(nx, nx, 0.2, 77), n)
    size = 8 * w.ndof
    u0 = torch.tensor(random_state(w.ndof, 5), device="cuda")
    x, outs = u0.clone(), [torch.empty_like(u0) for _ in range(3)]
    w.rk4(x, dt, 2)
    free = _free(torch)
    for call, out in enumerate(outs):
        out.copy_(u0)
        w.rk4(out, dt, 3)
        used = free - _free(torch)
        print(f"odd call {call}: {used / size:.2f} states more", flush=True)
        assert used == 0 if call == 0 else used <= size + (4 << 20)
    x.copy_(u0)
    w.rk4(x, dt, 2)
    w.rk4(x, dt, 1)
    assert all(torch.equal(x, o) for o in outs)


@pytest.mark.parametrize("precision,n,mb,buffer", [
    (capi.F64, 8, 75, False), (capi.F64, 5, 70, False), (capi.F32, 8, 75, False), (capi.F32, 3, 80, True),
    (capi.F64, 8, 60, True), (capi.F64, 8, 90, True)])
def test_copy_where_only_three_states_fit_the_cache(cuda, precision, n, mb, buffer):
    """States of 70-80 MB: three fit the 256 MB cache and four do not, unless
    the tables of small elements (FP32, n = 3) fill it."""
    torch = cuda
    rsz = 4 if precision == capi.F32 else 8
    nx = int((mb * 1e6 / (3 * n * n * rsz)) ** 0.5)
    gm = capi.Mesh(*meshgen.uniform_rect(nx, 0.0, 1.0, nx, 0.0, 1.0))
    w = capi.Wave2D(gm, n, np.ones(gm.n_boundary, dtype=np.int32), precision=precision)
    dt = 0.4 * gm.min_h() / n**2
    u0 = torch.tensor(random_state(w.ndof, 21), dtype=w.torch_dtype, device="cuda")
    a, b = u0.clone(), u0.clone()
    w.rk4(a, dt, 2)
    w.rk4(a, dt, 1)
    free = _free(torch)
    w.rk4(b, dt, 1)
    used = free - _free(torch)
    assert used >= rsz * w.ndof if buffer else used == 0
    a.copy_(u0)
    w.rk4(a, dt, 1)
    assert torch.equal(a, b)


def test_third_buffer_stays_below_a_sixteenth_of_the_free_memory(cuda):
    torch = cuda
    n, nx = 8, 512
    w, dt = _wave(*meshgen.uniform_rect(nx, 0.0, 1.0, nx, 0.0, 1.0), n)
    size = 8 * w.ndof
    x = torch.zeros(w.ndof, dtype=torch.float64, device="cuda")
    w.rk4(x, dt, 2)
    hold = []  # leave about eight states free
    while (left := _free(torch) - 8 * size) > (1 << 28):
        hold.append(torch.empty(min(left, 16 << 30), dtype=torch.uint8, device="cuda"))
    free = _free(torch)
    for _ in range(3):
        w.rk4(x, dt, 1)
    assert free - _free(torch) == 0
    assert float(x.abs().max()) == 0.0
    del hold
    torch.cuda.empty_cache()


def test_odd_steps_captured_with_the_third_buffer(cuda):
    """Odd steps recorded into a graph once the buffer is there: every replay,
    with eager steps of the same handle between them, gives the eager bits."""
    torch = cuda
    w, dt = _wave(*mesh_case("skewed6x5"), 5)
    u0 = torch.tensor(random_state(w.ndof, 9), device="cuda")
    ref = u0.clone()
    for _ in range(3):
        ref.copy_(u0)
        w.rk4(ref, dt, 3)
    other = u0.clone()
    w.rk4(other, dt, 1)
    x = u0.clone()
    torch.cuda.synchronize()
    s = torch.cuda.Stream()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        w.rk4(x, dt, 3)
    for _ in range(4):
        x.copy_(u0)
        g.replay()
        y = u0.clone()
        w.rk4(y, dt, 1)
        torch.cuda.synchronize()
        assert torch.equal(x, ref)
        assert torch.equal(y, other)
