"""The warm-start network's HIP kernels against the CPU oracle
(oracle/cnn_oracle.py): forward pass, loss, every parameter gradient, the
Adam update, determinism, and the DG <-> image maps.

The oracle runs in float64 with bf16 rounding at the points where the GPU
stores bf16; the remaining differences come from float32 accumulation order
and from the rare value that lands on the other side of a bf16 rounding
boundary, hence the tolerances below (1e-3 for the forward pass, 2e-2 per
layer gradient, 1e-2 overall)."""
from __future__ import annotations

import numpy as np
import pytest

from oracle import cnn_oracle as co
from wavedg_amd import capi

pytestmark = pytest.mark.gpu


def _rel(a, b):
    return float(np.linalg.norm(np.ravel(a) - np.ravel(b)) / max(np.linalg.norm(np.ravel(b)), 1e-300))


def _setup(torch, M=16, base=16, in_ld=32, out_ch=75, B=3, seed=0):
    net = capi.CNN(M, in_ld, out_ch, base, max_batch=B)
    p = co.init_params(in_ld, out_ch, base, seed=seed)
    net.set_params(p)
    rng = np.random.default_rng(seed + 1)
    x = co.bf16(rng.standard_normal((B, M, M, in_ld)))
    t = rng.standard_normal((B, M, M, net.out_ld)).astype(np.float32).astype(np.float64)
    t[..., out_ch:] = 0.0
    xd = torch.tensor(x, dtype=torch.float32, device="cuda").to(torch.bfloat16).contiguous()
    td = torch.tensor(t, dtype=torch.float32, device="cuda").contiguous()
    return net, p, x, t, xd, td


@pytest.mark.parametrize("M,base,B", [(16, 16, 3), (8, 32, 2)])
def test_forward_matches_oracle(cuda, M, base, B):
    torch = cuda
    print(f"cnn forward M={M} base={base} B={B}", flush=True)
    net, p, x, t, xd, td = _setup(torch, M=M, base=base, B=B)
    y = torch.empty((B, M, M, net.out_ld), dtype=torch.float32, device="cuda")
    net.forward(xd, y)
    torch.cuda.synchronize()
    yg = y.cpu().numpy().astype(np.float64)
    ye = co.Net(p, net.in_ld, 75, base, emulate_bf16=True).forward(x)
    y64 = co.Net(p, net.in_ld, 75, base).forward(x)
    assert _rel(yg[..., :75], ye[..., :75]) < 1e-3
    assert _rel(yg[..., :75], y64[..., :75]) < 3e-2


@pytest.mark.parametrize("M,base,B", [(16, 16, 3), (8, 32, 2)])
def test_gradient_matches_oracle(cuda, M, base, B):
    torch = cuda
    print(f"cnn gradient M={M} base={base} B={B}", flush=True)
    net, p, x, t, xd, td = _setup(torch, M=M, base=base, B=B, seed=4)
    loss, g = net.loss_grad(xd, td)
    onet = co.Net(p, net.in_ld, 75, base, emulate_bf16=True)
    lo, go = onet.loss_grad(x, t)
    assert abs(loss - lo) < 1e-3 * lo
    g = g.astype(np.float64)
    for name, wo, bo, shp in onet.layout:
        sl = slice(wo, bo + shp[1])
        assert _rel(g[sl], go[sl]) < 2e-2, name
    assert _rel(g, go) < 1e-2
    # bitwise reproducible
    loss2, g2 = net.loss_grad(xd, td)
    assert loss2 == loss and np.array_equal(g2, g.astype(np.float32))


def test_adam_first_step(cuda):
    torch = cuda
    net, p, x, t, xd, td = _setup(torch, M=8, base=16, B=2, seed=7)
    _, g = net.loss_grad(xd, td)
    lr = 1e-3
    net.train_step(xd, td, lr)
    p1 = net.get_params()
    # first Adam step: m_hat = g, v_hat = g^2
    g64 = g.astype(np.float64)
    expect = p.astype(np.float64) - lr * g64 / (np.abs(g64) + 1e-8)
    np.testing.assert_allclose(p1, expect, rtol=1e-5, atol=1e-7)


def test_training_fits_teacher(cuda):
    """The student (own forward/backward/Adam on the GPU) fits the outputs of a
    fixed random teacher network of the same shape."""
    torch = cuda
    M, base, B, in_ld, out_ch = 16, 16, 4, 32, 75
    teacher = co.Net(co.init_params(in_ld, out_ch, base, seed=11), in_ld, out_ch, base)
    rng = np.random.default_rng(12)
    x = co.bf16(rng.standard_normal((B, M, M, in_ld)))
    t = teacher.forward(x).astype(np.float32)
    net = capi.CNN(M, in_ld, out_ch, base, max_batch=B)
    net.set_params(co.init_params(in_ld, out_ch, base, seed=13))
    xd = torch.tensor(x, dtype=torch.float32, device="cuda").to(torch.bfloat16).contiguous()
    td = torch.tensor(t, device="cuda").contiguous()
    first = net.train_step(xd, td, 2e-3)
    for _ in range(150):
        last = net.train_step(xd, td, 2e-3)
    print(f"teacher fit: loss {first:.4f} -> {last:.4f}", flush=True)
    assert last < 0.3 * first


def test_dg_image_maps(cuda):
    torch = cuda
    M, n = 8, 5
    mesh = capi.Mesh.uniform_rect(M, 0.0, 1.0, M, 0.0, 1.0)
    nodes = mesh.nodes(n)
    src = np.array([[0.3, 0.6, 0.05, 1.5], [0.7, 0.2, 0.02, -0.7]])
    ld = 32
    xd = torch.empty((M * M, ld), dtype=torch.bfloat16, device="cuda")
    nd = torch.tensor(nodes.reshape(-1), device="cuda")
    sd = torch.tensor(src.reshape(-1), device="cuda")
    capi.ws_features(nd, n, M * M, sd, 2, 0.37, 0.0, -0.25, 0.0, (0.0, 0.0, 1.0, 1.0), ld, xd)
    torch.cuda.synchronize()
    got = xd.float().cpu().numpy().astype(np.float64)
    want = co.bf16(co.features(nodes, n, src, 0.37, -0.25, (0.0, 0.0, 1.0, 1.0), ld))
    # equal up to one bf16 ulp where exp() rounds differently
    assert np.all(np.abs(got - want) <= 2.0 ** -7 * np.abs(want) + 1e-30)
    # pixel e is element e: element centres follow the uniform-rectangle numbering
    ex, ey = np.arange(M * M) % M, np.arange(M * M) // M
    np.testing.assert_allclose(got[:, n * n + 1], co.bf16(2 * (ex + 0.5) / M - 1), atol=0)
    np.testing.assert_allclose(got[:, n * n + 2], co.bf16(2 * (ey + 0.5) / M - 1), atol=0)
    # with the free-space Green's-function channels
    ld2 = 80
    xg = torch.empty((M * M, ld2), dtype=torch.bfloat16, device="cuda")
    capi.ws_features(nd, n, M * M, sd, 2, 0.37, 40.0, 0.5, 3.0, (0.0, 0.0, 1.0, 1.0), ld2, xg)
    torch.cuda.synchronize()
    got = xg.float().cpu().numpy().astype(np.float64)
    want = co.bf16(co.features(nodes, n, src, 0.37, 0.5, (0.0, 0.0, 1.0, 1.0), ld2, omega=40.0, green_gain=3.0))
    assert np.all(np.abs(got - want) <= 2.0 ** -7 * np.abs(want) + 1e-6)
    # DG <-> image round trip
    nd3 = 3 * n * n
    W = torch.randn(M * M * nd3, dtype=torch.float64, device="cuda")
    img = torch.empty((M * M, 80), dtype=torch.float32, device="cuda")
    capi.ws_dg_to_image(W, n, M * M, 2.5, 80, img)
    W2 = torch.empty_like(W)
    capi.ws_image_to_dg(img, 80, n, M * M, 2.5, W2)
    torch.cuda.synchronize()
    assert torch.all(img[:, nd3:] == 0)
    np.testing.assert_allclose(img[:, :nd3].cpu().numpy().reshape(-1), (W.cpu().numpy() / 2.5).astype(np.float32))
    assert float(torch.linalg.norm(W2 - W) / torch.linalg.norm(W)) < 1e-7


@pytest.mark.parametrize("ns", [0, 1, 32, 33, 70])
def test_features_of_many_sources(cuda, ns):
    """Sources are staged 32 at a time, also by the idle threads of the last
    workgroup (35 elements of 9 nodes are 315 threads)."""
    torch = cuda
    n, ld = 3, 32
    mesh = capi.Mesh.uniform_rect(7, 0.0, 1.0, 5, 0.0, 1.0)
    nodes = mesh.nodes(n)
    r = np.random.default_rng(ns)
    src = np.column_stack([r.uniform(0.0, 1.0, (ns, 2)), r.uniform(0.05, 0.3, ns), r.uniform(0.5, 1.5, ns)])
    sd = torch.tensor(src.reshape(-1), device="cuda")
    xd = torch.full((35, ld), 5.0, dtype=torch.bfloat16, device="cuda")
    box = (0.0, 0.0, 1.0, 1.0)
    capi.ws_features(torch.tensor(nodes.reshape(-1), device="cuda"), n, 35, sd, ns, 0.7, 9.0, 0.5, 0.3, box, ld, xd)
    torch.cuda.synchronize()
    got = xd.float().cpu().numpy().astype(np.float64)
    want = co.bf16(co.features(nodes, n, src, 0.7, 0.5, box, ld, omega=9.0, green_gain=0.3))
    # one bf16 step where the Bessel polynomials (1e-7 each) round differently
    assert np.all(np.abs(got - want) <= 2.0 ** -7 * np.abs(want) + 1e-6)


def test_features_round_through_float(cuda):
    """A feature is the bf16 of the float of its double (as the oracle rounds).
    At a source's own node the forcing is gain * amp: a double just above the
    float that lies halfway between two bf16 values goes to the even one, and
    so does one just below it."""
    torch = cuda
    M, n, ld = 2, 3, 16
    mesh = capi.Mesh.uniform_rect(M, 0.0, 1.0, M, 0.0, 1.0)
    nodes = mesh.nodes(n)
    nd = torch.tensor(nodes.reshape(-1), device="cuda")
    x0, y0 = np.asarray(nodes).reshape(-1, 2)[0]
    sd = torch.tensor([x0, y0, 0.05, 1.0], dtype=torch.float64, device="cuda")
    xd = torch.empty((M * M, ld), dtype=torch.bfloat16, device="cuda")
    for half, even in ((1.0 + 2.0 ** -8, 1.0), (1.0 + 3 * 2.0 ** -8, 1.0 + 2.0 ** -6)):
        for off in (-(2.0 ** -40), 0.0, 2.0 ** -40):
            capi.ws_features(nd, n, M * M, sd, 1, half + off, 0.0, 0.0, 0.0, (0.0, 0.0, 1.0, 1.0), ld, xd)
            torch.cuda.synchronize()
            assert float(xd[0, 0]) == even, (half, off)


@pytest.mark.parametrize("M,B", [(128, 16), (32, 128), (32, 256)])
def test_convolution_tiles_agree(cuda, M, B):
    """Tiles of conv3_row_kernel against its smallest, which one image alone
    takes everywhere.  16 images of 128^2 run the widths 128, 64, 32 and 16 on
    512, 256, 128 and 64 pixels (backward-data also on 256 at width 32); 128
    and 256 images of 32^2 reach the taller tiles of the widths 32 and 16: 512
    at 32, 256 and 128 at 16.  The tiles add in the same order, so outputs are
    equal bit for bit; the batch gradient is the mean of the single ones up to
    the order of its float32 sums (the loss gradient is scaled by a power of
    two, exactly)."""
    torch = cuda
    net, p, x, t, xd, td = _setup(torch, M=M, base=32, in_ld=48, B=B, seed=21)
    y = torch.empty((B, M, M, net.out_ld), dtype=torch.float32, device="cuda")
    net.forward(xd, y)
    loss, g = net.loss_grad(xd, td)
    one = torch.empty((1, M, M, net.out_ld), dtype=torch.float32, device="cuda")
    mean, losses = np.zeros(net.n_params), []
    for k in range(B):
        net.forward(xd[k:k + 1], one)
        assert torch.equal(one[0], y[k]), k
        lk, gk = net.loss_grad(xd[k:k + 1], td[k:k + 1])
        losses.append(lk)
        mean += gk.astype(np.float64) / B
    assert abs(loss - np.mean(losses)) < 1e-6 * loss
    # float32 partial sums over at most 2^18 pixels in chunks: below 2^-24 * 2^7
    assert _rel(g, mean) < 1e-5


@pytest.mark.parametrize("M,base,B", [(128, 32, 9), (128, 64, 3), (64, 32, 13)])
def test_weight_gradient_of_an_odd_number_of_strips(cuda, M, base, B):
    """wgrad3_row_kernel<4, 16> takes two 16-pixel images per tile; an odd
    batch leaves the last tile with one, whose missing partner reads as zeros.
    The batch against itself twice over, which fills every tile: the mean loss
    and so each layer's gradient are the same (the loss gradient is halved,
    exactly) up to the order of the float32 sums, layer by layer."""
    torch = cuda
    H, L = 16, {128: 3, 64: 2}[M]
    cin, cout = {3: (8 * base, 8 * base), 2: (12 * base, 4 * base)}[L]
    assert M >> L == H and B % 2 == 1
    assert B * H * H // 512 * (cout // 32) * (cin // 32) >= 256, "the rule must choose the taller tile"
    net, p, x, t, xd, td = _setup(torch, M=M, base=base, in_ld=48, B=2 * B, seed=33)
    x2, t2 = torch.cat([xd[:B], xd[:B]]), torch.cat([td[:B], td[:B]])
    l1, g1 = net.loss_grad(xd[:B], td[:B])
    l2, g2 = net.loss_grad(x2, t2)
    assert abs(l1 - l2) < 1e-6 * l1
    for name, wo, bo, shp in co.Net(p, net.in_ld, 75, base).layout:
        sl = slice(wo, bo + shp[1])
        err = _rel(g1[sl], g2[sl].astype(np.float64))
        print(f"  {name}: {err:.2e}", flush=True)
        assert err < 1e-5, name  # below 2^-24 * 2^7, as above


@pytest.mark.parametrize("M,B,want", [(32, 2, 1.6441795826), (64, 1, 1.74118685722), (128, 2, 1.79015147686)])
def test_convolution_sums_in_tap_order(cuda, M, B, want):
    """Outputs add their slices and taps in one order at every width, that of
    conv3_k32_kernel, so a network's outputs do not move with the kernel that
    a layer takes.  The losses are those of a build that ran that kernel at
    every width; another order puts some values on the other side of a bf16
    boundary and moves them by 3e-7 to 4e-5, against the 11 digits given."""
    net, p, x, t, xd, td = _setup(cuda, M=M, base=32, in_ld=48, B=B, seed=9)
    loss, _ = net.loss_grad(xd, td)
    assert loss == pytest.approx(want, rel=2e-10)


def test_row_convolution_matches_oracle(cuda):
    """conv3_row_kernel at widths 32 and 16 (conv3_k32_kernel at 8 and 4), with
    a last slice of 16 input channels, against the oracle."""
    torch = cuda
    M, base, B = 32, 32, 1
    net, p, x, t, xd, td = _setup(torch, M=M, base=base, in_ld=48, B=B, seed=9)
    y = torch.empty((B, M, M, net.out_ld), dtype=torch.float32, device="cuda")
    net.forward(xd, y)
    loss, g = net.loss_grad(xd, td)
    onet = co.Net(p, net.in_ld, 75, base, emulate_bf16=True)
    # float32 sums in another order land a few values of every layer on the
    # other side of a bf16 boundary; fifteen layers of such flips stay below
    # the effect of all bf16 roundings, which the unrounded network shows
    ye, y64 = onet.forward(x)[..., :75], co.Net(p, net.in_ld, 75, base).forward(x)[..., :75]
    noise = _rel(ye, y64)
    assert noise < 1e-2
    yg = y.cpu().numpy()[..., :75]
    assert _rel(yg, ye) < noise and _rel(yg, y64) < 1.2 * noise
    lo, go = onet.loss_grad(x, t)
    assert abs(loss - lo) < 1e-3 * lo
    assert _rel(g, go) < 2e-2
