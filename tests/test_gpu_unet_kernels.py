"""The warm start's kernels at the edges of their tiles, against the oracle
(oracle/unet_ref.py): convolutions of 8 and 24 output channels and filter
gradients on rows one off a tile's width, heights one off its rows and few
planes; whole networks on problems whose rows are not multiples of the tiles,
over a window of the problems of a grid; and the fused passes (network input,
pool, concatenation, gate, head) against the layers they are made of, to the
bit."""
import os
import sys

import numpy as np
import pytest

torch = pytest.importorskip("torch")
sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(
    os.path.abspath(__file__))), "oracle"))
import unet_ref as U  # noqa: E402
from physis_amd.configs import poisson_problem  # noqa: E402

pytestmark = pytest.mark.gpu

# (n, d, h, w, cin, cout): tiles of 16, 32 and 64 positions by 8 and 16 rows
DIMS = [(1, 1, 1, 1, 8, 8), (1, 2, 7, 15, 8, 8), (2, 5, 9, 17, 8, 8),
        (1, 3, 16, 31, 24, 8), (1, 4, 17, 33, 24, 8), (1, 9, 8, 65, 8, 8),
        (1, 2, 15, 17, 8, 24), (1, 5, 17, 63, 8, 24), (3, 2, 3, 16, 16, 8),
        (1, 6, 5, 64, 48, 16), (1, 3, 4, 34, 16, 16)]


@pytest.mark.parametrize("dims", DIMS)
def test_layer(ps, dims):
    from physis_amd.warmstart import (conv_backward_data_host,
                                      conv_backward_filter_host,
                                      conv_forward_host)
    print(f"layer {dims}", flush=True)
    n, d, h, w, cin, cout = dims
    rng = np.random.default_rng(sum(dims))
    x = U.bf16_bits(rng.standard_normal(n * d * h * w * cin))
    dy = U.bf16_bits(rng.standard_normal(n * d * h * w * cout))
    wt = U.bf16_bits(rng.standard_normal(cout * 27 * cin) * 0.2)
    b = rng.standard_normal(cout).astype(np.float32)

    def close(got, ref):  # one BF16 rounding, and FP32 sums in another order
        g, r = U.bf16_float(got), U.bf16_float(ref)
        assert np.all(np.abs(g - r) <= 2.0 ** -7 * np.abs(r) +
                      1e-5 * np.max(np.abs(r)))

    for relu in (False, True):
        close(conv_forward_host(x, wt, b, relu, *dims),
              U.conv_forward(x, wt, b, relu, *dims))
    rdx, rdw, rdb = U.conv_backward(x, dy, wt, *dims)
    close(conv_backward_data_host(dy, wt, *dims), rdx)
    dw, db = conv_backward_filter_host(x, dy, *dims)
    assert np.max(np.abs(dw - rdw)) <= 1e-4 * np.max(np.abs(rdw))
    assert np.max(np.abs(db - rdb)) <= 1e-4 * np.max(np.abs(rdb))


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("shape,problems,first,count",
                         [((16, 16, 16), 3, 1, 2), ((48, 16, 32), 2, 1, 1),
                          ((80, 32, 16), 2, 0, 2), ((32, 48, 16), 3, 2, 1),
                          ((112, 16, 48), 1, 0, 1)])
def test_network(ps, shape, problems, first, count, dtype):
    """Gradient and prediction of problems [first, first + count): bounds as
    for the 32^3 network (tests/test_gpu_unet.py); the other problems of the
    output grid keep their values."""
    from physis_amd.warmstart import UNet
    print(f"network {shape} [{first}, {first + count}) {dtype.__name__}",
          flush=True)
    nx, ny, nzs = shape
    m = nx * ny * nzs
    coefs = poisson_problem(nx, ny, nzs, nbatch=problems, gaussians=(3, 6),
                            sigma=(2.0, 5.0), seed=43)
    rng = np.random.default_rng(8)
    target = (rng.standard_normal(m * problems).astype(np.float32) *
              coefs[10] * 3.0)
    grids = []
    for a in (coefs[11], coefs[10], target):
        grids.append(ps.PSGridNew((nx, ny, nzs * problems)))
        ps.PSGridCopyin(grids[-1], a)
    p = ps.PSGridNew((nx, ny, nzs * problems), dtype)
    ps.PSGridCopyin(p, np.full(m * problems, 7.0, dtype))
    cut = slice(first * m, (first + count) * m)
    net = UNet(nx, ny, nzs, count, 4.0, seed=7)
    try:
        par = net.get_params()
        loss, grad = net.loss_grad(*grids, first, count)
        rloss, rgrad = U.loss_grad(par, coefs[11][cut], coefs[10][cut],
                                   target[cut], shape, count, 4.0)
        err = np.linalg.norm(grad - rgrad) / np.linalg.norm(rgrad)
        print("loss", loss, rloss, "gradient", err, flush=True)
        assert abs(loss - rloss) <= 1.5e-4 * rloss
        assert err <= 1e-2
        # the first layer's unused input channels have no gradient
        w0 = grad[:8 * 27 * 8].reshape(8, 27, 8)
        assert np.all(w0[:, :, 2:] == 0) and np.any(w0[:, :, :2] != 0)
        net.predict(grids[0], grids[1], first, count, p)
        got = ps.PSGridCopyout(p)
        ref = U.predict(par, coefs[11][cut], coefs[10][cut], shape, count, 4.0)
        assert np.linalg.norm(got[cut] - ref) <= 1e-2 * np.linalg.norm(ref)
        assert np.all(got[cut][coefs[10][cut] == 0] == 0)
        assert np.all(np.delete(got, np.arange(m * problems)[cut]) == 7.0)
    finally:
        net.free()
        for g in grids + [p]:
            ps.PSGridFree(g)


def _round(a):
    return U.bf16_float(U.bf16_bits(a)).reshape(a.shape)


def _up(a):
    for axis in (1, 2, 3):
        a = a.repeat(4, axis)
    return a


def _pool(a, wave):
    """4x4x4 means of BF16 values, summed in FP32 one after another, or (wave)
    as the first pool sums: planes, then pairs of columns, then of rows."""
    n, d, h, w, c = a.shape
    a = a.reshape(n, d // 4, 4, h // 4, 4, w // 4, 4, c)
    if wave:
        s = ((a[:, :, 0] + a[:, :, 1]) + a[:, :, 2]) + a[:, :, 3]
        s = (s[..., 0, :] + s[..., 1, :]) + (s[..., 2, :] + s[..., 3, :])
        s = (s[:, :, :, 0] + s[:, :, :, 1]) + (s[:, :, :, 2] + s[:, :, :, 3])
    else:
        s = np.zeros((n, d // 4, h // 4, w // 4, c), np.float32)
        for z in range(4):
            for y in range(4):
                for x in range(4):
                    s += a[:, :, z, :, y, :, x]
    return _round(s * np.float32(1 / 64))


@pytest.mark.parametrize("shape,batch", [((16, 16, 16), 2), ((48, 32, 16), 1),
                                         ((80, 16, 32), 1)])
def test_network_is_its_layers(ps, shape, batch):
    """The prediction, and the gradients of the last two layers, are to the
    bit what the layers give one after another on whole 8-channel tensors:
    the network input as a tensor of 8 channels, pools, upsampling,
    concatenation, gate and head in numpy."""
    from physis_amd.warmstart import (UNet, conv_backward_data_host,
                                      conv_backward_filter_host,
                                      conv_forward_host)
    print(f"layers of {shape} x {batch}", flush=True)
    nx, ny, nzs = shape
    m = nx * ny * nzs * batch
    coefs = poisson_problem(nx, ny, nzs, nbatch=batch, gaussians=(3, 6),
                            sigma=(2.0, 5.0), seed=11)
    rhs, bnd = coefs[11].reshape(-1), coefs[10].reshape(-1)
    target = (np.random.default_rng(3).standard_normal(m) * bnd) \
        .astype(np.float32)
    grids = []
    for a in (rhs, bnd, target):
        grids.append(ps.PSGridNew((nx, ny, nzs * batch)))
        ps.PSGridCopyin(grids[-1], a)
    p = ps.PSGridNew((nx, ny, nzs * batch), np.float64)
    scale = np.float32(4.0)
    net = UNet(nx, ny, nzs, batch, float(scale), seed=5)
    try:
        par = net.get_params()
        _, grad = net.loss_grad(*grids, 0, batch)
        net.predict(grids[0], grids[1], 0, batch, p)
        got = ps.PSGridCopyout(p)
    finally:
        net.free()
        for g in grids + [p]:
            ps.PSGridFree(g)
    off, layers = 0, []
    for ci, co in ((8, 8), (8, 8), (8, 16), (16, 16), (16, 32), (32, 32),
                   (48, 16), (16, 16), (24, 8), (8, 8)):
        k = co * 27 * ci
        layers.append((ci, co, U.bf16_bits(par[off:off + k]),
                       par[off + k:off + k + co],
                       slice(off, off + k), slice(off + k, off + k + co)))
        off += k + co
    head = par[off:off + 9]

    def conv(l, a):
        ci, co, w, b = layers[l][:4]
        y = conv_forward_host(U.bf16_bits(a.reshape(-1)), w, b, True,
                              *a.shape[:4], ci, co)
        return U.bf16_float(y).reshape(a.shape[:4] + (co,))

    x = np.zeros((batch, nzs, ny, nx, 8), np.float32)
    x[..., 0] = _round(rhs).reshape(x.shape[:4])
    x[..., 1] = _round(bnd).reshape(x.shape[:4])
    a1 = conv(1, conv(0, x))
    a3 = conv(3, conv(2, _pool(a1, True)))
    a5 = conv(5, conv(4, _pool(a3, False)))
    a7 = conv(7, conv(6, np.concatenate([_up(a5), a3], 4)))
    c1 = np.concatenate([_up(a7), a1], 4)
    a8 = conv(8, c1)
    a9 = conv(9, a8)
    out = np.zeros(a9.shape[:4], np.float32)
    for c in range(8):
        out += head[c] * a9[..., c]
    out = (out + head[8]).reshape(-1)
    assert np.array_equal(got, (scale * out).astype(np.float64) * bnd)
    # the head's gradient, through the gates of the last two layers
    g = np.float32(2.0) * (out - target * (np.float32(1) / scale)) / \
        np.float32(m)
    dz = _round(np.where(a9 > 0, head[:8] * g.reshape(a9.shape[:4] + (1,)),
                         np.float32(0)))
    for l, below in ((9, a8), (8, c1)):
        ci, co, w, _, ws, bs = layers[l]
        dims = below.shape[:4] + (ci, co)
        bits = U.bf16_bits(dz.reshape(-1))
        dw, db = conv_backward_filter_host(U.bf16_bits(below.reshape(-1)),
                                           bits, *dims)
        assert np.array_equal(grad[ws], dw) and np.array_equal(grad[bs], db)
        if l == 9:
            dx = U.bf16_float(conv_backward_data_host(bits, w, *dims))
            dz = np.where(below > 0, dx.reshape(below.shape), np.float32(0))


def test_planes_of_more_than_2_gib(ps):
    """Positions outside a plane of more than 2 GiB are zeros like any others:
    convolutions and filter gradients of ones count the taps inside."""
    from physis_amd.warmstart import (conv_backward_filter_host,
                                      conv_forward_host)
    one = np.uint16(0x3f80)
    h, w, cin, cout = 6800, 6700, 24, 8
    print(f"forward {h} x {w} x {cin}", flush=True)
    assert h * w * cin * 2 > 2 ** 31
    y = conv_forward_host(np.full(h * w * cin, one),
                          U.bf16_bits(np.full(cout * 27 * cin, 1 / 256)),
                          np.zeros(cout, np.float32), True, 1, 1, h, w, cin,
                          cout).reshape(h, w, cout)
    rows = np.full(h, 3)
    rows[[0, -1]] = 2
    cols = np.full(w, 3)
    cols[[0, -1]] = 2
    want = U.bf16_bits(rows[:, None] * cols[None, :] * (cin / 256)) \
        .reshape(h, w)
    assert all(np.array_equal(y[:, :, c], want) for c in range(cout))
    h, w, cin, cout = 4800, 4700, 16, 48
    print(f"filter gradient {h} x {w} x {cout}", flush=True)
    assert h * w * cout * 2 > 2 ** 31
    dw, db = conv_backward_filter_host(np.full(h * w * cin, one),
                                       np.full(h * w * cout, one),
                                       1, 1, h, w, cin, cout)
    k = np.array([h - 1, h, h - 1], np.float64)[:, None] * \
        np.array([w - 1, w, w - 1])[None, :]
    ref = np.zeros((3, 3, 3))
    ref[1] = k  # one plane: no taps in z
    dw = dw.reshape(cout, 27, cin)
    # FP32 sums of whole numbers: exact below 2^24, then half a unit each for
    # the last few additions
    assert np.all(np.abs(dw - ref.reshape(1, 27, 1)) <= 1e-6 * h * w)
    assert np.all(np.abs(db - h * w) <= 1e-6 * h * w)


def test_infinite_input_reaches_its_taps_only(ps):
    """8 -> 24 channels: results that no tap leads to stay finite."""
    from physis_amd.warmstart import conv_forward_host
    n, d, h, w, cin, cout = dims = (1, 5, 9, 40, 8, 24)
    rng = np.random.default_rng(2)
    x = rng.standard_normal((d, h, w, cin)).astype(np.float32)
    wt = U.bf16_bits(rng.standard_normal(cout * 27 * cin))
    for at in ((2, 4, 20), (2, 5, 31), (0, 0, 0), (4, 8, 39)):
        print(f"infinite at {at}", flush=True)
        xi = x.copy()
        xi[at + (3,)] = np.inf
        y = U.bf16_float(conv_forward_host(
            U.bf16_bits(xi.reshape(-1)), wt, np.zeros(cout, np.float32), False,
            *dims)).reshape(d, h, w, cout)
        near = np.zeros((d, h, w), bool)
        near[tuple(slice(max(c - 1, 0), c + 2) for c in at)] = True
        assert np.all(np.isfinite(y).all(3) == ~near)
