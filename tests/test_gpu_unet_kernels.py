"""The warm start's kernels at the edges of their tiles, against the oracle
(oracle/unet_ref.py): convolutions of 8 and 24 output channels and filter
gradients on rows one off a tile's width, heights one off its rows and few
planes; whole networks on problems whose rows are not multiples of the tiles,
over a window of the problems of a grid."""
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
