"""Resident-tile passes (include/physis/hip/tile.h: small grids, four sweeps
of a fused pair or two red-black iterations per launch) against the oracle,
bit for bit on both grids: extents below the halo, at and one off the tiles'
edges, on both sides of the tile-size and of the grid-size rule, where
whole-grid pairs take two and four points per lane; odd and even counts."""
import ctypes as C

import numpy as np
import pytest

from oracle_lib import lib

pytestmark = pytest.mark.gpu

COEF = (0.11, 0.09, 0.12, 0.08, 0.105, 0.095, 0.39)
SHAPES = [(1, 2, 1), (2, 3, 1), (3, 3, 3), (5, 4, 6), (15, 7, 7), (16, 8, 8),
          (17, 9, 9), (33, 17, 12), (64, 64, 64), (65, 64, 64), (96, 40, 70),
          (130, 130, 130), (131, 130, 130),
          # thin grids in tiles, and pairs at two points per lane
          (16, 300, 290), (47, 260, 181), (121, 120, 123), (127, 153, 139),
          (257, 90, 101), (383, 70, 122), (385, 70, 122)]


def _bits(a):
    return a.view(np.uint32)


@pytest.mark.parametrize("periodic", [False, True])
@pytest.mark.parametrize("shape", SHAPES)
def test_pairs(ps, shape, periodic):
    from physis_amd.programs import Diffusion7
    d7 = Diffusion7()
    a = np.random.default_rng(sum(shape)).random(int(np.prod(shape))) \
        .astype(np.float32)
    g1, g2 = ps.PSGridNew(shape), ps.PSGridNew(shape)
    for pairs in (2, 3, 4, 5):
        print(f"pairs {shape} periodic={periodic} x {pairs}", flush=True)
        ps.PSGridCopyin(g1, a)
        ps.PSGridCopyin(g2, a)
        d7.run(g1, g2, 2 * pairs, COEF, periodic=periodic)
        o1, o2 = a.copy(), a.copy()
        lib().oracle_diffusion7_run_omp(o1, o2, *shape, 2 * pairs,
                                        int(periodic), *COEF, 8)
        assert np.array_equal(_bits(ps.PSGridCopyout(g1)), _bits(o1)), pairs
        assert np.array_equal(_bits(ps.PSGridCopyout(g2)), _bits(o2)), pairs
    ps.PSGridFree(g1)
    ps.PSGridFree(g2)


@pytest.mark.parametrize("shape", [s for s in SHAPES if min(s) > 2])
def test_red_black(ps, shape):
    from physis_amd.programs import RedBlack7
    rb = RedBlack7()
    nx, ny, nz = shape
    a = np.random.default_rng(nx).random(nx * ny * nz).astype(np.float32)
    g = ps.PSGridNew(shape)
    for count in (1, 2, 3, 4, 5):
        print(f"red-black {shape} x {count}", flush=True)
        ps.PSGridCopyin(g, a)
        rb.run(g, count, COEF)
        o = a.copy()
        lib().oracle_redblack7_run(o, nx, ny, nz, count,
                                   np.array(COEF, np.float32))
        assert np.array_equal(_bits(ps.PSGridCopyout(g)), _bits(o)), count
    ps.PSGridFree(g)


@pytest.mark.parametrize("shape", [(3, 3, 3), (18, 10, 10), (19, 11, 9),
                                   (67, 66, 66), (131, 30, 40)])
def test_interior_pairs(ps, shape):
    """Pairs over the interior: points outside it alternate between the two
    grids' own values."""
    L = ps.load_program("ragged")
    L.ragged_inner.argtypes = [ps.PSGridPtr, ps.PSGridPtr, C.c_int, C.c_float]
    nx, ny, nz = shape
    rng = np.random.default_rng(nx)
    a, b = rng.standard_normal((2, nz, ny, nx)).astype(np.float32)
    w = np.float32(0.2)
    g, g2 = ps.PSGridNew(shape), ps.PSGridNew(shape)
    for count in (2, 3, 4, 5):
        print(f"interior {shape} x {count}", flush=True)
        ps.PSGridCopyin(g, a)
        ps.PSGridCopyin(g2, b)
        L.ragged_inner(g.handle, g2.handle, count, w)
        u = [a.copy(), b.copy()]
        i = (slice(1, -1),) * 3
        for k in range(2 * count):
            s = u[k % 2]
            v = s[i] + s[1:-1, :-2, 2:] + s[1:-1, 2:, :-2] + \
                s[2:, 1:-1, 1:-1] + s[:-2, 1:-1, 1:-1]
            u[1 - k % 2][i] = v * w
        assert np.array_equal(ps.PSGridCopyout(g), u[0].reshape(-1)), count
        assert np.array_equal(ps.PSGridCopyout(g2), u[1].reshape(-1)), count
    ps.PSGridFree(g)
    ps.PSGridFree(g2)
