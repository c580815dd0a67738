"""Resident-tile passes (include/physis/hip/tile.h: small grids, four sweeps
of a fused pair or two red-black iterations per launch) against the oracle,
bit for bit on both grids: extents below the halo, at and one off the tiles'
edges, on both sides of the tile-size and of the grid-size rule, where
whole-grid pairs take two and four points per lane; odd and even counts; pairs
over a box of the grid and their results per sweep, against numpy."""
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


# (shape, box): the interior, boxes off the grid's origin in tiles of both
# sizes, and one in a grid too large for tiles (z-marching passes)
BOXES = [((18, 10, 10), None), ((70, 40, 30), (21, 58, 9, 31, 5, 24)),
         ((130, 128, 128), None), ((130, 128, 128), (5, 126, 3, 67, 60, 127)),
         ((260, 100, 90), (130, 171, 50, 61, 33, 45))]


@pytest.mark.parametrize("square", [False, True])
@pytest.mark.parametrize("shape,box,counts",
                         [s + ((1, 2, 3, 4, 5),) for s in BOXES] +
                         # more executions than fold at once (256), from an
                         # even and from an odd first pass
                         [BOXES[0] + ((256, 257, 258, 513),)])
def test_reducing_pairs(ps, shape, box, counts, square):
    """Pairs over a box, with a result per sweep: every result, and both
    grids bit for bit."""
    L = ps.load_program("ragged")
    G, N = ps.PSGridPtr, [C.c_int] * 7 + [C.c_float, C.c_void_p, C.c_void_p]
    L.ragged_settle.argtypes = [G, G, G] + N
    L.ragged_settle_square.argtypes = [G, G] + N
    nx, ny, nz = shape
    x0, x1, y0, y1, z0, z1 = box = box or (1, nx - 1, 1, ny - 1, 1, nz - 1)
    rng = np.random.default_rng(nx + x0)
    a, b, c = rng.standard_normal((3, nz, ny, nx)).astype(np.float32)
    w, dtype = np.float32(0.2), np.float64 if square else np.float32
    i = (slice(z0, z1), slice(y0, y1), slice(x0, x1))
    u, want, ends = [a.copy(), b.copy()], [], {}
    for k in range(2 * max(counts)):
        s = u[k % 2]
        v = s[i] + s[z0:z1, y0 - 1:y1 - 1, x0 + 1:x1 + 1] + \
            s[z0:z1, y0 + 1:y1 + 1, x0 - 1:x1 - 1] + \
            s[z0 + 1:z1 + 1, y0:y1, x0:x1] + s[z0 - 1:z1 - 1, y0:y1, x0:x1]
        v = v * w if square else v * w + c[i]
        d = v - s[i]
        want.append(np.sum(d.astype(np.float64) ** 2) if square else d.max())
        u[1 - k % 2][i] = v
        if (k + 1) % 2 == 0 and (k + 1) // 2 in counts:
            ends[(k + 1) // 2] = [x.copy() for x in u]
    grids = [ps.PSGridNew(shape) for _ in range(3)]
    ps.PSGridCopyin(grids[2], c)
    for count in counts:
        print(f"reducing {shape} {box} x {count} square={square}", flush=True)
        for g, x in zip(grids, (a, b)):
            ps.PSGridCopyin(g, x)
        got = np.full((2, count), -1, dtype)
        args = list(box) + [count, w, got[0].ctypes.data, got[1].ctypes.data]
        if square:
            L.ragged_settle_square(*[g.handle for g in grids[:2]], *args)
        else:
            L.ragged_settle(*[g.handle for g in grids], *args)
        for g, x in zip(grids, ends[count]):
            assert np.array_equal(ps.PSGridCopyout(g), x.reshape(-1)), count
        ref = np.array(want[:2 * count], dtype).reshape(count, 2).T
        if square:  # FP64 sums of (at most) this many terms, all positive
            err = np.abs(got - ref)
            assert np.all(err <= d.size * 2.0 ** -53 * ref), \
                (count, np.argwhere(err > d.size * 2.0 ** -53 * ref))
        else:
            assert np.array_equal(got, ref), (count, np.argwhere(got != ref))
    for g in grids:
        ps.PSGridFree(g)
