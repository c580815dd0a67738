"""Run kernels on rows whose extents are not multiples of the vector width
(tests/programs/ragged.c), bit for bit against numpy: the points past the
end of a row (the next row's, 0 outside the grid, the wrapped ones of a
periodic get) at the sizes where a lane's vector hangs over a row's end, a
tile's end or the grid's end; and pairs over boxes anywhere in a grid."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPES = [(1, 3, 4), (3, 5, 4), (5, 1, 3), (6, 7, 2), (63, 4, 5), (65, 17, 3),
          (255, 3, 4), (257, 16, 9), (258, 5, 3), (511, 4, 3), (64, 9, 4)]


@pytest.fixture(scope="module")
def prog(ps):
    L = ps.load_program("ragged")
    G = ps.PSGridPtr
    for f in ("corners", "corners_double", "corners2d", "wrap2"):
        getattr(L, "ragged_" + f).argtypes = [G, G]
    L.ragged_inner.argtypes = [G, G, C.c_int, C.c_float]
    L.ragged_box.argtypes = [G, G] + [C.c_int] * 7 + [C.c_float]
    L.ragged_box2d.argtypes = [G, G] + [C.c_int] * 5 + [C.c_float]
    return L


def _run(ps, fn, a, shape2=None, b=None):
    """Grids with a and b (zeros) in, fn(g, g2), both grids out."""
    dims = a.shape[::-1]
    g = ps.PSGridNew(dims, a.dtype)
    g2 = ps.PSGridNew((shape2 or dims), a.dtype)
    ps.PSGridCopyin(g, a)
    if b is not None:
        ps.PSGridCopyin(g2, b)
    fn(g.handle, g2.handle)
    out = [ps.PSGridCopyout(x) for x in (g, g2)]
    ps.PSGridFree(g)
    ps.PSGridFree(g2)
    return out


def _linear(a, x, y, z, d):
    """Element at the linear offset of (x, y, z) + d, 0 outside the grid."""
    nz, ny, nx = a.shape
    off = x + d[0] + (y + d[1]) * nx + (z + d[2]) * nx * ny
    ok = (off >= 0) & (off < a.size)
    return np.where(ok, a.reshape(-1)[np.clip(off, 0, a.size - 1)],
                    a.dtype.type(0))


def _sum(get, terms, t):
    v = None
    for w, d in terms:
        p = get(d) if w is None else t(w) * get(d)
        v = p if v is None else v + p
    return v


CORNERS = [(0.5, (0, 0, 0)), (None, (1, 0, 0)), (2.0, (1, -1, 0)),
           (3.0, (-1, 1, 0)), (4.0, (1, 1, 1)), (5.0, (-1, -1, -1)),
           (6.0, (1, 0, -1))]


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("shape", SHAPES)
def test_rows_past_their_ends(ps, prog, shape, dtype):
    print(f"corners {shape} {dtype.__name__}", flush=True)
    nx, ny, nz = shape
    a = np.random.default_rng(nx).standard_normal((nz, ny, nx)).astype(dtype)
    fn = prog.ragged_corners if dtype == np.float32 else \
        prog.ragged_corners_double
    got = _run(ps, fn, a)[1]
    z, y, x = np.meshgrid(*map(np.arange, (nz, ny, nx)), indexing="ij")
    want = _sum(lambda d: _linear(a, x, y, z, d), CORNERS, dtype)
    assert np.array_equal(got, want.reshape(-1))


@pytest.mark.parametrize("shape,shape2", [((5, 4, 3), (9, 3, 3)),
                                          ((61, 5, 4), (67, 5, 3))])
def test_domain_wider_than_the_grid_read(ps, prog, shape, shape2):
    """The map covers g2, whose rows are longer than those it reads."""
    print(f"corners {shape} -> {shape2}", flush=True)
    nx, ny, nz = shape
    a = np.random.default_rng(nx).standard_normal((nz, ny, nx)) \
        .astype(np.float32)
    got = _run(ps, prog.ragged_corners, a, shape2)[1]
    z, y, x = np.meshgrid(*map(np.arange, shape2[::-1]), indexing="ij")
    want = _sum(lambda d: _linear(a, x, y, z, d), CORNERS, np.float32)
    assert np.array_equal(got, want.reshape(-1))


@pytest.mark.parametrize("shape", [(3, 4), (5, 1), (63, 7), (257, 9),
                                   (1023, 5)])
def test_two_dimensional_rows(ps, prog, shape):
    print(f"corners2d {shape}", flush=True)
    nx, ny = shape
    a = np.random.default_rng(nx).standard_normal((ny, nx)).astype(np.float32)
    got = _run(ps, prog.ragged_corners2d, a)[1]
    y, x = np.meshgrid(np.arange(ny), np.arange(nx), indexing="ij")
    want = _sum(lambda d: _linear(a[None], x, y, 0 * x, d),
                [(0.5, (0, 0, 0)), (2.0, (1, -1, 0)), (3.0, (-1, 1, 0)),
                 (4.0, (1, 0, 0))], np.float32)
    assert np.array_equal(got, want.reshape(-1))


@pytest.mark.parametrize("shape", SHAPES)
def test_periodic_rows(ps, prog, shape):
    print(f"wrap2 {shape}", flush=True)
    nx, ny, nz = shape
    a = np.random.default_rng(nx).standard_normal((nz, ny, nx)) \
        .astype(np.float32)
    got = _run(ps, prog.ragged_wrap2, a)[1]
    want = _sum(lambda d: np.roll(a, (-d[2], -d[1], -d[0]), (0, 1, 2)),
                [(0.5, (0, 0, 0)), (2.0, (2, -1, 0)), (3.0, (-2, 1, 0)),
                 (4.0, (1, 0, 1)), (5.0, (-1, 0, -1))], np.float32)
    assert np.array_equal(got, want.reshape(-1))


@pytest.mark.parametrize("count", [1, 2, 3])
@pytest.mark.parametrize("shape", [(3, 3, 3), (7, 5, 4), (65, 18, 6),
                                   (257, 14, 5), (259, 30, 4), (64, 9, 5)])
def test_interior_pairs(ps, prog, shape, count):
    """Pairs over the interior: both grids as single sweeps leave them."""
    print(f"inner {shape} x {count}", flush=True)
    nx, ny, nz = shape
    rng = np.random.default_rng(nx)
    a, b = rng.standard_normal((2, nz, ny, nx)).astype(np.float32)
    w = np.float32(0.2)
    got = _run(ps, lambda g, g2: prog.ragged_inner(g, g2, count, w), a, None,
               b)
    z, y, x = np.meshgrid(*(np.arange(1, n - 1) for n in (nz, ny, nx)),
                          indexing="ij")
    u = [a.copy(), b.copy()]
    for k in range(2 * count):
        v = _sum(lambda d: u[k % 2][z + d[2], y + d[1], x + d[0]],
                 [(None, (0, 0, 0)), (None, (1, -1, 0)), (None, (-1, 1, 0)),
                  (None, (0, 0, 1)), (None, (0, 0, -1))], np.float32)
        u[1 - k % 2][1:-1, 1:-1, 1:-1] = v * w
    for k in range(2):
        assert np.array_equal(got[k], u[k].reshape(-1)), k


# In 2-D: rows passes whose first column tile is not the grid's, boxes that
# begin and end inside a lane's four points or cross a column tile (248
# points), thin and single-point ones.  In 3-D: resident tiles of both sizes,
# z-marching passes in a grid too large for them, a box crossing x tiles.
BOXES = [((300, 40), (1, 299, 1, 39)), ((301, 40), (5, 9, 3, 36)),
         ((700, 90), (301, 650, 17, 80)), ((520, 300), (242, 262, 1, 299)),
         ((64, 1000), (3, 61, 400, 410)), ((9, 9), (4, 5, 4, 5)),
         ((30, 20, 25), (7, 12, 2, 19, 11, 24)),
         ((97, 90, 80), (30, 96, 20, 81, 1, 79)),
         ((300, 90, 90), (250, 270, 30, 50, 7, 9)),
         ((515, 140, 60), (3, 512, 2, 137, 1, 59)),
         ((40, 9, 9), (20, 21, 4, 5, 4, 5))]


@pytest.mark.parametrize("shape,box", BOXES)
def test_pairs_over_a_box(ps, prog, shape, box):
    """1 to 7 pairs (odd and even counts of passes), both grids.  The passes'
    scratch grids hold NaN from a run over such grids before."""
    dims = len(shape)
    run = prog.ragged_box if dims == 3 else prog.ragged_box2d
    rng = np.random.default_rng(sum(shape))
    a, b = rng.standard_normal((2,) + shape[::-1]).astype(np.float32)
    w = np.float32(0.2)
    offsets = [(0, 0, 0), (1, -1, 0), (-1, 1, 0), (0, 0, 1), (0, 0, -1)] \
        if dims == 3 else [(0, 0), (1, -1), (-1, 1), (-1, 0), (1, 1)]

    def at(u, d):
        return u[tuple(slice(box[2 * k] + d[k], box[2 * k + 1] + d[k])
                       for k in reversed(range(dims)))]

    g, g2 = ps.PSGridNew(shape, np.float32), ps.PSGridNew(shape, np.float32)
    all_of = sum(([1, n - 1] for n in shape), [])
    u = [a.copy(), b.copy()]
    for count in range(1, 8):
        print(f"box {box} of {shape} x {count}", flush=True)
        for x in (g, g2):
            ps.PSGridCopyin(x, np.full(shape[::-1], np.nan, np.float32))
        run(g.handle, g2.handle, *all_of, 5, w)  # both scratch grids
        ps.PSGridCopyin(g, a)
        ps.PSGridCopyin(g2, b)
        run(g.handle, g2.handle, *box, count, w)
        for k in range(2):  # the pair
            v = _sum(lambda d: at(u[k], d), [(None, d) for d in offsets],
                     np.float32)
            at(u[1 - k], (0,) * dims)[...] = v * w
        for x, want in zip((g, g2), u):
            assert np.array_equal(ps.PSGridCopyout(x), want.reshape(-1)), count
    ps.PSGridFree(g)
    ps.PSGridFree(g2)


def test_rows_too_long_for_passes(ps, prog):
    """Rows whose windows fit single sweeps but not a rows pass: the pair runs
    as single sweeps."""
    nx, x0, x1, w = 60_000_000, 29_999_900, 30_000_100, np.float32(0.2)
    print(f"pairs over rows of {nx}", flush=True)
    n = x1 - x0 + 2
    a = np.zeros((3, nx), np.float32)
    a[:, x0 - 1:x1 + 1] = np.random.default_rng(1).standard_normal((3, n))
    g, g2 = ps.PSGridNew((nx, 3)), ps.PSGridNew((nx, 3))
    ps.PSGridCopyin(g, a)
    ps.PSGridCopyin(g2, a)
    prog.ragged_box2d(g.handle, g2.handle, x0, x1, 1, 2, 3, w)
    got = [ps.PSGridCopyout(x).reshape(3, nx) for x in (g, g2)]
    ps.PSGridFree(g)
    ps.PSGridFree(g2)
    u = [a[:, x0 - 1:x1 + 1].copy() for _ in range(2)]
    for k in range(6):
        s = u[k % 2]
        v = s[1, 1:-1] + s[0, 2:] + s[2, :-2] + s[1, :-2] + s[2, 2:]
        u[1 - k % 2][1, 1:-1] = v * w
    for k in range(2):
        assert np.array_equal(got[k][:, x0 - 1:x1 + 1], u[k]), k
        a[:, x0 - 1:x1 + 1] = got[k][:, x0 - 1:x1 + 1]
        assert np.array_equal(got[k], a)


@pytest.mark.parametrize("shape", [(9, 7, 5), (66, 33, 20), (257, 30, 9)])
def test_red_black_double(ps, prog, shape):
    """A red-black map of an 8-byte grid (its colour sweeps are not fused: two
    rings of 8-byte planes do not fit LDS)."""
    print(f"red-black double {shape}", flush=True)
    nx, ny, nz = shape
    a = np.random.default_rng(nx).standard_normal((nz, ny, nx))
    z, y, x = np.meshgrid(*map(np.arange, a.shape), indexing="ij")
    inside = np.zeros(a.shape, bool)
    inside[1:-1, 1:-1, 1:-1] = True
    prog.ragged_relax_double.argtypes = [ps.PSGridPtr, C.c_int]
    for count in (1, 2, 3):
        g = ps.PSGridNew(shape, np.float64)
        ps.PSGridCopyin(g, a)
        prog.ragged_relax_double(g.handle, count)
        got = ps.PSGridCopyout(g)
        ps.PSGridFree(g)
        u = a.copy()
        for k in range(2 * count):
            v = u.copy()
            for axis, d in ((2, -1), (2, 1), (1, -1), (1, 1), (0, -1), (0, 1)):
                v += np.roll(u, d, axis)
            u = np.where(inside & ((x + y + z + k) % 2 == 0), v * 0.125, u)
        assert np.array_equal(got, u.reshape(-1)), count
