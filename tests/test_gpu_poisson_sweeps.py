"""Jacobi sweeps of the Poisson solver at the edges of their tiles (64 points
per row of lanes at one point per lane, 128 at two; 8 rows), for even and odd
numbers of two-sweep passes and calls in a row, bit for bit against the
oracle; plain FP32 sweeps on solvers of every storage type."""
import numpy as np
import pytest

import oracle_lib as O
from physis_amd.configs import himeno_inputs, poisson_problem

pytestmark = pytest.mark.gpu


def _grids(ps, arrays, shape):
    out = []
    for a in arrays:
        out.append(ps.PSGridNew(shape))
        ps.PSGridCopyin(out[-1], a)
    return out


def _solver(grids, nbatch, storage):
    from physis_amd.poisson import PoissonSolver
    return PoissonSolver(grids, nbatch, {0: "fp32", 1: "bf16",
                                         2: "fp16"}[storage])


@pytest.mark.parametrize("storage", [0, 1, 2])
@pytest.mark.parametrize("shape,nb", [((4, 3, 3), 1), ((62, 9, 10), 2),
                                      ((64, 8, 7), 1), ((66, 17, 5), 1),
                                      ((126, 10, 6), 2), ((130, 7, 9), 1),
                                      ((194, 5, 4), 1)])
def test_inner_sweeps(ps, shape, nb, storage):
    print(f"inner sweeps {shape} x {nb} storage {storage}", flush=True)
    coefs = poisson_problem(shape[0], shape[1], shape[2] // nb, nbatch=nb,
                            gaussians=(2, 4), sigma=(1.5, 4.0), seed=5)
    n = int(np.prod(shape))
    rng = np.random.default_rng(n)
    e, rhs = (O.to_storage(storage, rng.uniform(-1, 1, n).astype(np.float32) *
                           coefs[10]) for _ in range(2))
    grids = _grids(ps, coefs, shape)
    s = _solver(grids, nb, storage)
    fields = [O.to_storage(storage, c) for c in coefs[:11]] + [rhs]
    try:
        s.set_field(0, e)
        s.set_field(1, rhs)
        for count in (2, 6, 4):
            s.inner_sweeps(count)
            for _ in range(count):
                e = O.poisson_sweep(storage, e, fields, shape, nb)
            assert np.array_equal(s.get_field(0), e), count
    finally:
        s.free()
        for g in grids:
            ps.PSGridFree(g)


@pytest.mark.parametrize("storage", [0, 1, 2])
@pytest.mark.parametrize("shape", [(66, 17, 9), (130, 8, 6)])
def test_plain_sweeps(ps, shape, storage):
    print(f"plain sweeps {shape} on storage {storage}", flush=True)
    coefs, p = himeno_inputs(*shape, seed=13)
    grids = _grids(ps, coefs + [p], shape)
    s = _solver(grids[:12], 1, storage)
    try:
        p0, p1 = p.copy(), p.copy()
        for count in (2, 4, 6):
            s.plain_sweeps(grids[12], count)
            O.lib().oracle_himeno_run(p0, p1, O.coef_array(coefs), *shape,
                                      count, np.float32(0.8), None)
            got = ps.PSGridCopyout(grids[12])
            assert np.array_equal(got.view(np.uint32), p0.view(np.uint32)), \
                count
    finally:
        s.free()
        for g in grids:
            ps.PSGridFree(g)
