"""GPU parity of the Poisson extensions (libphysis_poisson_hip) against the
oracle (oracle/poisson.c) on the same seeded inputs.

Bit-exact: storage conversion of the coefficients, storage-type sweeps
(BF16 / FP16 / FP32), the FP32 plain sweep against the Himeno oracle, the
FP64 residual pass's updated p and scaled RHS, and whole refinement runs on
a fixed schedule.  Reductions: max |r| exact, sums within 1e-12 relative
(FP64 partial sums in a different order).  Solves to 1e-6 are verified by
the oracle's FP64 residual of the returned solution.
"""
from __future__ import annotations

import numpy as np
import pytest

import oracle_lib as O
from physis_amd.configs import himeno_inputs, poisson_problem

pytestmark = pytest.mark.gpu

STORAGE_NAMES = {0: "fp32", 1: "bf16", 2: "fp16"}
# (shape, nbatch): odd sizes, a batch of two, and a wide grid that takes the
# 2-points-per-lane 16-bit sweep (128-point tiles) with a ragged last tile
CASES = [((40, 22, 18), 1), ((34, 14, 18), 2), ((260, 14, 10), 1)]


def _grids(ps, arrays, shape, dtype=np.float32):
    out = []
    for a in arrays:
        g = ps.PSGridNew(shape, dtype)
        ps.PSGridCopyin(g, a)
        out.append(g)
    return out


def _free(ps, grids):
    for g in grids:
        ps.PSGridFree(g)


def _solver(coef_grids, nbatch, storage):
    from physis_amd.poisson import PoissonSolver
    return PoissonSolver(coef_grids, nbatch, STORAGE_NAMES[storage])


@pytest.mark.parametrize("storage", [0, 1, 2])
@pytest.mark.parametrize("case", CASES)
def test_inner_sweeps_bit_exact(ps, storage, case):
    shape, nb = case
    print(f"inner sweeps storage={storage} shape={shape} nbatch={nb}",
          flush=True)
    nz = shape[2]
    coefs = poisson_problem(shape[0], shape[1], nz // nb, nbatch=nb,
                            gaussians=(2, 4), sigma=(1.5, 4.0), seed=21)
    grids = _grids(ps, coefs, shape)
    s = _solver(grids, nb, storage)
    try:
        rng = np.random.default_rng(7)
        n = int(np.prod(shape))
        for k in range(11):  # storage copies of a0 .. c2, bnd
            got = s.get_field(2 + k)
            assert np.array_equal(got, O.to_storage(storage, coefs[k])), k
        e = O.to_storage(storage, rng.uniform(-1, 1, n).astype(np.float32) *
                         coefs[10])
        rhs = O.to_storage(storage, rng.uniform(-1, 1, n).astype(np.float32) *
                           coefs[10])
        s.set_field(0, e)
        s.set_field(1, rhs)
        s.inner_sweeps(6)
        got = s.get_field(0)
        fields = [O.to_storage(storage, c) for c in coefs[:11]] + [rhs]
        ref = e
        for _ in range(6):
            ref = O.poisson_sweep(storage, ref, fields, shape, nb)
        assert np.array_equal(got, ref)
    finally:
        s.free()
        _free(ps, grids)


@pytest.mark.parametrize("shape", [(40, 22, 18), (260, 14, 10)])
def test_plain_sweeps_match_the_himeno_oracle(ps, shape):
    print(f"plain sweeps shape={shape}", flush=True)
    nx, ny, nz = shape
    coefs, p = himeno_inputs(nx, ny, nz, seed=13)
    coefs[11] = (np.random.default_rng(3).uniform(-0.1, 0.1, p.size)
                 .astype(np.float32) * coefs[10])
    grids = _grids(ps, coefs, shape)
    pg = _grids(ps, [p], shape)[0]
    s = _solver(grids, 1, 0)
    try:
        s.plain_sweeps(pg, 8)
        got = ps.PSGridCopyout(pg)
        p0, p1 = p.copy(), p.copy()
        O.lib().oracle_himeno_run(p0, p1, O.coef_array(coefs), nx, ny, nz, 8,
                                  np.float32(0.8), None)
        assert np.array_equal(got.view(np.uint32), p0.view(np.uint32))
    finally:
        s.free()
        _free(ps, grids + [pg])


@pytest.mark.parametrize("storage", [0, 1, 2])
@pytest.mark.parametrize("case", CASES)
def test_residual_pass(ps, storage, case):
    shape, nb = case
    print(f"residual storage={storage} shape={shape} nbatch={nb}", flush=True)
    nz = shape[2]
    coefs = poisson_problem(shape[0], shape[1], nz // nb, nbatch=nb,
                            gaussians=(2, 4), sigma=(1.5, 4.0), seed=22)
    n = int(np.prod(shape))
    rng = np.random.default_rng(11)
    p64 = rng.uniform(-2, 2, n) * coefs[10]
    e = O.to_storage(storage, rng.uniform(-1, 1, n).astype(np.float32) *
                     coefs[10])
    grids = _grids(ps, coefs, shape)
    pg, qg = _grids(ps, [p64, np.zeros(n)], shape, np.float64)
    p32g = _grids(ps, [p64.astype(np.float32)], shape)[0]
    s = _solver(grids, nb, storage)
    try:
        s.set_field(0, e)
        # update + residual + scaled RHS
        sums = s.residual(pg, qg, inv_sigma=0.25, sigma=8.0)
        p_out, rhs, ref = O.poisson_residual(storage, p64, coefs, shape, nb,
                                             e=e, inv_sigma=0.25, sigma=8.0)
        assert np.array_equal(ps.PSGridCopyout(qg).view(np.uint64),
                              p_out.view(np.uint64))
        assert np.array_equal(s.get_field(1), rhs)
        assert np.array_equal(sums[:, 1], ref[:, 1])
        np.testing.assert_allclose(sums[:, [0, 2]], ref[:, [0, 2]],
                                   rtol=1e-12)
        # norms only, FP32 p
        sums = s.residual(p32g)
        _, _, ref = O.poisson_residual(storage, p64.astype(np.float32),
                                       coefs, shape, nb)
        assert np.array_equal(sums[:, 1], ref[:, 1])
        np.testing.assert_allclose(sums[:, [0, 2]], ref[:, [0, 2]],
                                   rtol=1e-12)
    finally:
        s.free()
        _free(ps, grids + [pg, qg, p32g])


@pytest.mark.parametrize("storage", [1, 2])
def test_refinement_schedule_bit_exact(ps, storage):
    shape, nb = (34, 14, 18), 2
    print(f"refinement schedule storage={storage}", flush=True)
    coefs = poisson_problem(shape[0], shape[1], 9, nbatch=nb,
                            gaussians=(2, 4), sigma=(1.5, 4.0), seed=23)
    n = int(np.prod(shape))
    grids = _grids(ps, coefs, shape)
    pg = _grids(ps, [np.zeros(n)], shape, np.float64)[0]
    s = _solver(grids, nb, storage)
    try:
        st = s.solve_mixed(pg, tol=0.0, inner=8, max_sweeps=40)
        ref, rst = O.poisson_solve_mixed(storage, coefs, np.zeros(n), shape,
                                         nb, 0.8, 0.0, 8, 40)
        assert (st["outer"], st["sweeps"]) == (rst["outer"], rst["sweeps"])
        assert np.array_equal(ps.PSGridCopyout(pg).view(np.uint64),
                              ref.view(np.uint64))
    finally:
        s.free()
        _free(ps, grids + [pg])


def _rel_fp64(coefs, p, shape, nb):
    _, _, sums = O.poisson_residual(0, p, coefs, shape, nb)
    return np.sqrt(sums[:, 0] / sums[:, 2])


@pytest.mark.parametrize("storage", [1, 2])
def test_mixed_solve_reaches_1e6(ps, storage):
    """BF16 / FP16 storage, FP64 refinement: every problem of a batch
    reaches relative residual 1e-6, verified by the oracle's FP64 residual;
    the error against the FP64 Jacobi solution is bounded by 1e-4
    relative (measured ~1e-6)."""
    shape, nb = (32, 30, 56), 2
    print(f"mixed solve storage={storage}", flush=True)
    coefs = poisson_problem(32, 30, 28, nbatch=nb, gaussians=(4, 8),
                            sigma=(2.0, 6.0), seed=31)
    n = int(np.prod(shape))
    grids = _grids(ps, coefs, shape)
    pg = _grids(ps, [np.zeros(n)], shape, np.float64)[0]
    s = _solver(grids, nb, storage)
    try:
        st = s.solve_mixed(pg, tol=1e-6, inner=50)
        p = ps.PSGridCopyout(pg)
        rel = _rel_fp64(coefs, p, shape, nb)
        print("stats", st, "oracle rel", rel, flush=True)
        assert st["converged"] and np.all(rel <= 1e-6 * (1 + 1e-9))
        ref, _, _ = O.poisson_jacobi_fp64(coefs, np.zeros(n), shape, nb,
                                          tol=1e-12, check=100)
        err = np.linalg.norm(p - ref) / np.linalg.norm(ref)
        print("error vs FP64 Jacobi", err, flush=True)
        assert err < 1e-4
    finally:
        s.free()
        _free(ps, grids + [pg])


def test_plain_fp32_solve(ps):
    """Plain FP32 Jacobi with FP64 residual checks: converges (or reports
    stagnation) and its reported residual is the oracle's FP64 residual of
    the returned FP32 field."""
    shape = (32, 30, 28)
    coefs = poisson_problem(*shape, nbatch=1, gaussians=(4, 8),
                            sigma=(2.0, 6.0), seed=31)
    n = int(np.prod(shape))
    grids = _grids(ps, coefs, shape)
    pg = _grids(ps, [np.zeros(n, np.float32)], shape)[0]
    s = _solver(grids, 1, 0)
    try:
        st = s.solve_plain(pg, tol=1e-6, check=50)
        p = ps.PSGridCopyout(pg)
        rel = _rel_fp64(coefs, p, shape, 1)
        print("plain stats", st, "oracle rel", rel, flush=True)
        assert st["converged"] or st["stagnated"]
        np.testing.assert_allclose(rel[0], st["rel_residual"], rtol=1e-9)
    finally:
        s.free()
        _free(ps, grids + [pg])
