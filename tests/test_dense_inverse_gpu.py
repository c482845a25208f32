"""The dense inverse of the coarsest multigrid level: operators small enough to be solved by it
alone (one level), at the edges of its 16 / 32 / 64 tiles and of its size range, real and complex,
with FP64 and FP32 vectors and in blocks of every width.  An exact inverse leaves PCG one
iteration, or two or three when its vectors are rounded to FP32 (2^-24 of error per iteration
against the 1e-10 asked for), so the iteration count judges the inverse itself; the solution is
within cond(A) x 1e-10 of numpy's."""
import numpy as np
import pytest
import scipy.sparse as sp

import metriko_amd as mk

pytestmark = pytest.mark.gpu


def _operator(n, cplx, rng):
    """Random sparse Hermitian, made diagonally dominant by 5 percent: cond(A) <= 41."""
    S = sp.random(n, n, density=min(1.0, 6.0 / n), random_state=int(rng.integers(1 << 30)), format="csr")
    if cplx:
        S = S.astype(np.complex128)
        S.data = S.data * np.exp(2j * np.pi * rng.random(S.nnz))
    S = S + S.getH()
    S.setdiag(0)
    d = np.asarray(abs(S).sum(axis=1)).ravel()
    return (S + sp.diags(1.05 * np.maximum(d, 1e-3))).tocsr()


@pytest.mark.parametrize("precision,most", [(mk.PREC_FP64, 1), (mk.PREC_MIXED_MG, 3)])
@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("n", [1, 2, 15, 16, 17, 31, 32, 33, 63, 64, 65, 127, 129, 401, 1000, 2100, 2399, 2400])
def test_one_level_solve(gpu_ctx, n, cplx, precision, most):
    if cplx and n > 2100:
        pytest.skip("beyond the complex limit")
    rng = np.random.default_rng(n)
    A = _operator(n, cplx, rng)
    b = rng.standard_normal(n) + (1j * rng.standard_normal(n) if cplx else 0.0)
    op = gpu_ctx.op_complex(A) if cplx else gpu_ctx.op_real(A)
    x, st = op.solve(b, o=mk.opts(precision=precision))
    ref = np.linalg.solve(A.toarray(), b)
    assert st["mg_levels"] == 1 and st["iterations"] <= most, st
    assert np.linalg.norm(x - ref) <= 41 * 1e-10 * np.linalg.norm(ref)


@pytest.mark.parametrize("precision,most", [(mk.PREC_FP64, 1), (mk.PREC_MIXED_MG, 3)])
@pytest.mark.parametrize("m", [5, 8, 11, 16, 23, 32, 50, 64])
@pytest.mark.parametrize("n", [7, 64, 121, 778])
def test_one_level_block(gpu_ctx, n, m, precision, most):
    rng = np.random.default_rng(n * m)
    A = _operator(n, False, rng)
    B = rng.standard_normal((n, m))
    X, st = gpu_ctx.op_real(A).solve_many(B, o=mk.opts(precision=precision))
    ref = np.linalg.solve(A.toarray(), B)
    assert st["mg_levels"] == 1 and st["iterations"] <= most, st
    assert (np.linalg.norm(X - ref, axis=0) <= 41 * 1e-10 * np.linalg.norm(ref, axis=0)).all()


def test_beyond_the_limits_is_smoothed(gpu_ctx):
    rng = np.random.default_rng(0)
    for n, cplx in ((2401, False), (2101, True)):
        A = _operator(n, cplx, rng)
        b = rng.standard_normal(n) + (1j * rng.standard_normal(n) if cplx else 0.0)
        op = gpu_ctx.op_complex(A) if cplx else gpu_ctx.op_real(A)
        x, st = op.solve(b)
        assert st["mg_levels"] >= 2
        assert np.linalg.norm(A @ x - b) <= 1e-10 * np.linalg.norm(b)
