"""Consistent systems of singular and nearly singular operators (a grid without boundary values, shifted by up
to 1e-12): the dense inverse of the coarsest level leaves out the unknown whose pivot is rounding, and an
FP32 Krylov solve that breaks down goes on without the direction that only FP64 resolves."""
import numpy as np
import pytest
import scipy.sparse as sp

import metriko_amd as mk

pytestmark = pytest.mark.gpu


def _neumann(n):
    d = np.full(n, 2.0)
    d[0] = d[-1] = 1.0
    return sp.diags([-np.ones(n - 1), d, -np.ones(n - 1)], [-1, 0, 1])


def _system(nx, ny, cplx, shift, parts=1):
    """`parts` uncoupled grids: as many directions of zero."""
    A = sp.kron(_neumann(ny), sp.identity(nx)) + sp.kron(sp.identity(ny), _neumann(nx))
    A = sp.block_diag([A] * parts, format="csr") + shift * sp.identity(parts * nx * ny)
    n = A.shape[0]
    rng = np.random.default_rng(nx)
    if cplx:
        G = sp.diags(np.exp(2j * np.pi * rng.random(n)))
        A = G @ A @ G.getH()
    A = sp.csr_matrix(A)
    return A, A @ (rng.standard_normal(n) + (1j * rng.standard_normal(n) if cplx else 0.0))


# one-level (dense), two-level with an explicit finest level, three levels
@pytest.mark.parametrize("precision", [mk.PREC_FP64, mk.PREC_MIXED, mk.PREC_MIXED_MG])
@pytest.mark.parametrize("shift", [0.0, 1e-12])
@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("nx,ny,parts", [(15, 16, 1), (30, 31, 1), (45, 44, 1), (20, 21, 4), (49, 50, 1), (60, 61, 1),
                                         (30, 31, 5), (95, 94, 1), (150, 151, 1)])
def test_consistent_system(gpu_ctx, nx, ny, parts, cplx, shift, precision):
    A, b = _system(nx, ny, cplx, shift, parts)
    x, st = (gpu_ctx.op_complex if cplx else gpu_ctx.op_real)(A).solve(b, o=mk.opts(precision=precision))
    assert st["rel_residual"] <= 1e-10 and np.linalg.norm(A @ x - b) <= 1.01e-10 * np.linalg.norm(b), st


@pytest.mark.parametrize("precision", [mk.PREC_FP64, mk.PREC_MIXED_MG])
@pytest.mark.parametrize("nx,ny,parts", [(15, 16, 1), (45, 44, 1), (20, 21, 4), (60, 61, 1), (95, 94, 1)])
def test_consistent_block(gpu_ctx, nx, ny, parts, precision):
    A, _ = _system(nx, ny, False, 0.0, parts)
    B = A @ np.random.default_rng(ny).standard_normal((A.shape[0], 11))
    X, st = gpu_ctx.op_real(A).solve_many(B, o=mk.opts(precision=precision))
    assert (np.linalg.norm(A @ X - B, axis=0) <= 1.01e-10 * np.linalg.norm(B, axis=0)).all(), st
