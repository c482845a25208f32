"""The scalars between the kernels of a PCG iteration are added up by the kernel that needs them (up
to 2,048 partials) or by a one-block kernel in between: on both sides of that line (524,288 rows for
the vector kernels), and for one row and one block, every mode reaches the solution.

Bound: the solvers stop at |r| <= 1e-10 |b|, so |x - x*| <= |A^-1| |r| <= 1e-10 |b| / lambda_min, and
lambda_min >= shift; the recurrence's residual drifts from the true one by less than that again."""
import numpy as np
import pytest
import scipy.sparse as sp

import metriko_amd as mk

pytestmark = pytest.mark.gpu

SHIFT = 0.5
MODES = [(mk.PREC_FP64, mk.PRECOND_NONE), (mk.PREC_FP64, mk.PRECOND_JACOBI), (mk.PREC_MIXED, mk.PRECOND_JACOBI),
         (mk.PREC_FP64, mk.PRECOND_AMG), (mk.PREC_MIXED_MG, mk.PRECOND_AMG)]


def _grid(nx, ny, phase):
    def t(n):
        u = np.full(n - 1, np.exp(1j * phase)) if phase else np.ones(n - 1)
        return sp.diags([-np.conj(u), np.full(n, 2.0), -u], [-1, 0, 1], format="csr") if n > 1 else sp.csr_matrix([[2.0]])
    A = (sp.kron(t(ny), sp.identity(nx)) + sp.kron(sp.identity(ny), t(nx)) + SHIFT * sp.identity(nx * ny)).tocsr()
    return A


SIZES = [(1, 1, 0.0), (16, 16, 0.0), (17, 16, 0.3), (723, 725, 0.0), (725, 724, 0.0), (725, 724, 0.3)]
# the multigrid set-up refuses the large complex grid (its aggregation stalls)
CASES = [(m, s) for m in MODES for s in SIZES if not (m[1] == mk.PRECOND_AMG and s == SIZES[-1])]


@pytest.mark.parametrize("mode,size", CASES)
def test_both_sides_of_the_fold(gpu_ctx, mode, size):
    (precision, precond), (nx, ny, phase) = mode, size
    A = _grid(nx, ny, phase)
    n = A.shape[0]
    rng = np.random.default_rng(nx)
    x = rng.standard_normal(n) + (1j * rng.standard_normal(n) if phase else 0.0)
    b = A @ x
    op = (gpu_ctx.op_complex if phase else gpu_ctx.op_real)(A)
    got, st = op.solve(b, o=mk.opts(precision=precision, precond=precond))
    assert np.linalg.norm(got - x) <= 2.0 * 1e-10 * np.linalg.norm(b) / SHIFT, st
    again, _ = op.solve(b, o=mk.opts(precision=precision, precond=precond))
    assert np.array_equal(got, again)
