"""Block PCG column bookkeeping (mk_spd_solve_many): every block width and the column counts at
their edges, with columns that are empty, converge at once or break down, each column judged by
its own residual against the 1e-10 the call promises."""
import numpy as np
import pytest
import scipy.sparse as sp

import metriko_amd as mk

pytestmark = pytest.mark.gpu


def _grid(nx, ny, shift):
    T = lambda n: sp.diags([-np.ones(n - 1), 2.0 * np.ones(n), -np.ones(n - 1)], [-1, 0, 1])  # noqa: E731
    return (sp.kron(T(ny), sp.identity(nx)) + sp.kron(sp.identity(ny), T(nx)) + shift * sp.identity(nx * ny)).tocsr()


@pytest.mark.parametrize("precision", [mk.PREC_MIXED_MG, mk.PREC_FP64])
@pytest.mark.parametrize("m", [1, 8, 9, 16, 17, 32, 33, 64, 65])
def test_columns_at_the_block_widths(gpu_ctx, m, precision):
    A = _grid(83, 61, 1e-3)
    n = A.shape[0]
    rng = np.random.default_rng(m)
    B = rng.standard_normal((n, m))
    if m > 2:
        B[:, 1] = 0.0                     # finished before the first iteration
        B[:, 2] = A @ np.ones(n) * 1e-30  # a tiny column: its own norm is the reference
    X, st = gpu_ctx.op_real(A).solve_many(B, o=mk.opts(precision=precision))
    res = np.linalg.norm(A @ X - B, axis=0) / np.maximum(np.linalg.norm(B, axis=0), 1e-300)
    assert res.max() <= 1e-10 and st["solves"] == m
    if m > 2:
        assert np.abs(X[:, 1]).max() == 0.0


def test_a_column_with_nan_is_reported(gpu_ctx):
    A = _grid(40, 37, 1e-3)
    B = np.random.default_rng(0).standard_normal((A.shape[0], 12))
    B[5, 7] = np.nan
    op = gpu_ctx.op_real(A)
    with pytest.raises(mk.MetrikoError) as ei:
        op.solve_many(B)
    assert ei.value.status == 5
    B[5, 7] = 0.0
    X, _ = op.solve_many(B)  # the operator is still usable
    assert np.linalg.norm(A @ X - B) <= 1e-10 * np.linalg.norm(B)


@pytest.mark.parametrize("precision", [mk.PREC_MIXED_MG, mk.PREC_FP64])
@pytest.mark.parametrize("nx,ny", [(1, 1), (3, 1), (9, 7), (83, 61)])
@pytest.mark.parametrize("m", [3, 16, 31, 64])
def test_short_medium_and_long_rows(gpu_ctx, m, nx, ny, precision):
    """Rows of every kind of the layout (5 entries; 24 to 60; hundreds to all of them), at counts below
    and beside a wavefront's share; a right-hand side that is solved at once among the others, whose
    last step is applied while they go on."""
    A = _grid(nx, ny, 1e-2) if nx * ny > 1 else sp.csr_matrix([[3.0]])
    n = A.shape[0]
    rng = np.random.default_rng(n + m)
    for _ in range(5):
        k = rng.choice(n, min(30, n), replace=False)
        v = sp.csr_matrix((np.full(k.size, 0.3 / np.sqrt(k.size)), (k, np.zeros(k.size, int))), shape=(n, 1))
        A = A + v @ v.T
    for row, size in ((0, n), (n // 2, (n + 1) // 2), (n - 1, min(n, 300))):  # couplings below the shift
        k = rng.choice(n, size, replace=False)
        v = sp.csr_matrix((np.full(size, 1e-3 / np.sqrt(size)), (np.full(size, row), k)), shape=(n, n))
        A = A + v + v.T
    B = rng.standard_normal((n, m))
    B[:, 1] = A @ np.ones(n)
    op = gpu_ctx.op_real(A)
    X, st = op.solve_many(B, o=mk.opts(precision=precision))
    res = np.linalg.norm(A @ X - B, axis=0) / np.linalg.norm(B, axis=0)
    assert res.max() <= 1e-10
    again, _ = op.solve_many(B, o=mk.opts(precision=precision))
    assert np.array_equal(X, again)


@pytest.mark.parametrize("height", [64, 128, 192, 256])
@pytest.mark.parametrize("m", [8, 13, 64])
def test_slice_heights(gpu_ctx, m, height):
    A = _grid(37, 29, 1e-2)
    B = np.random.default_rng(height).standard_normal((A.shape[0], m))
    X, _ = gpu_ctx.op_real(A, o=mk.opts(slice_height=height)).solve_many(B)
    assert (np.linalg.norm(A @ X - B, axis=0) / np.linalg.norm(B, axis=0)).max() <= 1e-10


@pytest.mark.parametrize("m", [3, 40])
@pytest.mark.parametrize("precision", [mk.PREC_FP64, mk.PREC_MIXED_MG])
def test_true_residual_of_a_strongly_scaled_operator(gpu_ctx, m, precision):
    """The block recurrence carries A P along (q = A z + beta q) and reports its own residual, driven to half
    the target.  Rows and columns scaled by 10^-2 to 10^2: the true residual, whose drift is of the order
    of eps |A| |x| / |b| per iteration, still meets the target."""
    nx = 90
    T = sp.diags([-np.ones(nx - 1), 2.0 * np.ones(nx), -np.ones(nx - 1)], [-1, 0, 1])
    rng = np.random.default_rng(m)
    S = sp.diags(10.0 ** rng.uniform(-2.0, 2.0, nx * nx))
    A = (S @ (sp.kron(T, sp.identity(nx)) + sp.kron(sp.identity(nx), T) + 1e-2 * sp.identity(nx * nx)) @ S).tocsr()
    B = rng.standard_normal((A.shape[0], m))
    X, st = gpu_ctx.op_real(A).solve_many(B, o=mk.opts(precision=precision))
    assert (np.linalg.norm(A @ X - B, axis=0) <= 1e-10 * np.linalg.norm(B, axis=0)).all(), st
