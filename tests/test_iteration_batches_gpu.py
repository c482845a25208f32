"""How many iterations a solver queues before it looks changes nothing but launches: for every
check interval and whatever the operator solved last (an easy, a hard, a zero or an already solved
right-hand side) the solution and its iteration count are the same, bit for bit, and an iteration
limit stops the solve at that count."""
import numpy as np
import pytest
import scipy.sparse as sp

import metriko_amd as mk

pytestmark = pytest.mark.gpu


def _grid(nx, ny, shift):
    T = lambda n: sp.diags([-np.ones(n - 1), 2.0 * np.ones(n), -np.ones(n - 1)], [-1, 0, 1])  # noqa: E731
    return (sp.kron(T(ny), sp.identity(nx)) + sp.kron(sp.identity(ny), T(nx)) + shift * sp.identity(nx * ny)).tocsr()


MODES = [(mk.PREC_MIXED_MG, mk.PRECOND_AMG), (mk.PREC_FP64, mk.PRECOND_AMG), (mk.PREC_FP64, mk.PRECOND_JACOBI)]


@pytest.mark.parametrize("precision,precond", MODES)
def test_result_does_not_depend_on_the_batches(gpu_ctx, precision, precond):
    A = _grid(71, 53, 1e-3)
    rng = np.random.default_rng(1)
    b = rng.standard_normal(A.shape[0])
    smooth = A @ np.ones(A.shape[0])
    fresh = gpu_ctx.op_real(A)
    ref, st0 = fresh.solve(b, o=mk.opts(precision=precision, precond=precond))
    op = gpu_ctx.op_real(A)
    for every in (1, 3, 16, 1000):
        o = mk.opts(precision=precision, precond=precond, check_every=every)
        for before in (b, smooth, np.zeros_like(b)):  # what the batch is planned from
            op.solve(before, o=o)
            x, st = op.solve(b, o=o)
            assert np.array_equal(x, ref) and st["iterations"] == st0["iterations"], (every, st)
        x, st = op.solve(b, x0=ref, o=o)  # converged before the first iteration, up to the recomputed residual
        assert st["iterations"] <= 2 and st["rel_residual"] <= 1e-10
        x, st = op.solve(np.zeros_like(b), o=o)
        assert st["iterations"] == 0 and np.abs(x).max() == 0.0


@pytest.mark.parametrize("precision,precond", MODES)
@pytest.mark.parametrize("limit", [1, 2, 5])
def test_iteration_limit(gpu_ctx, precision, precond, limit):
    A = _grid(71, 53, 1e-4)
    b = np.random.default_rng(2).standard_normal(A.shape[0])
    op = gpu_ctx.op_real(A)
    o = mk.opts(precision=precision, precond=precond)
    need = op.solve(b, o=o)[1]["iterations"]
    assert need > 5
    with pytest.raises(mk.MetrikoError) as ei:
        op.solve(b, o=mk.opts(precision=precision, precond=precond, maxiter=limit))
    assert ei.value.status == 4
    if precond == mk.PRECOND_AMG:
        with pytest.raises(mk.MetrikoError) as ei:
            op.solve_many(np.stack([b, -b], 1), o=mk.opts(precision=precision, precond=precond, maxiter=limit))
        assert ei.value.status == 4
    assert op.solve(b, o=o)[1]["iterations"] == need


def test_block_result_does_not_depend_on_the_batches(gpu_ctx):
    A = _grid(71, 53, 1e-3)
    rng = np.random.default_rng(3)
    B = rng.standard_normal((A.shape[0], 11))
    ref, st0 = gpu_ctx.op_real(A).solve_many(B)
    op = gpu_ctx.op_real(A)
    for every in (1, 3, 16, 1000):
        o = mk.opts(check_every=every)
        for before in (B, np.zeros_like(B)):
            op.solve_many(before, o=o)
            X, st = op.solve_many(B, o=o)
            assert np.array_equal(X, ref) and st["iterations"] == st0["iterations"]
