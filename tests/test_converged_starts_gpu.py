"""Solves whose start already meets the tolerance (a zero right-hand side, a warm start at the solution), between
ordinary solves of the same operator: no iteration is taken, x stays as it is, and of the iterations
that the last solve would have needed only the first few are queued (their products are counted)."""
import numpy as np
import pytest
import scipy.sparse as sp

import metriko_amd as mk

pytestmark = pytest.mark.gpu


def _grid(nx, ny, phase):
    def t(n):
        u = np.full(n - 1, np.exp(1j * phase)) if phase else np.ones(n - 1)
        return sp.diags([-np.conj(u), np.full(n, 2.0), -u], [-1, 0, 1], format="csr")
    return (sp.kron(t(ny), sp.identity(nx)) + sp.kron(sp.identity(ny), t(nx)) + 1e-2 * sp.identity(nx * ny)).tocsr()


MODES = [(mk.PREC_FP64, mk.PRECOND_NONE), (mk.PREC_FP64, mk.PRECOND_JACOBI), (mk.PREC_FP64, mk.PRECOND_AMG),
         (mk.PREC_MIXED_MG, mk.PRECOND_AMG)]


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("nx,ny,phase", [(25, 24, 0.0), (70, 71, 0.0), (60, 61, 0.3)])
def test_no_iteration_and_few_products(gpu_ctx, mode, nx, ny, phase):
    precision, precond = mode
    A = _grid(nx, ny, phase)
    n = A.shape[0]
    rng = np.random.default_rng(ny)
    b = rng.standard_normal(n) + (1j * rng.standard_normal(n) if phase else 0.0)
    op = (gpu_ctx.op_complex if phase else gpu_ctx.op_real)(A)
    o, loose = (mk.opts(precision=precision, precond=precond, tol=t) for t in (1e-10, 1e-9))
    x, st = op.solve(b, o=o)
    calls = {"zero": [], "warm": []}
    for _ in range(4):
        y, s = op.solve(b, o=o)
        assert np.array_equal(y, x) and s["iterations"] == st["iterations"]
        z, sz = op.solve(0.0 * b, o=o)
        assert sz["iterations"] == 0 and not z.any()
        op.solve(b, o=o)
        w, sw = op.solve(b, x0=x, o=loose)
        assert sw["iterations"] == 0 and np.array_equal(w, x)
        calls["zero"].append(sz["spmv_calls"])
        calls["warm"].append(sw["spmv_calls"])
    # the host gives up waiting for a slow device after 300 us: the best of the four
    if st["iterations"] >= 6:
        assert max(min(calls["zero"]), min(calls["warm"])) <= 0.6 * s["spmv_calls"], (calls, s)


@pytest.mark.parametrize("precision", [mk.PREC_FP64, mk.PREC_MIXED_MG])
@pytest.mark.parametrize("m", [3, 20, 64])
def test_blocks_of_zeros(gpu_ctx, m, precision):
    A = _grid(70, 71, 0.0)
    B = np.random.default_rng(m).standard_normal((A.shape[0], m))
    op, o = gpu_ctx.op_real(A), mk.opts(precision=precision)
    X, st = op.solve_many(B, o=o)
    calls = []
    for _ in range(4):
        Z, sz = op.solve_many(0.0 * B, o=o)
        assert sz["iterations"] == 0 and not Z.any()
        calls.append(sz["spmv_calls"])
        Y, s = op.solve_many(B, o=o)
        assert np.array_equal(Y, X) and s["iterations"] == st["iterations"]
    assert st["iterations"] >= 6 and min(calls) <= 0.6 * s["spmv_calls"], (calls, s)
