"""Operators whose rows name a column more than once (the entries add up, as in the product): the hierarchy
is that of the summed operator, on the host and on the device, whichever way its finest level is held (a
dense inverse, explicit products)."""
import numpy as np
import pytest
import scipy.sparse as sp

import metriko_amd as mk


def _grid(nx, ny, cplx):
    t = lambda n: sp.diags([-np.ones(n - 1), np.full(n, 2.0), -np.ones(n - 1)], [-1, 0, 1])  # noqa: E731
    A = (sp.kron(t(ny), sp.identity(nx)) + sp.kron(sp.identity(ny), t(nx)) + 0.5 * sp.identity(nx * ny)).tocsr()
    if cplx:
        G = sp.diags(np.exp(2j * np.pi * np.random.default_rng(nx).random(nx * ny)))
        A = sp.csr_matrix(G @ A @ G.getH())
    A.sort_indices()
    return A


def _split(A, rng):
    """Every entry in two parts whose sum is exact (1/4 and 3/4 of it), each row in random order."""
    ptr, col, val = [0], [], []
    for i in range(A.shape[0]):
        c, v = A.indices[A.indptr[i]:A.indptr[i + 1]], A.data[A.indptr[i]:A.indptr[i + 1]]
        p = rng.permutation(2 * c.size)
        col.append(np.concatenate([c, c])[p])
        val.append(np.concatenate([0.25 * v, 0.75 * v])[p])
        ptr.append(ptr[-1] + 2 * c.size)
    return sp.csr_matrix((np.concatenate(val), np.concatenate(col), ptr), shape=A.shape)


# dense on the host (up to 500 / 400) and on the device (2,400 / 2,100); dense on the device only; explicit
SIZES = [(16, 15), (33, 31), (61, 60)]


@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("nx,ny", SIZES)
def test_host(nx, ny, cplx):
    rng = np.random.default_rng(ny)
    A = _grid(nx, ny, cplx)
    D = _split(A, rng)
    b = rng.standard_normal(A.shape[0]) + (1j * rng.standard_normal(A.shape[0]) if cplx else 0.0)
    x, it, levels, rel = mk.mg_host_pcg(A, b)
    xd, itd, levelsd, reld = mk.mg_host_pcg(D, b)
    assert (itd, levelsd) == (it, levels) and reld <= 1e-10
    assert np.linalg.norm(xd - x) <= 1e-10 * np.linalg.norm(b) / 0.5  # both stop at 1e-10; |A^-1| <= 1 / 0.5


@pytest.mark.gpu
@pytest.mark.parametrize("precision", [mk.PREC_FP64, mk.PREC_MIXED, mk.PREC_MIXED_MG])
@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("nx,ny", SIZES)
def test_device(gpu_ctx, nx, ny, cplx, precision):
    rng = np.random.default_rng(ny)
    A = _grid(nx, ny, cplx)
    D = _split(A, rng)
    b = rng.standard_normal(A.shape[0]) + (1j * rng.standard_normal(A.shape[0]) if cplx else 0.0)
    make = gpu_ctx.op_complex if cplx else gpu_ctx.op_real
    o = mk.opts(precision=precision)
    x, st = make(A).solve(b, o=o)
    xd, std = make(D).solve(b, o=o)
    assert (std["iterations"], std["mg_levels"]) == (st["iterations"], st["mg_levels"])
    assert np.linalg.norm(xd - x) <= 2e-10 * np.linalg.norm(b) / 0.5
    if not cplx:
        B = rng.standard_normal((A.shape[0], 5))
        X, stm = make(D).solve_many(B, o=o)
        assert np.linalg.norm(A @ X - B, axis=0).max() <= 1e-10 * np.linalg.norm(B, axis=0).max()
        assert stm["iterations"] == make(A).solve_many(B, o=o)[1]["iterations"]
