"""Small multigrid levels as two explicit products: one V-cycle of the device (the first PCG step from
zero is a multiple of M^-1 b) against the host's smoothed V-cycle on the same two-level hierarchy,
and solves on operators whose products do not fit.  In FP64 both V-cycles round each of a few dozen
products per entry, cond of the smoothed level below 10: 1e-12 of the norm is a hundred times that."""
import ctypes as C

import numpy as np
import pytest
import scipy.sparse as sp

import metriko_amd as mk

pytestmark = pytest.mark.gpu


def _T(n, periodic=False):
    T = sp.lil_matrix(sp.diags([-np.ones(n - 1), 2.0 * np.ones(n), -np.ones(n - 1)], [-1, 0, 1]))
    if periodic:
        T[0, n - 1] = T[n - 1, 0] = -1.0
    return T.tocsr()


def _operator(kind, nx, ny, rng):
    n = nx * ny
    if kind == "five":
        K = sp.kron(_T(ny), sp.identity(nx)) + sp.kron(sp.identity(ny), _T(nx))
    elif kind == "nine":
        M = lambda k: sp.identity(k) - _T(k) / 6  # noqa: E731
        K = sp.kron(_T(ny), M(nx)) + sp.kron(M(ny), _T(nx))
    else:
        K = sp.kron(_T(ny, True), sp.identity(nx)) + sp.kron(sp.identity(ny), _T(nx, True))
        G = sp.diags(np.exp(2j * np.pi * rng.random(n)))
        return sp.csr_matrix(G @ (K + 1e-2 * sp.identity(n)) @ G.getH())
    S = sp.diags(rng.uniform(0.7, 1.4, n))
    return sp.csr_matrix(S @ (K + 1e-2 * sp.identity(n)) @ S)


def _first_step(ctx, op, b, o):
    x = np.zeros_like(op._pack(b))
    bp = op._pack(b)
    d = C.POINTER(C.c_double)
    st = mk.Stats()
    s = ctx.L.mk_spd_solve(ctx.h, op.h, bp.ctypes.data_as(d), x.ctypes.data_as(d), C.byref(o), C.byref(st))
    assert s == 4 and st.iterations == 1  # stopped by the limit, x written
    return op._unpack(x), st.mg_levels


# two levels on both sides: above the dense limit (2,400 / 2,100), coarse below the host's 500 / 400
@pytest.mark.parametrize("kind,nx,ny", [("five", 49, 50), ("five", 7, 351), ("nine", 61, 43), ("nine", 61, 59),
                                        ("hpd", 46, 47), ("hpd", 9, 235)])
def test_v_cycle_matches_the_smoothed_one(gpu_ctx, kind, nx, ny):
    rng = np.random.default_rng(nx)
    A = _operator(kind, nx, ny, rng)
    n = A.shape[0]
    b = rng.standard_normal(n) + (1j * rng.standard_normal(n) if kind == "hpd" else 0.0)
    op = gpu_ctx.op_complex(A) if kind == "hpd" else gpu_ctx.op_real(A)
    z, _, levels, _ = mk.mg_host_pcg(A, b, maxit=0)
    for precision, tol in ((mk.PREC_FP64, 1e-12), (mk.PREC_MIXED_MG, 1e-5)):
        x, dev_levels = _first_step(gpu_ctx, op, b, mk.opts(precision=precision, maxiter=1))
        assert levels == dev_levels == 2
        c = np.vdot(z, x) / np.vdot(z, z)
        assert np.linalg.norm(x - c * z) <= tol * np.linalg.norm(x), precision


@pytest.mark.parametrize("n,row", [(3000, 40), (5000, 12)])
def test_products_that_do_not_fit_are_smoothed(gpu_ctx, n, row):
    """Random couplings: three steps reach more columns than a row of the products may have."""
    rng = np.random.default_rng(n)
    S = sp.random(n, n, density=row / (2.0 * n), random_state=3, format="csr")
    S = -(S + S.T)
    S.setdiag(0)
    A = (S + sp.diags(-1.02 * np.asarray(S.sum(axis=1)).ravel() + 1e-2)).tocsr()
    b = rng.standard_normal(n)
    for precision in (mk.PREC_FP64, mk.PREC_MIXED_MG):
        x, st = gpu_ctx.op_real(A).solve(b, o=mk.opts(precision=precision))
        assert st["mg_levels"] >= 2 and np.linalg.norm(A @ x - b) <= 1e-10 * np.linalg.norm(b)


def test_long_rows_are_smoothed(gpu_ctx):
    """A node coupled to 900 others is a long row: its level keeps the smoother."""
    n = 60 * 61
    rng = np.random.default_rng(5)
    A = _operator("five", 60, 61, rng).tolil()
    hub = rng.choice(np.arange(1, n), 900, replace=False)
    for j in hub:
        A[0, j] = A[j, 0] = A[0, j] - 0.05
        A[j, j] += 0.05
    A[0, 0] += 0.05 * 900
    A = A.tocsr()
    b = rng.standard_normal(n)
    x, st = gpu_ctx.op_real(A).solve(b)
    assert st["mg_levels"] >= 2 and np.linalg.norm(A @ x - b) <= 1e-10 * np.linalg.norm(b)


def _random_couplings(n, row):
    S = sp.random(n, n, density=row / (2.0 * n), random_state=3, format="csr")
    S = -(S + S.T)
    S.setdiag(0)
    return (S + sp.diags(-1.02 * np.asarray(S.sum(axis=1)).ravel() + 1e-2)).tocsr()


def _hub(nx, ny):
    A = _operator("five", nx, ny, np.random.default_rng(5)).tolil()
    for j in np.random.default_rng(5).choice(np.arange(1, nx * ny), 900, replace=False):
        A[0, j] = A[j, 0] = A[0, j] - 0.05
        A[j, j] += 0.05
    A[0, 0] += 0.05 * 900
    return A.tocsr()


def _thirteen(nx, ny):
    K = sp.kron(_T(ny), sp.identity(nx)) + sp.kron(sp.identity(ny), _T(nx))
    return (K @ K + 1e-2 * sp.identity(nx * ny)).tocsr()


# M of the thirteen-point operator has 85 + 10 to 15 entries a row, 8 bytes each: 64 MiB are about 86,000 rows
@pytest.mark.parametrize("what,explicit", [(("five", 49, 50), True), (("nine", 61, 43), True), (("hpd", 46, 47), True),
                                           (("rows", 362, 362), True), (("rows", 363, 362), False),
                                           (("bytes", 270, 270), True), (("bytes", 310, 310), False),
                                           (("random", 3000, 40), False), (("random", 5000, 12), False),
                                           (("hub", 60, 61), False)])
def test_which_finest_levels_are_explicit(gpu_ctx, what, explicit):
    """On both sides of every limit (131,072 rows, 64 MiB, 896 entries a row, long rows), by the kernels
    that a first PCG step runs on the finest level."""
    kind, p, q = what
    A = (_random_couplings(p, q) if kind == "random" else _hub(p, q) if kind == "hub" else
         _thirteen(p, q) if kind == "bytes" else _operator("five" if kind == "rows" else kind, p, q, np.random.default_rng(p)))
    op = gpu_ctx.op_complex(A) if kind == "hpd" else gpu_ctx.op_real(A)
    for precision, tag in ((mk.PREC_FP64, "fp64"), (mk.PREC_MIXED_MG, "fp32")):
        try:
            gpu_ctx.set_timing(True)
            gpu_ctx.timing_report(reset=True)
            _first_step(gpu_ctx, op, np.ones(A.shape[0]), mk.opts(precision=precision, maxiter=1))
            keys = {k["key"] for k in gpu_ctx.timing_report(reset=True)}
        finally:
            gpu_ctx.set_timing(False)
        assert (f"op_mg0_M:cheb_level:{tag}" in keys) == explicit, keys
        assert any(k.startswith("op_mg0:cheb") and k.endswith(tag) for k in keys) != explicit, keys


def _band(n, w):
    """Half-width w: T has 6 w + 1 entries a row (three steps), four strong couplings on either side."""
    v = {d: -0.1 if d <= 4 else -0.1 / (w - 4) for d in range(1, w + 1)}
    S = sp.diags([np.full(n - abs(d), v[abs(d)]) for d in range(-w, w + 1) if d], [d for d in range(-w, w + 1) if d])
    return sp.csr_matrix(S - sp.diags(np.asarray(S.sum(axis=1)).ravel()) + 0.05 * sp.identity(n))


# rows of 169, 187 | 193, 361 and 841: on both sides of the small table (192) and up to the largest
@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("w", [28, 31, 32, 60, 140])
def test_v_cycle_of_the_tables(gpu_ctx, w, cplx):
    n = 2999
    rng = np.random.default_rng(w)
    A = _band(n, w)
    b = rng.standard_normal(n) + (1j * rng.standard_normal(n) if cplx else 0.0)
    if cplx:
        G = sp.diags(np.exp(2j * np.pi * rng.random(n)))
        A = sp.csr_matrix(G @ A @ G.getH())
    op = gpu_ctx.op_complex(A) if cplx else gpu_ctx.op_real(A)
    z, _, levels, _ = mk.mg_host_pcg(A, b, maxit=0)
    for precision, tol, tag in ((mk.PREC_FP64, 1e-12, "fp64"), (mk.PREC_MIXED_MG, 1e-5, "fp32")):
        try:
            gpu_ctx.set_timing(True)
            gpu_ctx.timing_report(reset=True)
            x, dev_levels = _first_step(gpu_ctx, op, b, mk.opts(precision=precision, maxiter=1))
            keys = {k["key"] for k in gpu_ctx.timing_report(reset=True)}
        finally:
            gpu_ctx.set_timing(False)
        assert levels == dev_levels == 2 and f"op_mg0_M:cheb_level:{tag}" in keys
        c = np.vdot(z, x) / np.vdot(z, z)
        assert np.linalg.norm(x - c * z) <= tol * np.linalg.norm(x), precision
