"""PCG breakdowns found by a fold (p^H A p or r^H z not positive, a NaN): the kernel that finds one hands
it to the next kernel in a word that none of its own blocks reads, so every block leaves x alone.
x after a breakdown in iteration k + 1 is the k-th iterate bit for bit (k = 0: the start vector), run
after run, on both sides of the fold's limit (524,288 rows) and for every mode."""
import ctypes as C

import numpy as np
import pytest
import scipy.sparse as sp

import metriko_amd as mk

pytestmark = pytest.mark.gpu

NOT_SPD, NO_CONVERGENCE, NAN = 3, 4, 5
MODES = [(mk.PREC_FP64, mk.PRECOND_NONE), (mk.PREC_FP64, mk.PRECOND_JACOBI), (mk.PREC_FP64, mk.PRECOND_AMG),
         (mk.PREC_MIXED_MG, mk.PRECOND_AMG)]
# one block, a dense hierarchy; several blocks, an explicit level; the largest folded one; unfolded
SIZES = [(17, 15, 0.0), (17, 16, 0.3), (61, 60, 0.0), (61, 60, 0.3), (723, 725, 0.0), (725, 724, 0.0)]


def _grid(nx, ny, phase, shift):
    def t(n):
        u = np.full(n - 1, np.exp(1j * phase)) if phase else np.ones(n - 1)
        return sp.diags([-np.conj(u), np.full(n, 2.0), -u], [-1, 0, 1], format="csr")
    return (sp.kron(t(ny), sp.identity(nx)) + sp.kron(sp.identity(ny), t(nx)) + shift * sp.identity(nx * ny)).tocsr()


def _solve(ctx, op, b, x0, o):
    x, bp = op._pack(x0).copy(), op._pack(b)
    d = C.POINTER(C.c_double)
    st = mk.Stats()
    s = ctx.L.mk_spd_solve(ctx.h, op.h, bp.ctypes.data_as(d), x.ctypes.data_as(d), C.byref(o), C.byref(st))
    return s, op._unpack(x), st.iterations


def _op(ctx, A, phase):
    return (ctx.op_complex if phase else ctx.op_real)(A)


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("nx,ny,phase", SIZES)
def test_x_keeps_its_last_iterate(gpu_ctx, mode, nx, ny, phase):
    """Eigenvalues from -0.5 to 7.5: without multigrid some iterations pass before a direction is
    negative; the V-cycle of such an operator is not positive either, or not finite."""
    precision, precond = mode
    A = _grid(nx, ny, phase, -0.5)
    n = A.shape[0]
    rng = np.random.default_rng(nx)
    b = rng.standard_normal(n) + (1j * rng.standard_normal(n) if phase else 0.0)
    x0 = 0.1 * rng.standard_normal(n) + (0.1j * rng.standard_normal(n) if phase else 0.0)
    op = _op(gpu_ctx, A, phase)
    s, x, it = _solve(gpu_ctx, op, b, x0, mk.opts(precision=precision, precond=precond))
    print(mode, nx, ny, phase, "status", s, "iterations", it)
    assert s in ((NOT_SPD, NAN) if precond == mk.PRECOND_AMG else (NOT_SPD,))
    assert np.isfinite(x).all()
    assert it > 0 or precond == mk.PRECOND_AMG
    again = _solve(gpu_ctx, op, b, x0, mk.opts(precision=precision, precond=precond))
    assert again[0] == s and again[2] == it and np.array_equal(again[1], x)
    if it == 0:
        assert np.array_equal(x, x0)
    else:
        s, kept, k = _solve(gpu_ctx, op, b, x0, mk.opts(precision=precision, precond=precond, maxiter=it))
        assert s == NO_CONVERGENCE and k == it and np.array_equal(kept, x)


@pytest.mark.parametrize("mode", MODES[:2])
@pytest.mark.parametrize("nx,ny", [(17, 15), (723, 725), (725, 724)])
def test_first_direction_negative(gpu_ctx, mode, nx, ny):
    """Unit diagonal and -1 to every neighbour: negative along the constant vector."""
    A = _grid(nx, ny, 0.0, -3.0)
    n = A.shape[0]
    x0 = np.full(n, 0.5)
    s, x, it = _solve(gpu_ctx, gpu_ctx.op_real(A), np.ones(n), x0, mk.opts(precision=mode[0], precond=mode[1]))
    assert s == NOT_SPD and it == 0 and np.array_equal(x, x0)


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("nx,ny,phase", SIZES)
def test_nan_right_hand_side(gpu_ctx, mode, nx, ny, phase):
    precision, precond = mode
    A = _grid(nx, ny, phase, 0.5)
    n = A.shape[0]
    b = np.ones(n) + (1j if phase else 0.0)
    b[n // 2] = np.nan
    x0 = np.full(n, 0.25) + (0.5j if phase else 0.0)
    s, x, it = _solve(gpu_ctx, _op(gpu_ctx, A, phase), b, x0, mk.opts(precision=precision, precond=precond))
    assert s == NAN and it == 0 and np.array_equal(x, x0)


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("nx,ny,phase", SIZES + [(47, 45, 0.0)])
def test_negative_last_pivot(gpu_ctx, mode, nx, ny, phase):
    """One negative eigenvalue, -0.38, along the last unknown.  The dense inverse of the whole operator (up
    to 2,400 / 2,100 unknowns) replaces its last pivot by a tiny positive one: finite, and p points
    along the negative direction at once."""
    precision, precond = mode
    A = _grid(nx, ny, phase, 0.5).tolil()
    n = A.shape[0]
    A[n - 1, n - 1] = 0.1
    A = A.tocsr()
    rng = np.random.default_rng(ny)
    b = rng.standard_normal(n) + (1j * rng.standard_normal(n) if phase else 0.0)
    x0 = 0.1 * rng.standard_normal(n) + (0.1j * rng.standard_normal(n) if phase else 0.0)
    op = _op(gpu_ctx, A, phase)
    s, x, it = _solve(gpu_ctx, op, b, x0, mk.opts(precision=precision, precond=precond))
    print(mode, nx, ny, phase, "status", s, "iterations", it)
    assert s in ((NOT_SPD,) if n < 2400 else (NOT_SPD, NAN)) and np.isfinite(x).all()
    assert it == 0 or n > 2400 or precond != mk.PRECOND_AMG
    again = _solve(gpu_ctx, op, b, x0, mk.opts(precision=precision, precond=precond))
    assert again[0] == s and again[2] == it and np.array_equal(again[1], x)
    if it == 0:
        assert np.array_equal(x, x0)
    else:
        s, kept, k = _solve(gpu_ctx, op, b, x0, mk.opts(precision=precision, precond=precond, maxiter=it))
        assert s == NO_CONVERGENCE and k == it and np.array_equal(kept, x)
