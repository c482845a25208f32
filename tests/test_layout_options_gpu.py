"""Layout options of a solve that no kernel is built for are refused with MK_ERR_ARG before anything is
built, whichever way the hierarchy's levels are held (a dense inverse, explicit products, smoothed), and
the operator stays usable."""
import numpy as np
import pytest
import scipy.sparse as sp

import metriko_amd as mk

pytestmark = pytest.mark.gpu


def _grid(nx, ny, cplx):
    t = lambda n: sp.diags([-np.ones(n - 1), np.full(n, 2.0), -np.ones(n - 1)], [-1, 0, 1])  # noqa: E731
    A = (sp.kron(t(ny), sp.identity(nx)) + sp.kron(sp.identity(ny), t(nx)) + 0.5 * sp.identity(nx * ny)).tocsr()
    if not cplx:
        return A
    G = sp.diags(np.exp(2j * np.pi * np.random.default_rng(nx).random(nx * ny)))
    return sp.csr_matrix(G @ A @ G.getH())


BAD = [{"block_size": b} for b in (0, -64, 32, 96, 512)] + [{"slice_height": h} for h in (0, 32, 96)] + [{"sigma": 0}]


@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("nx,ny", [(16, 15), (47, 44), (61, 60)])
def test_refused_and_usable_after(gpu_ctx, cplx, nx, ny):
    A = _grid(nx, ny, cplx)
    n = A.shape[0]
    b = A @ np.ones(n)
    op = (gpu_ctx.op_complex if cplx else gpu_ctx.op_real)(A)
    for bad in BAD:
        for precision in (mk.PREC_FP64, mk.PREC_MIXED, mk.PREC_MIXED_MG):
            with pytest.raises(mk.MetrikoError) as ei:
                op.solve(b, o=mk.opts(precision=precision, **bad))
            assert ei.value.status == 1, bad
    x, _ = op.solve(b)
    # |x - 1| <= |A^-1| |r| <= 1e-10 |b| / 0.5
    assert np.linalg.norm(x - 1.0) <= 2e-10 * np.linalg.norm(b)
    if cplx:
        with pytest.raises(mk.MetrikoError) as ei:
            gpu_ctx.smallest_eig(gpu_ctx.op_complex(A), np.ones(n), np.ones(n, complex), 2, mk.opts(block_size=0))
        assert ei.value.status == 1
