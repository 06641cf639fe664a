"""The adjoint's tiled transposed product against the global one (same bits),
and the loss of the reverse sweep against numpy, at the edges of their
batches, tiles and running sums."""
import numpy as np
import pytest

from mfrbf import _lib as L
from mfrbf.clouds import cloud_square

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("eq,side,k", [("euler", 4, 3), ("advection", 4, 3), ("euler", 16, 4), ("euler", 17, 9),
                                       ("advection", 33, 15), ("euler", 33, 30), ("advection", 64, 30),
                                       ("euler", 128, 16), ("euler", 370, 6), ("advection", 370, 6)])
def test_reverse_sweep(eq, side, k):
    """One to a few tiles, widths below and above the batches, one and more
    than one node of each running sum (1024 of them), and more than two tiles
    per CU.  The loss sums N squares: N eps relative to it."""
    rng = np.random.default_rng(side + k)
    x, y, _, _, _ = cloud_square(side, side)
    n, v = len(x), 4 if eq == "euler" else 1
    ctx = L.Context(0)
    if v == 4:
        ctx.set_equations(L.MF_EQ_EULER_2D, 1.4)
    else:
        ctx.set_equations(L.MF_EQ_ADVECTION_2D, 1.0, 0.5)
    ctx.set_points(x, y)
    ctx.set_stencil(ctx.knn(k)[0])
    ctx.set_operator(L.MF_OP_FLUX, rng.standard_normal((n, k)), rng.standard_normal((n, k)))
    u0 = 0.1 * rng.standard_normal((v, n))
    u0[0] += 1.0
    if v == 4:
        u0[3] += 5.0
    lam = rng.standard_normal((v, n))
    out = []
    for tiles in (1, 0):
        print("reverse sweep", eq, side, k, "tiles", tiles, flush=True)
        ctx.set_tuning(L.MF_TUNE_TILES, tiles)
        ctx.upload(L.MF_BUF_U, np.ascontiguousarray(u0))
        ctx.upload(L.MF_BUF_AUX0, lam)
        ctx.rhs_vjp(0.0)
        product = ctx.download(L.MF_BUF_AUX1)
        loss = ctx.ssprk33_vjp(0.0, 1e-6, 3, 2)
        out.append((product, loss, ctx.download(L.MF_BUF_AUX1)))
    for a, b in zip(*out):
        assert np.isfinite(a).all() and np.array_equal(a, b)
    ctx.upload(L.MF_BUF_U, np.ascontiguousarray(u0))
    ctx.ssprk33(0.0, 1e-6, 3, L.MF_PREC_F64)
    rho = ctx.download(L.MF_BUF_U)[0]
    assert abs(out[0][1] - np.sum(rho * rho)) <= n * np.finfo(float).eps * out[0][1]
