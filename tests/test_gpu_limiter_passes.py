"""The limiter's two passes in a stage (one copy back after both) against one
pass after another, and its minimum over the tiles against the global gathers,
at the edges of its batches."""
import numpy as np
import pytest

from mfrbf import _lib as L
from mfrbf.clouds import cloud_square

pytestmark = pytest.mark.gpu

THR = ((0.6, L.MF_VAR_DENSITY), (1.0, L.MF_VAR_PRESSURE))


def problem(side, k, nvar=4):
    rng = np.random.default_rng(side + k)
    x, y, _, _, _ = cloud_square(side, side)
    n = len(x)
    ctx = L.Context(0)
    if nvar == 4:
        ctx.set_equations(L.MF_EQ_EULER_2D, 1.4)
    else:
        ctx.set_equations(L.MF_EQ_ADVECTION_2D, 1.0, 0.5)
    ctx.set_points(x, y)
    ctx.set_stencil(ctx.knn(k)[0])
    ctx.set_operator(L.MF_OP_FLUX, np.zeros((n, k)), np.zeros((n, k)))
    u = np.ascontiguousarray(np.stack([1.0 + 0.1 * rng.random(n), 0.1 * rng.standard_normal(n),
                                       0.1 * rng.standard_normal(n), 5.0 + rng.random(n)])[:nvar])
    u[0, rng.permutation(n)[: max(1, n // 20)]] = 0.3
    if nvar == 4:
        u[3, rng.permutation(n)[: max(1, n // 20)]] = 1.0
    return ctx, u


def passes(ctx, u, thr):
    ctx.upload(L.MF_BUF_U, np.ascontiguousarray(u))
    for t, v in thr:
        ctx.limiter_zhang_shu(t, v)
    return ctx.download(L.MF_BUF_U)


@pytest.mark.parametrize("side,k", [(4, 3), (16, 15), (17, 16), (17, 17), (33, 30), (33, 32), (40, 33), (40, 48),
                                    (40, 64), (61, 64)])
@pytest.mark.parametrize("nvar", [1, 4])
def test_limiter_passes(side, k, nvar):
    """With a zero operator a step is S = U, T = (3 U + S) / 4,
    U = (U + 2 T) / 3, each limited: a few roundings of each value apart from
    the same on the host."""
    ctx, u0 = problem(side, k, nvar)
    thr = THR if nvar == 4 else ((0.6, L.MF_VAR_DENSITY), (0.7, L.MF_VAR_DENSITY))
    out = []
    for tiles in (1, 0):
        print("limiter", side, k, nvar, tiles, flush=True)
        ctx.set_tuning(L.MF_TUNE_TILES, tiles)
        ctx.set_stage_limiter([t for t, _ in thr], [v for _, v in thr])
        ctx.upload(L.MF_BUF_U, u0.copy())
        ctx.ssprk33(0.0, 1e-3, 1, L.MF_PREC_F64, L.MF_STEP_LIMITER)
        stepped = ctx.download(L.MF_BUF_U)
        out.append((stepped, passes(ctx, u0, thr[:1]), passes(ctx, u0, thr)))
    for a, b in zip(*out):
        assert np.array_equal(a, b)
    stepped, first, both = out[0]
    assert not np.array_equal(first, u0)
    assert nvar == 1 or not np.array_equal(first, both)
    s = passes(ctx, u0, thr)
    t = passes(ctx, (3.0 * u0 + s) / 4.0, thr)
    assert np.allclose(stepped, passes(ctx, (u0 + 2.0 * t) / 3.0, thr), rtol=1e-12, atol=1e-12)
