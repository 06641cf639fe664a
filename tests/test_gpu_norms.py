"""The residual viscosity's norms (hyperviscosity.jl:289-311) on states whose
lexicographic maximum is decided in every way the reductions distinguish: by
one node, by ties within a wavefront, across wavefronts and across blocks, by
later components, and with NaN and infinity (NaN above every number).  The
reductions select, they do not round: exact equality with numpy."""
import numpy as np
import pytest

from mfrbf import _lib as L
from mfrbf.clouds import cloud_square

pytestmark = pytest.mark.gpu


def brute_ninf(u, mean):
    d = np.abs(u - mean[:, None])
    live = np.arange(d.shape[1])
    for v in range(4):
        c = d[v, live]
        live = live[np.isnan(c)] if np.isnan(c).any() else live[c == c.max()]
    best = d[:, live[0]]
    return np.where(best == 0.0, np.finfo(float).eps, best)


def states(n, rng):
    u = np.stack([1.0 + 0.1 * rng.random(n), rng.standard_normal(n), rng.standard_normal(n), 5.0 + rng.random(n)])
    yield "one node", u.copy()
    for name, nodes in (("wave", [3, 17, 30]), ("waves", [q for q in (5, 70, 200, 7000) if q < n]),
                        ("all", np.arange(n))):
        t = u.copy()
        t[0] = 1.0
        t[0, nodes] = 3.0
        yield "tie in density, " + name, t.copy()
        t[1] = -0.5
        yield "tie in density and momentum, " + name, t
    yield "constant", np.repeat([[1.0], [0.5], [0.25], [5.0]], n, axis=1)
    for name, val in (("nan", np.nan), ("inf", np.inf)):
        for v in (0, 2):
            t = u.copy()
            t[v, n // 2] = val
            yield "%s in component %d" % (name, v), t


@pytest.mark.parametrize("side", [6, 16, 17, 47, 100])
def test_norms_exact(side):
    rng = np.random.default_rng(side)
    x, y, _, _, _ = cloud_square(side, 40 + side)
    n = len(x)
    ctx = L.Context(0)
    ctx.set_equations(L.MF_EQ_EULER_2D, 1.4)
    ctx.set_points(x, y)
    _, _, _, h = ctx.knn(15, want_idx=False)
    ctx.compute_operator(3, 2, 1, L.MF_OP_FLUX, want=False)
    ctx.set_source_viscosity(L.MF_VISC_RESIDUAL, 1.0, 1.0, h, 3, True)
    for tiles in (1, 0):
        ctx.set_tuning(L.MF_TUNE_TILES, tiles)
        for name, u in states(n, rng):
            u = np.ascontiguousarray(u)
            ctx.upload(L.MF_BUF_U, u)
            for prec in (L.MF_PREC_F64, L.MF_PREC_F64_REF, L.MF_PREC_SPLIT32):
                ctx.rhs(0.0, prec)
                mean, ninf = ctx.viscosity_norms()
                assert np.array_equal(ninf, brute_ninf(u, mean), equal_nan=True), (side, tiles, name, prec)
