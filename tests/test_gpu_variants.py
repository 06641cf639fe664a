"""Every compiled variant of the stencil and transposed kernels (entries in
flight, one or two batches in turn, LDS tiles or global gathers) keeps the
per-node operation order: the same bits for each stencil size, source and
precision, on clouds whose last tile is partly filled."""
import numpy as np
import pytest

import mfrbf
from mfrbf import _lib as L
from mfrbf.clouds import cloud_square

pytestmark = pytest.mark.gpu

BASES = {15: (3, 2), 20: (5, 3), 30: (5, 3), 23: (5, 3)}


def context(side, k, sources):
    p, deg = BASES[k]
    x, y, tag, nx, ny = cloud_square(side, 70 + side)
    ctx = L.Context(0)
    ctx.set_equations(L.MF_EQ_EULER_2D, 1.4)
    ctx.set_points(x, y)
    _, _, dx_min, dx_avg = ctx.knn(k, want_idx=False)
    ctx.compute_operator(p, deg, 1, L.MF_OP_FLUX, want=False)
    if "flyer" in sources:
        ctx.compute_operator(p, deg, 4, L.MF_OP_HYPERVISCOSITY, want=False)
        ctx.set_source_hyperviscosity(1e-4 * dx_min ** 4)
    if "tominec" in sources:
        ctx.compute_operator(p, deg, 2, L.MF_OP_LAPLACIAN, want=False)
        ctx.set_source_hyperviscosity_tominec(dx_min ** 4.5)
    if "residual" in sources:
        ctx.set_source_viscosity(L.MF_VISC_RESIDUAL, 1.0, 1.0, dx_avg, 3, True)
    ctx.set_source_order([{"flyer": L.MF_SRC_FLYER, "residual": L.MF_SRC_VISCOSITY, "tominec": L.MF_SRC_TOMINEC}[s]
                          for s in sources])
    inflow, wall = np.nonzero(tag == 1)[0], np.nonzero(tag == 2)[0]
    wave = mfrbf.DensityWave()
    ctx.set_boundary([0, len(inflow), len(inflow) + len(wall)], [L.MF_BC_DIRICHLET, L.MF_BC_SLIP_WALL],
                     [L.MF_FN_WAVE, L.MF_FN_CONST], np.tile(wave.params(), 2), np.r_[inflow, wall],
                     np.c_[nx, ny][np.r_[inflow, wall]])
    u = np.ascontiguousarray(wave(np.c_[x, y], 0.0, mfrbf.CompressibleEulerEquations2D(1.4)))
    for q in range(4):
        ctx.upload(L.MF_BUF_U, u * (1.0 + 1e-4 * q * np.cos(9.0 * x)))
        ctx.history_update(1e-3 * q, q)
    return ctx, u


@pytest.mark.parametrize("prec", [L.MF_PREC_F64, L.MF_PREC_SPLIT32, L.MF_PREC_F64_REF])
@pytest.mark.parametrize("k", sorted(BASES))
@pytest.mark.parametrize("sources", [(), ("flyer",), ("flyer", "residual"), ("residual", "tominec"), ("tominec",),
                                     ("flyer", "residual", "tominec")])
def test_variants_bitwise(sources, k, prec):
    for side in (8, 17, 33):
        ctx, u0 = context(side, k, sources)
        ref = None
        for tiles in (0, 1):
            ctx.set_tuning(L.MF_TUNE_TILES, tiles)
            for fb in (0, 3, 5, 6, 10) if tiles else (0,):
                for tb in (0, 2, 4, 8) if tiles and "residual" in sources else (0,):
                    ctx.set_tuning(L.MF_TUNE_FLUX_BATCH, fb, prec)
                    ctx.set_tuning(L.MF_TUNE_TRANSPOSE_BATCH, tb, prec)
                    u, du = u0.copy(), np.empty_like(u0)
                    ctx.rhs_host(0.004, u, du, prec)
                    if ref is None:
                        ref = (u, du)
                    assert np.isfinite(du).all()
                    assert np.array_equal(u, ref[0]) and np.array_equal(du, ref[1]), (side, tiles, fb, tb)


@pytest.mark.parametrize("prec", [L.MF_PREC_F64, L.MF_PREC_SPLIT32, L.MF_PREC_F64_REF])
@pytest.mark.parametrize("side,k", [(8, 15), (17, 20), (33, 30), (33, 23), (321, 20)])
def test_tominec_transposed_batches(side, k, prec):
    """The transposed product of the Tominec source alone: each batch by the
    tuning value, with tiles and without, and the default (side 321: more than
    one and a half tiles per compute unit)."""
    ctx, u0 = context(side, k, ("tominec",))
    out = []
    for tiles in (0, 1):
        ctx.set_tuning(L.MF_TUNE_TILES, tiles)
        for tb in (0, 2, 4, 8):
            ctx.set_tuning(L.MF_TUNE_TRANSPOSE_BATCH, tb, prec)
            u, du = u0.copy(), np.empty_like(u0)
            ctx.rhs_host(0.004, u, du, prec)
            assert ctx.tile_info()["tiles_b"] == tiles
            out.append(du)
    assert np.isfinite(out[0]).all()
    for du in out[1:]:
        assert np.array_equal(du, out[0])


@pytest.mark.parametrize("prec", [L.MF_PREC_F64, L.MF_PREC_SPLIT32, L.MF_PREC_F64_REF])
@pytest.mark.parametrize("side,k,sources", [(300, 20, ("residual", "tominec")), (600, 15, ("residual",)),
                                            (520, 20, ("residual", "tominec")), (300, 30, ("flyer",))])
def test_default_batches_on_large_clouds(side, k, sources, prec):
    """The defaults that depend on the tiles per compute unit, against the global
    gathers."""
    ctx, u0 = context(side, k, sources)
    out = []
    for tiles in (0, 1):
        ctx.set_tuning(L.MF_TUNE_TILES, tiles)
        u, du = u0.copy(), np.empty_like(u0)
        ctx.rhs_host(0.004, u, du, prec)
        out.append(du)
    assert np.isfinite(out[0]).all() and np.array_equal(out[0], out[1])
