"""Resumed integrations: a stored stage that was handed over with its next
boundary pass when the boundary conditions change between the calls, and
calls between two resumed ones that must leave the stored stage alone or
make the resume an error."""
import numpy as np
import pytest

import mfrbf
from mfrbf import _lib as L
from mfrbf.clouds import cloud_square

pytestmark = pytest.mark.gpu

GENERAL, HANDED = L.MF_STEP_LIMITER, 0  # the limiter: no stage is handed over
DT = 1e-3


def euler(residual, table=False):
    x, y, tag, nx, ny = cloud_square(23, 41)
    ctx = L.Context(0)
    ctx.set_equations(L.MF_EQ_EULER_2D, 1.4)
    ctx.set_points(x, y)
    _, _, _, dx_avg = ctx.knn(20, want_idx=False)
    ctx.compute_operator(5, 3, 1, L.MF_OP_FLUX, want=False)
    if residual:
        ctx.set_source_viscosity(L.MF_VISC_RESIDUAL, 1.0, 1.0, dx_avg, 3, True)
    wave = mfrbf.DensityWave()
    inflow, wall = np.nonzero(tag == 1)[0], np.nonzero(tag == 2)[0]
    nodes = np.r_[inflow, wall]

    def boundary(scale):
        """The inflow's density scaled, through the table or the wave's parameters."""
        params = np.tile(wave.params(), 2)
        params[0] *= scale
        if not table:
            ctx.set_boundary([0, len(inflow), len(nodes)], [L.MF_BC_DIRICHLET, L.MF_BC_SLIP_WALL],
                             [L.MF_FN_WAVE, L.MF_FN_CONST], params, nodes, np.c_[nx, ny][nodes])
            return
        v = np.asarray(wave(np.c_[x, y][nodes], 0.0, mfrbf.CompressibleEulerEquations2D(1.4)))
        ctx.set_boundary_values(np.ascontiguousarray((scale * v).T))

    if table:
        ctx.set_boundary([0, len(inflow), len(nodes)], [L.MF_BC_DIRICHLET, L.MF_BC_SLIP_WALL],
                         [L.MF_FN_TABLE, L.MF_FN_CONST], np.tile(wave.params(), 2), nodes, np.c_[nx, ny][nodes])
    boundary(1.0)
    ctx.set_stage_limiter([-1e30], [L.MF_VAR_DENSITY])  # no state reaches the threshold
    u = np.asarray(wave(np.c_[x, y], 0.0, mfrbf.CompressibleEulerEquations2D(1.4)))
    return ctx, np.ascontiguousarray(u * (1.0 + 0.01 * np.sin(7.0 * x + 3.0 * y))), boundary


@pytest.mark.parametrize("change", ["values", "boundary", "gamma"])
@pytest.mark.parametrize("residual", [False, True])
def test_boundary_changes_between_resumed_calls(residual, change):
    """Against the path that runs every boundary pass by itself.  Without the
    residual viscosity the bits; with it the means are summed in another order:
    a few hundred roundings of a mean of order 1 (1e-13), through the norms
    into the viscosity and at most 6 steps.  The stale boundary is off by the
    change, 1e-2."""
    ctx, u0, boundary = euler(residual, table=change == "values")
    flags = L.MF_STEP_HISTORY if residual else 0
    out = {}
    for mode in (GENERAL, HANDED, HANDED | L.MF_STEP_GRAPH):
        ctx.set_equations(L.MF_EQ_EULER_2D, 1.4)
        boundary(1.0)
        ctx.upload(L.MF_BUF_U, u0)
        t, got = 0.0, []
        for q, steps in enumerate((2, 1, 3)):
            ctx.ssprk33(t, DT, steps, L.MF_PREC_F64, mode | flags, resume=q > 0)
            t += steps * DT
            got.append(ctx.download(L.MF_BUF_U))
            if change == "gamma":
                ctx.set_equations(L.MF_EQ_EULER_2D, 1.4 + 0.01 * (q + 1))
            else:
                boundary(1.0 + 0.01 * (q + 1))
        out[mode] = got
    for mode in (HANDED, HANDED | L.MF_STEP_GRAPH):
        for a, b in zip(out[mode], out[GENERAL]):
            assert np.isfinite(a).all()
            assert np.abs(a - b).max() <= (1e-10 * np.abs(b).max() if residual else 0.0)


@pytest.mark.parametrize("table", [False, True])
def test_adjoint_between_resumed_calls(table):
    """mf_rhs_vjp leaves the state and the stored stage alone, also when the
    boundary values change after it: the same bits as without it."""
    ctx, u0, boundary = euler(False, table)
    ctx.upload(L.MF_BUF_AUX0, np.ascontiguousarray(u0[::-1]))
    out = []
    for vjp in (False, True):
        boundary(1.0)
        ctx.upload(L.MF_BUF_U, u0)
        ctx.ssprk33(0.0, DT, 2, L.MF_PREC_F64, 0)
        if vjp:
            ctx.rhs_vjp(2 * DT)
        boundary(1.01)
        ctx.ssprk33(2 * DT, DT, 3, L.MF_PREC_F64, 0, resume=True)
        out.append(ctx.download(L.MF_BUF_U))
    assert np.isfinite(out[0]).all() and np.array_equal(out[0], out[1])


def test_limiter_ends_a_resumable_integration():
    """mf_limiter_zhang_shu changes the state that the stored stage was formed
    from, as an upload does: the next call starts anew or is an error."""
    ctx, u0, _ = euler(False)
    ctx.upload(L.MF_BUF_U, u0)
    ctx.ssprk33(0.0, DT, 2, L.MF_PREC_F64, 0)
    ctx.limiter_zhang_shu(float(ctx.download(L.MF_BUF_U)[0].mean()), L.MF_VAR_DENSITY)
    u = ctx.download(L.MF_BUF_U)
    with pytest.raises(L.MfError) as e:
        ctx.ssprk33(2 * DT, DT, 1, L.MF_PREC_F64, 0, resume=True)
    assert e.value.code == L.MF_ERR_STATE
    ctx.ssprk33(2 * DT, DT, 1, L.MF_PREC_F64, 0)
    got = ctx.download(L.MF_BUF_U)
    ctx.upload(L.MF_BUF_U, u)
    ctx.ssprk33(2 * DT, DT, 1, L.MF_PREC_F64, 0)
    assert np.isfinite(got).all() and np.array_equal(got, ctx.download(L.MF_BUF_U))
