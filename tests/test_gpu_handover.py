"""SSPRK33 stages handed over with the next rhs!'s first boundary pass against
the general path: a stage limiter whose threshold no state reaches changes
nothing but runs every boundary pass by itself.  Same bits, eager and from
graphs, in one call and resumed, with the handover switched on and off and
the boundary values changed between the calls."""
import numpy as np
import pytest

import mfrbf
from mfrbf import _lib as L
from mfrbf.clouds import cloud_square

pytestmark = pytest.mark.gpu

OFF, ON = 0, L.MF_STEP_LIMITER  # the limiter: handover on, off


def euler(sources, table):
    x, y, tag, nx, ny = cloud_square(19, 33)
    ctx = L.Context(0)
    ctx.set_equations(L.MF_EQ_EULER_2D, 1.4)
    ctx.set_points(x, y)
    _, _, dx_min, dx_avg = ctx.knn(20, want_idx=False)
    ctx.compute_operator(5, 3, 1, L.MF_OP_FLUX, want=False)
    if "flyer" in sources:
        ctx.compute_operator(5, 3, 4, L.MF_OP_HYPERVISCOSITY, want=False)
        ctx.set_source_hyperviscosity(1e-4 * dx_min ** 4)
    if "tominec" in sources:
        ctx.compute_operator(5, 3, 2, L.MF_OP_LAPLACIAN, want=False)
        ctx.set_source_hyperviscosity_tominec(dx_min ** 4.5)
    if "upwind" in sources:
        ctx.set_source_viscosity(L.MF_VISC_UPWIND, 1.0, 1.0, dx_avg, 3, True)
    inflow, wall = np.nonzero(tag == 1)[0], np.nonzero(tag == 2)[0]
    nodes = np.r_[inflow, wall]
    wave = mfrbf.DensityWave()
    ctx.set_boundary([0, len(inflow), len(nodes)], [L.MF_BC_DIRICHLET, L.MF_BC_SLIP_WALL],
                     [L.MF_FN_TABLE if table else L.MF_FN_WAVE, L.MF_FN_CONST], np.tile(wave.params(), 2), nodes,
                     np.c_[nx, ny][nodes])
    eq = mfrbf.CompressibleEulerEquations2D(1.4)
    ctx.set_stage_limiter([-1e30], [L.MF_VAR_DENSITY])

    def values(t):
        return np.ascontiguousarray(np.asarray(wave(np.c_[x, y][nodes], t, eq)).T)
    u = np.asarray(wave(np.c_[x, y], 0.0, eq))
    return ctx, np.ascontiguousarray(u * (1.0 + 0.01 * np.sin(7.0 * x + 3.0 * y))), values


def advection():
    x, y, tag, _, _ = cloud_square(19, 34)
    ctx = L.Context(0)
    ctx.set_equations(L.MF_EQ_ADVECTION_2D, 1.0, 1.0)
    ctx.set_points(x, y)
    ctx.knn(15, want_idx=False)
    ctx.compute_operator(3, 2, 1, L.MF_OP_FLUX, want=False)
    nodes = np.nonzero(tag == 1)[0]
    pulse = mfrbf.GaussianPulse()
    ctx.set_boundary([0, len(nodes)], [L.MF_BC_DIRICHLET], [L.MF_FN_PULSE], pulse.params(), nodes,
                     np.zeros((len(nodes), 2)))
    ctx.set_stage_limiter([-1e30], [L.MF_VAR_DENSITY])
    return ctx, np.ascontiguousarray(np.asarray(pulse(np.c_[x, y], 0.0, None)).reshape(1, -1)), None


def run(ctx, u0, prec, calls, values=None):
    ctx.upload(L.MF_BUF_U, u0)
    t, out, dt = 0.0, [], 1e-3
    for q, (n, flags) in enumerate(calls):
        if values is not None:
            ctx.set_boundary_values(values(t))
        ctx.ssprk33(t, dt, n, prec, flags, resume=q > 0)
        t += n * dt
        out.append(ctx.download(L.MF_BUF_U))
    return out


@pytest.mark.parametrize("prec", [L.MF_PREC_F64, L.MF_PREC_SPLIT32, L.MF_PREC_F64_REF])
@pytest.mark.parametrize("case", ["advection", "", "flyer", "upwind", "flyer upwind", "tominec", "table", "flyer table"])
def test_handover_bitwise(case, prec):
    words = case.split()
    ctx, u0, values = advection() if case == "advection" else euler(words, "table" in words)
    values = values if "table" in words else None
    for graph in (0, L.MF_STEP_GRAPH):
        for steps in ([5], [2, 1, 3, 0, 2], [17]):
            ref = run(ctx, u0, prec, [(n, ON) for n in steps], values)
            for pattern in ([OFF], [OFF, ON], [ON, OFF]):
                calls = [(n, pattern[q % len(pattern)] | graph) for q, n in enumerate(steps)]
                got = run(ctx, u0, prec, calls, values)
                for q, (a, b) in enumerate(zip(got, ref)):
                    assert np.isfinite(a).all()
                    assert np.array_equal(a, b), (graph, steps, pattern, q)
