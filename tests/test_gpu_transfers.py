"""States and arrays across the transfer paths (pinned in one kernel, pageable,
several threads through pinned chunks): sizes at the edges of each, odd node
counts, several host threads at once, and every context closed in between."""
import ctypes as C
import threading

import numpy as np
import pytest

from mfrbf import _lib as L

pytestmark = pytest.mark.gpu

# nodes of a 4-variable state: 1 MiB is 32,768, 4 MiB 131,072, 8 MiB 262,144; chunks of 2 MiB
SIZES = [2, 2209, 32767, 32768, 32769, 65537, 131071, 131072, 200003, 262144, 262145, 700001]


def context(n, seed, nvar=4):
    rng = np.random.default_rng(seed)
    ctx = L.Context(0)
    if nvar == 4:
        ctx.set_equations(L.MF_EQ_EULER_2D, 1.4)
    else:
        ctx.set_equations(L.MF_EQ_ADVECTION_2D, 1.0, 1.0)
    ctx.set_points(rng.random(n), rng.random(n))
    return ctx, rng.standard_normal((nvar, n))


def round_trip(n, seed, nvar=4):
    ctx, u = context(n, seed, nvar)
    ctx.upload(L.MF_BUF_U, u)
    ctx.copy(L.MF_BUF_AUX0, L.MF_BUF_U)
    assert np.array_equal(ctx.download(L.MF_BUF_AUX0), u)
    wide = np.full((nvar, n + 7), -1.0)
    ctx.download_rows(L.MF_BUF_AUX0, wide[:, 3:3 + n])
    assert np.array_equal(wide[:, 3:3 + n], u)
    assert (wide[:, :3] == -1.0).all() and (wide[:, 3 + n:] == -1.0).all()


@pytest.mark.parametrize("nvar", [1, 4])
@pytest.mark.parametrize("n", SIZES)
def test_round_trip(n, nvar):
    round_trip(n, n, nvar)


def test_threads():
    """Eight threads with contexts of their own share the pinned chunks."""
    errors = []

    def work(t):
        try:
            for q in range(3):
                round_trip(SIZES[(3 * t + q) % len(SIZES)], 100 * t + q)
        except Exception as e:  # noqa: BLE001
            errors.append(e)
    th = [threading.Thread(target=work, args=(t,)) for t in range(8)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not errors, errors


@pytest.mark.parametrize("n", [1000, 33000, 140000, 300001])
def test_stencils_and_operators(n):
    """Indices, distances and operators in and out at every transfer size."""
    rng = np.random.default_rng(n)
    ctx, u = context(n, n)
    k = 9
    idx, dist, _, _ = ctx.knn(k, want_dist=True)
    assert np.array_equal(idx[:, 0], np.arange(n)) and (np.diff(dist, axis=1) >= 0).all()
    wx, wy = rng.standard_normal((n, k)), rng.standard_normal((n, k))
    outs = []
    for _ in range(2):
        ctx.set_stencil(idx)
        ctx.set_operator(L.MF_OP_FLUX, wx, wy)
        v, du = np.abs(u) + 1.0, np.empty_like(u)
        ctx.rhs_host(0.0, v, du, L.MF_PREC_F64_REF)
        outs.append(du)
    f = v[1]  # du of the density: -(Dx m1 + Dy m2)
    want = -((wx * f[idx]).sum(1) + (wy * v[2][idx]).sum(1))
    scale = (np.abs(wx * f[idx]) + np.abs(wy * v[2][idx])).sum(1)
    # 2 k products and additions in some order: 2 k roundings of the sum of magnitudes, twice
    assert np.all(np.abs(outs[0][0] - want) <= 4 * k * 2.0 ** -53 * scale)
    assert np.array_equal(outs[0], outs[1])


def test_rhs_host_aliased_fields():
    """du and u the same arrays: u's values stay, as the last ones copied."""
    ctx, u = context(500, 1)
    ctx.knn(15, want_idx=False)
    ctx.compute_operator(3, 2, 1, L.MF_OP_FLUX, want=False)
    u = np.abs(u) + 1.0
    v = u.copy()
    ctx.rhs_host(0.0, v, v)
    assert np.array_equal(v, u)


# 40 MiB, from which several threads upload, is 1,310,720 nodes
@pytest.mark.parametrize("n", [2209, 131072, 262145, 1310719, 1310721])
def test_pinned_arrays(n):
    """Arrays that the runtime knows (allocated pinned) cross directly; pageable
    ones of the same size, and both in one call, give the same."""
    hip = C.CDLL("libamdhip64.so")
    hip.hipHostMalloc.argtypes = [C.POINTER(C.c_void_p), C.c_size_t, C.c_uint]
    hip.hipHostFree.argtypes = [C.c_void_p]
    ctx, u = context(n, n)
    p = C.c_void_p()
    assert hip.hipHostMalloc(C.byref(p), 4 * 8 * n, 0) == 0
    try:
        pin = np.ctypeslib.as_array(C.cast(p, C.POINTER(C.c_double)), shape=(4 * n,)).reshape(4, n)
        pin[:] = u
        ctx.upload(L.MF_BUF_U, pin)
        assert np.array_equal(ctx.download(L.MF_BUF_U), u)
        ctx.upload(L.MF_BUF_U, u)
        pin[:] = 0.0
        ctx.download(L.MF_BUF_U, pin)
        assert np.array_equal(pin, u)
        mixed = [pin[0], np.empty(n), pin[2], np.empty(n)]
        pin[:] = 0.0
        fields = (C.POINTER(C.c_double) * 4)(*[m.ctypes.data_as(C.POINTER(C.c_double)) for m in mixed])
        assert L.lib().mf_state_download(ctx.h, L.MF_BUF_U, fields) == L.MF_OK
        assert all(np.array_equal(m, v) for m, v in zip(mixed, u))
    finally:
        assert hip.hipHostFree(p) == 0


@pytest.mark.parametrize("n", [262145, 1310719])
def test_refused_call_reads_no_more(n):
    """A refused rhs! has taken its pinned arrays when it returns: writing to
    them at once changes nothing of the state that it uploaded."""
    hip = C.CDLL("libamdhip64.so")
    hip.hipHostMalloc.argtypes = [C.POINTER(C.c_void_p), C.c_size_t, C.c_uint]
    hip.hipHostFree.argtypes = [C.c_void_p]
    ctx, u = context(n, n)
    p = C.c_void_p()
    assert hip.hipHostMalloc(C.byref(p), 4 * 8 * n, 0) == 0
    try:
        pin = np.ctypeslib.as_array(C.cast(p, C.POINTER(C.c_double)), shape=(4 * n,)).reshape(4, n)
        pin[:] = u
        du = np.empty((4, n))
        rc = L.lib().mf_rhs_host(ctx.h, 0.0, L.MF_PREC_F64, ctx._fields(pin), ctx._fields(du))
        pin[::-1] = -1.0
        assert rc == L.MF_ERR_STATE  # no operator
        assert np.array_equal(ctx.download(L.MF_BUF_U), u)
    finally:
        ctx.close()
        assert hip.hipHostFree(p) == 0
