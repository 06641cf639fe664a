"""The LDS tiles and the transposed operator built on the device: halo sizes
and padded entries against numpy, clouds whose halos do not fit, stencils
that hold a node twice, columns of more than 64 entries, and the results of
the tiled kernels against the global gathers (same bits)."""
import numpy as np
import pytest

import mfrbf
from mfrbf import _lib as L
from mfrbf.clouds import cloud_square

pytestmark = pytest.mark.gpu


def operators(ctx, idx, rng):
    n, k = idx.shape
    ctx.set_stencil(idx)
    ctx.set_operator(L.MF_OP_FLUX, rng.standard_normal((n, k)), rng.standard_normal((n, k)))


def expected(idx, order):
    """halo and padding totals of 256-node tiles in the internal order."""
    n = len(idx)
    inv = np.empty(n, np.int64)
    inv[order] = np.arange(n)
    rows = inv[idx[order]]  # internal node -> internal neighbours
    tile = np.arange(n) // 256
    col = [[] for _ in range(n)]
    for r in range(n):
        for j in rows[r]:
            col[j].append(r)
    ha = [len(np.unique(rows[tile == t])) for t in range(tile[-1] + 1)]
    hb, padded = [], 0
    for t in range(tile[-1] + 1):
        mine = [col[i] for i in np.nonzero(tile == t)[0]]
        hb.append(len(set(sum(mine, []))))
        deg = sorted([len(c) for c in mine] + [0] * (256 - len(mine)), reverse=True)
        padded += 64 * sum(deg[0::64])
    return sum(ha), sum(hb), max(ha), max(hb), padded


def both_ways(ctx, n, rng, visc=True):
    """rhs! and its VJP with the tiles and with global gathers: the same bits."""
    u0 = np.ascontiguousarray(np.stack([1.0 + 0.1 * rng.random(n), rng.standard_normal(n), rng.standard_normal(n),
                                        5.0 + rng.random(n)]))
    lam = rng.standard_normal((4, n))
    out = []
    for tiles in (1, 0):
        ctx.set_tuning(L.MF_TUNE_TILES, tiles)
        got = []
        for prec in (L.MF_PREC_F64, L.MF_PREC_F64_REF, L.MF_PREC_SPLIT32):
            u, du = u0.copy(), np.empty_like(u0)
            ctx.set_source_viscosity(L.MF_VISC_UPWIND, 1.0, 1.0, 0.01, 3, True)
            ctx.rhs_host(0.0, u, du, prec)
            got.append(du)
        ctx.set_source_viscosity(L.MF_VISC_NONE, 1.0, 1.0, 0.01, 3, True)
        ctx.upload(L.MF_BUF_U, u0)
        ctx.upload(L.MF_BUF_AUX0, lam)
        ctx.rhs_vjp(0.0)
        got.append(ctx.download(L.MF_BUF_AUX1))
        out.append(got)
    for a, b in zip(*out):
        assert np.isfinite(a).all() and np.array_equal(a, b)


@pytest.mark.parametrize("side,k", [(4, 3), (8, 15), (16, 30), (17, 30), (33, 20), (61, 64)])
def test_tiles_against_numpy(side, k):
    rng = np.random.default_rng(side)
    x, y, _, _, _ = cloud_square(side, 90 + side)
    ctx = L.Context(0)
    ctx.set_equations(L.MF_EQ_EULER_2D, 1.4)
    ctx.set_points(x, y)
    idx = ctx.knn(k)[0]
    operators(ctx, idx, rng)
    both_ways(ctx, len(x), rng)
    ctx.set_tuning(L.MF_TUNE_TILES, 1)
    ctx.set_source_viscosity(L.MF_VISC_UPWIND, 1.0, 1.0, 0.01, 3, True)
    ctx.upload(L.MF_BUF_U, np.ones((4, len(x))))
    ctx.rhs(0.0)
    ti = ctx.tile_info()
    want = expected(idx, ctx.node_order())
    assert ti["tiles_a"] and ti["tiles_b"]
    assert (ti["halo_a_total"], ti["halo_b_total"], ti["halo_a_max"], ti["halo_b_max"], ti["b_entries_padded"]) == want


@pytest.mark.parametrize("n", [1100, 5000])
def test_halos_that_do_not_fit(n):
    """Scattered stencils (the caller's order, random neighbours): every tile
    reaches more nodes than LDS holds, the kernels gather globally."""
    rng = np.random.default_rng(n)
    ctx = L.Context(0)
    ctx.set_equations(L.MF_EQ_EULER_2D, 1.4)
    ctx.set_points(rng.random(n), rng.random(n))
    idx = np.stack([np.r_[i, rng.choice(np.delete(np.arange(n), i), 29, replace=False)] for i in range(n)])
    operators(ctx, idx.astype(np.int32), rng)
    both_ways(ctx, n, rng)
    ctx.set_tuning(L.MF_TUNE_TILES, 1)
    ctx.upload(L.MF_BUF_U, np.ones((4, n)))
    ctx.rhs(0.0)
    assert not ctx.tile_info()["tiles_a"]


def test_repeated_nodes_and_long_columns():
    """A node twice in one stencil, and columns of more than 64 entries (a hub
    in every stencil)."""
    rng = np.random.default_rng(3)
    x, y, _, _, _ = cloud_square(20, 5)
    n = len(x)
    ctx = L.Context(0)
    ctx.set_equations(L.MF_EQ_EULER_2D, 1.4)
    ctx.set_points(x, y)
    idx = ctx.knn(20)[0].copy()
    idx[:, 7] = 11  # the hub
    idx[::3, 9] = idx[::3, 4]  # repeated
    operators(ctx, idx, rng)
    both_ways(ctx, n, rng)


def test_advection_tiles_and_vjp():
    """One variable: the larger halo limit, the transposed tiles of one value."""
    rng = np.random.default_rng(9)
    x, y, _, _, _ = cloud_square(40, 6)
    n = len(x)
    ctx = L.Context(0)
    ctx.set_equations(L.MF_EQ_ADVECTION_2D, 1.0, 0.5)
    ctx.set_points(x, y)
    idx = ctx.knn(15)[0]
    operators(ctx, idx, rng)
    u, lam = rng.standard_normal((1, n)), rng.standard_normal((1, n))
    out = []
    for tiles in (1, 0):
        ctx.set_tuning(L.MF_TUNE_TILES, tiles)
        ctx.upload(L.MF_BUF_U, u)
        ctx.upload(L.MF_BUF_AUX0, lam)
        ctx.rhs_vjp(0.0)
        ctx.rhs(0.0)
        out.append((ctx.download(L.MF_BUF_AUX1), ctx.download(L.MF_BUF_DU)))
        if tiles:
            assert ctx.tile_info()["tiles_a"] and ctx.tile_info()["tiles_b"]
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])


@pytest.mark.parametrize("n,unnamed", [(1000, 64), (1000, 300), (1024, 1), (1024, 600), (129, 65)])
def test_slices_that_no_stencil_names(n, unnamed):
    """The last nodes, and 64 in the middle, are in no stencil: their slices of
    the transposed operator have no entries (a whole tile of them with 300 and
    600), and the kernels load none."""
    rng = np.random.default_rng(n + unnamed)
    k = 12
    ctx = L.Context(0)
    ctx.set_equations(L.MF_EQ_EULER_2D, 1.4)
    ctx.set_points(rng.random(n), rng.random(n))
    ctx.set_stencil(np.tile(np.arange(k, dtype=np.int32), (n, 1)))
    order = ctx.node_order()
    named = np.setdiff1d(np.arange(n - unnamed), np.arange(64, 128) if n > 200 else [])
    row = np.minimum(np.arange(n), len(named) - k)
    idx = np.empty((n, k), np.int32)
    idx[order] = order[named[row[:, None] + np.arange(k)]]
    operators(ctx, idx, rng)
    both_ways(ctx, n, rng)
    assert ctx.tile_info()["tiles_a"] == 0  # the last pass was the one without


def test_transposed_halos_that_do_not_fit():
    """Stencils of 64 nodes: the stencil halos fit (1,024 records), the transposed
    ones of G and L together (682) do not: tiled stencil kernel, global
    transposed gather."""
    rng = np.random.default_rng(11)
    x, y, _, _, _ = cloud_square(61, 151)
    n = len(x)
    ctx = L.Context(0)
    ctx.set_equations(L.MF_EQ_EULER_2D, 1.4)
    ctx.set_points(x, y)
    idx = ctx.knn(64)[0]
    operators(ctx, idx, rng)
    ctx.set_operator(L.MF_OP_LAPLACIAN, rng.standard_normal(idx.shape))
    ctx.set_source_hyperviscosity_tominec(1e-3)
    ctx.set_source_viscosity(L.MF_VISC_UPWIND, 1.0, 1.0, 0.01, 3, True)
    ctx.set_source_order([L.MF_SRC_VISCOSITY, L.MF_SRC_TOMINEC])
    u0 = np.ascontiguousarray(np.stack([1.0 + 0.1 * rng.random(n), rng.standard_normal(n), rng.standard_normal(n),
                                        5.0 + rng.random(n)]))
    for prec in (L.MF_PREC_F64, L.MF_PREC_F64_REF, L.MF_PREC_SPLIT32):
        out = []
        for tiles in (1, 0):
            ctx.set_tuning(L.MF_TUNE_TILES, tiles)
            u, du = u0.copy(), np.empty_like(u0)
            ctx.rhs_host(0.0, u, du, prec)
            assert (ctx.tile_info()["tiles_a"], ctx.tile_info()["tiles_b"]) == (tiles, 0)
            out.append(du)
        assert np.isfinite(out[0]).all() and np.array_equal(out[0], out[1])


def test_halos_in_ranges():
    """One variable and more tiles than one range of the temporary ids holds (682
    for the stencils, 512 for the transposed entries)."""
    rng = np.random.default_rng(12)
    n = 682 * 256 + 4001
    ctx = L.Context(0)
    ctx.set_equations(L.MF_EQ_ADVECTION_2D, 1.0, 0.5)
    ctx.set_points(rng.random(n), rng.random(n))
    idx = ctx.knn(5)[0]
    operators(ctx, idx, rng)
    u, lam = rng.standard_normal((1, n)), rng.standard_normal((1, n))
    out = []
    for tiles in (0, 1):
        ctx.set_tuning(L.MF_TUNE_TILES, tiles)
        ctx.upload(L.MF_BUF_U, u)
        ctx.upload(L.MF_BUF_AUX0, lam)
        ctx.rhs_vjp(0.0)
        ctx.rhs(0.0)
        out.append((ctx.download(L.MF_BUF_AUX1), ctx.download(L.MF_BUF_DU)))
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])
    ti = ctx.tile_info()
    assert ti["tiles_a"] and ti["tiles_b"]
    assert (ti["halo_a_total"], ti["halo_b_total"], ti["halo_a_max"], ti["halo_b_max"],
            ti["b_entries_padded"]) == expected(idx, ctx.node_order())
