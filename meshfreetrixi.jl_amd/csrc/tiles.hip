// LDS tiles of the stencil operators (built once per stencil / operator).
//
// The neighbour gathers of the rhs! kernels touch one cache line per lane
// per load: a wavefront's 64 lanes read 64 scattered 32- or 64-byte node
// records.  With the nodes in Morton order, the 256 nodes of a workgroup
// form a compact patch whose stencils reach only ~2x as many distinct
// nodes.  Each workgroup therefore loads that halo once into LDS (runs of
// consecutive node records) and the stencil loops read LDS through 16-bit
// halo positions stored in place of the 32-bit node indices.
//
// Phase A (flux divergence, sources, viscosity phase A): halo = the union
// of the tile's stencils; positions, and copies of the operators, in the
// tile-major layout (tm_pos: a tile's K slots back to back), so that one
// tile's entries of an array share a few pages: with the slot-major layout
// (slot stride N) a tile touched K pages per array, and on multi-million
// node sets the address translation (UTCL2 busy 91% of the time) limited
// the stencil kernel.
// Phase B (transposed gathers D^T G, lap^T L): rows of the tile sorted by their
// transposed degree (long rows first) so that the 64 rows of a wavefront
// have similar lengths, stored SELL-64 per wavefront; entries of a row in
// ascending caller index (the reference's CSC order); halo = the union of
// the rows' entries.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <type_traits>
#include <vector>

#include "mf_device.h"

namespace mf {

constexpr int kTile = 256;
constexpr int kSlicesPerTile = kTile / kSellC;  // 4
constexpr size_t kTileLdsBytes = 48 * 1024;     // largest phase-A halo staged in LDS
constexpr size_t kTileLdsBytesB = 64 * 1024;    // phase B (records of G and lap u)

void free_tiles_b(mf_ctx* c)
{
    dfree(c->d_hb_off);
    dfree(c->d_hb_ids);
    dfree(c->d_sb_off);
    dfree(c->d_sb_w);
    dfree(c->d_rowb);
    dfree(c->d_lb);
    dfree(c->d_twb);
    dfree(c->d_twb32);
    dfree(c->d_tb_src);
    dfree(c->d_twl);
    dfree(c->d_twl32);
    c->d_tb_src = nullptr;
    c->d_twl = nullptr;
    c->d_twl32 = nullptr;
    c->lap_tb = false;
    c->tiles_b_rec = 0;
    c->d_hb_off = c->d_sb_off = nullptr;
    c->d_hb_ids = c->d_sb_w = nullptr;
    c->d_lb = nullptr;
    c->d_rowb = nullptr;
    c->d_twb = nullptr;
    c->d_twb32 = nullptr;
    c->tiles_b = false;
    c->tried_b = false;
    c->hb_max = 0;
}

static void free_tile_ops(mf_ctx* c)
{
    dfree(c->d_wxy_t);
    dfree(c->d_wxy32_t);
    dfree(c->d_hv_t);
    dfree(c->d_hv32_t);
    dfree(c->d_lap_t);
    dfree(c->d_lap32_t);
    dfree(c->d_wx_s_t);
    dfree(c->d_wy_s_t);
    dfree(c->d_hv_s_t);
    dfree(c->d_lap_s_t);
    c->d_wxy_t = nullptr;
    c->d_wxy32_t = nullptr;
    c->d_hv_t = c->d_lap_t = c->d_wx_s_t = c->d_wy_s_t = c->d_hv_s_t = c->d_lap_s_t = nullptr;
    c->d_hv32_t = c->d_lap32_t = nullptr;
    c->tm_dirty = true;
}

void free_tiles(mf_ctx* c)
{
    free_tiles_b(c);
    free_tile_ops(c);
    dfree(c->d_ha_off);
    dfree(c->d_ha_ids);
    dfree(c->d_la);
    dfree(c->d_la_s);
    c->d_ha_off = nullptr;
    c->d_ha_ids = nullptr;
    c->d_la = nullptr;
    c->d_la_s = nullptr;
    c->tiles_a = false;
    c->tried_a = false;
    c->n_tiles = 0;
    c->ha_max = 0;
}

// (Dx, Dy) of each transposed entry from the forward operator: src[e] is
// the slot-major position s*N + j of the entry, or -1 for padding.
__global__ void k_fill_tile_weights(int64_t n, const int64_t* src, const double2* wxy, double2* tw, float2* tw32)
{
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= n) return;
    const int64_t q = src[e];
    const double2 w = q >= 0 ? wxy[q] : make_double2(0.0, 0.0);
    tw[e] = w;
    tw32[e] = make_float2((float)w.x, (float)w.y);
}

// Slot-major (s N + i) operator array to the tile-major layout (tm_pos);
// the padding entries of the last tile are zero.
template <class T>
__global__ void k_to_tile_major(int64_t N, int K, int64_t n_out, const T* src, T* dst)
{
    const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= n_out) return;
    const int64_t r = q % kTile, ts = q / kTile;  // ts = t K + s
    const int64_t t = ts / K, sl = ts % K;
    const int64_t i = t * kTile + r;
    dst[q] = i < N ? src[sl * N + i] : T{};
}

// The tile-major copies of every operator array present, after the tiles
// are built and whenever an operator changed since the last copy.
int ensure_tile_ops(mf_ctx* c)
{
    if (!c->tiles_a || !c->tm_dirty) return MF_OK;
    const int64_t n_out = c->n_tiles * (int64_t)c->k * kTile;
    int rc;
    auto copy = [&](auto* src, auto** dst) -> int {
        using T = std::remove_pointer_t<decltype(src)>;
        if (!src) return MF_OK;
        if (!*dst && (rc = dalloc(c, dst, (size_t)n_out))) return rc;
        hipLaunchKernelGGL(k_to_tile_major<T>, dim3((unsigned)((n_out + 255) / 256)), dim3(256), 0, c->stream,
                           c->N, c->k, n_out, (const T*)src, *dst);
        MF_HIP(c, hipGetLastError());
        return MF_OK;
    };
    if ((rc = copy(c->d_wxy, &c->d_wxy_t)) || (rc = copy(c->d_wxy32, &c->d_wxy32_t)) ||
        (rc = copy(c->d_hv, &c->d_hv_t)) || (rc = copy(c->d_hv32, &c->d_hv32_t)) ||
        (rc = copy(c->d_lap, &c->d_lap_t)) || (rc = copy(c->d_lap32, &c->d_lap32_t)) ||
        (rc = copy(c->d_wx_s, &c->d_wx_s_t)) || (rc = copy(c->d_wy_s, &c->d_wy_s_t)) ||
        (rc = copy(c->d_hv_s, &c->d_hv_s_t)) || (rc = copy(c->d_lap_s, &c->d_lap_s_t)))
        return rc;
    c->tm_dirty = false;
    return MF_OK;
}

template <class T>
static int upload(mf_ctx* c, T** dst, const std::vector<T>& v)
{
    int rc = dalloc(c, dst, v.size());
    if (rc) return rc;
    if (!v.empty())
        MF_HIP(c, hipMemcpyAsync(*dst, v.data(), sizeof(T) * v.size(), hipMemcpyHostToDevice, c->stream));
    return MF_OK;
}

// ------------------------------------------------- halos of the tiles
// One workgroup per tile collects the distinct node ids of its entries in an
// LDS hash table (open addressing), sorts the table (the empty slots last)
// and looks every entry's position up in it by bisection.  Built on the
// host, the tiles of 62,500 nodes took 70 ms, most of a new cloud's set-up
// (bound by one core's cache misses); k_halo_a and k_halo_b take 0.11 ms each.
constexpr int32_t kNoId = INT32_MAX;

__device__ __forceinline__ void halo_clear(int32_t* tab, int T, int* cnt)
{
    for (int q = threadIdx.x; q < T; q += kTile) tab[q] = kNoId;
    if (threadIdx.x == 0) *cnt = 0;
    __syncthreads();
}

// Inserts id; at most cap + kTile ids enter the table (T above that, so a
// probe always ends at an empty slot or the id).
__device__ __forceinline__ void halo_insert(int32_t* tab, int T, int cap, int* cnt, int32_t id)
{
    uint32_t h = ((uint32_t)id * 2654435761u) >> (__clz(T) + 1);
    for (;;) {
        int32_t cur = reinterpret_cast<volatile int32_t*>(tab)[h];
        if (cur == id) return;
        if (cur == kNoId) {
            if (*reinterpret_cast<volatile int*>(cnt) > cap) return;
            cur = atomicCAS(&tab[h], kNoId, id);
            if (cur == id) return;
            if (cur == kNoId) {
                atomicAdd(cnt, 1);
                return;
            }
        }
        h = (h + 1) & (uint32_t)(T - 1);
    }
}

// Bitonic sort of the whole table, ascending.
__device__ __forceinline__ void halo_sort(int32_t* tab, int T)
{
    for (int w = 2; w <= T; w <<= 1)
        for (int d = w >> 1; d > 0; d >>= 1) {
            for (int p = threadIdx.x; p < T / 2; p += kTile) {
                const int lo = 2 * p - (p & (d - 1));  // bit d clear
                const int32_t x = tab[lo], y = tab[lo + d];
                if ((x > y) == ((lo & w) == 0)) {
                    tab[lo] = y;
                    tab[lo + d] = x;
                }
            }
            __syncthreads();
        }
}

__device__ __forceinline__ uint16_t halo_pos(const int32_t* tab, int n, int32_t id)
{
    int lo = 0, hi = n - 1;
    while (lo < hi) {
        const int m = (lo + hi) >> 1;
        if (tab[m] < id)
            lo = m + 1;
        else
            hi = m;
    }
    return (uint16_t)lo;
}

// The block's tile's ids (at blockIdx.x cap) and their number (above cap: the
// halo does not fit).
__device__ __forceinline__ int halo_finish(int32_t* tab, int T, int cap, const int* cnt, int32_t* ids, int32_t* count)
{
    __syncthreads();
    const int n = *cnt;
    if (threadIdx.x == 0) count[blockIdx.x] = n;
    if (n > cap) return -1;
    halo_sort(tab, T);
    for (int q = threadIdx.x; q < n; q += kTile) ids[(int64_t)blockIdx.x * cap + q] = tab[q];
    return n;
}

// Phase A: the union of the tile's stencils, and the tile-major positions of
// the entries of both stencil copies (0 past the last node).  Tiles t0 on.
__global__ __launch_bounds__(kTile) void k_halo_a(int64_t t0, int64_t N, int K, const int32_t* idx, const int32_t* idx_s,
                                                  int T, int cap, int32_t* ids, int32_t* count, uint16_t* la,
                                                  uint16_t* la_s)
{
    extern __shared__ int32_t tab[];
    __shared__ int cnt;
    const int64_t t = t0 + blockIdx.x, i = t * kTile + threadIdx.x;
    halo_clear(tab, T, &cnt);
    if (i < N)
        for (int s = 0; s < K; ++s) halo_insert(tab, T, cap, &cnt, idx[(int64_t)s * N + i]);
    const int n = halo_finish(tab, T, cap, &cnt, ids, count);
    if (n < 0) return;
    for (int s = 0; s < K; ++s) {
        const int64_t q = (t * K + s) * kTile + threadIdx.x;
        la[q] = i < N ? halo_pos(tab, n, idx[(int64_t)s * N + i]) : 0;
        la_s[q] = i < N ? halo_pos(tab, n, idx_s[(int64_t)s * N + i]) : 0;
    }
}

// Phase B: the tile's rows by transposed degree, longest first (ties by
// node; rows past the last node have degree 0), and the longest row of each
// 64-row slice.
__global__ __launch_bounds__(kTile) void k_rows_b(int64_t N, const int32_t* deg, uint8_t* rowb, int32_t* sw)
{
    __shared__ int32_t d[kTile], s[kTile];
    const int64_t t = blockIdx.x, i = t * kTile + threadIdx.x;
    const int r = threadIdx.x, mine = i < N ? deg[i] : 0;
    d[r] = mine;
    __syncthreads();
    int at = 0;
    for (int q = 0; q < kTile; ++q) at += d[q] > mine || (d[q] == mine && q < r);
    rowb[t * kTile + at] = (uint8_t)r;
    s[at] = mine;
    __syncthreads();
    if (r < kSlicesPerTile) sw[t * kSlicesPerTile + r] = s[r * kSellC];  // sorted: the slice's first row
}

// The union of the rows' entries, and each entry's halo position and source
// in the slice layout (rows of the global transpose, already in ascending
// caller index).  Tiles t0 on.
__global__ __launch_bounds__(kTile) void k_halo_b(int64_t t0, int64_t N, const int32_t* deg, const int64_t* toff,
                                                  const int32_t* trow, const int64_t* tsrc, const uint8_t* rowb,
                                                  const int64_t* soff, const int32_t* sw, int T, int cap, int32_t* ids,
                                                  int32_t* count, uint16_t* lb, int64_t* src)
{
    extern __shared__ int32_t tab[];
    __shared__ int cnt;
    const int64_t t = t0 + blockIdx.x;
    halo_clear(tab, T, &cnt);
    {
        const int64_t i = t * kTile + threadIdx.x;
        if (i < N) {
            const int64_t b = toff[i / kSellC] + i % kSellC;
            const int n = deg[i];
            for (int e = 0; e < n; ++e) halo_insert(tab, T, cap, &cnt, trow[b + (int64_t)e * kSellC]);
        }
    }
    const int n = halo_finish(tab, T, cap, &cnt, ids, count);
    if (n < 0) return;
    const int p = threadIdx.x;
    const int64_t i = t * kTile + rowb[t * kTile + p];
    const int64_t sl = t * kSlicesPerTile + p / kSellC, o = soff[sl] + p % kSellC;
    const int W = sw[sl], d = i < N ? deg[i] : 0;
    const int64_t b = i < N ? toff[i / kSellC] + i % kSellC : 0;
    for (int e = 0; e < W; ++e) {
        const int64_t at = o + (int64_t)e * kSellC;
        lb[at] = e < d ? halo_pos(tab, n, trow[b + (int64_t)e * kSellC]) : 0;
        src[at] = e < d ? tsrc[b + (int64_t)e * kSellC] : -1;
    }
}

// ids[off[t] - off[0] + q] = tmp[t cap + q]
__global__ void k_halo_pack(const int32_t* tmp, int cap, const int64_t* off, int32_t* ids)
{
    const int64_t t = blockIdx.x, o = off[t] - off[0];
    const int n = (int)(off[t + 1] - off[t]);
    for (int q = threadIdx.x; q < n; q += blockDim.x) ids[o + q] = tmp[t * cap + q];
}

static int halo_table(int cap)
{
    int T = 512;
    while (T < cap + 2 * kTile) T *= 2;
    return T;
}

// Before its ids are packed a tile has room for cap of them, 3 to 24 times what
// its halo takes: the tiles go through it in ranges of this size (with room for
// all of them at once one variable took 96 bytes per node of the cloud).
constexpr size_t kHaloTempBytes = (size_t)16 << 20;

// The halos by launch(t0, n, ids, count) of the n tiles from t0 on: offsets, the
// packed ids and the largest size; fits = false if some tile's halo has more
// than cap ids.
template <class Launch>
static int collect_halos(mf_ctx* c, int64_t nt, int cap, Launch launch, int64_t** off, int32_t** ids, int* hmax,
                         int64_t* total, bool* fits)
{
    const int64_t range = std::min<int64_t>(nt, (int64_t)(kHaloTempBytes / (sizeof(int32_t) * cap)));
    int32_t *tmp = nullptr, *count = nullptr;
    std::vector<int32_t> size(range);
    std::vector<int64_t> o(nt + 1, 0);
    std::vector<int32_t*> part;  // each range's packed ids
    part.reserve((size_t)((nt + range - 1) / range));
    *hmax = 0;
    *fits = false;
    auto body = [&]() -> int {
        int rc;
        if ((rc = dalloc(c, &tmp, (size_t)range * cap)) || (rc = dalloc(c, &count, (size_t)range)) ||
            (rc = dalloc(c, off, (size_t)nt + 1)))
            return rc;
        for (int64_t t0 = 0; t0 < nt; t0 += range) {
            const int64_t n = std::min(range, nt - t0);
            launch(t0, (unsigned)n, tmp, count);
            MF_HIP(c, hipGetLastError());
            MF_HIP(c, hipMemcpyAsync(size.data(), count, sizeof(int32_t) * n, hipMemcpyDeviceToHost, c->stream));
            MF_HIP(c, hipStreamSynchronize(c->stream));
            for (int64_t t = 0; t < n; ++t) {
                *hmax = std::max<int>(*hmax, size[t]);
                o[t0 + t + 1] = o[t0 + t] + size[t];
            }
            if (*hmax > cap) return MF_OK;
            MF_HIP(c, hipMemcpyAsync(*off + t0, o.data() + t0, sizeof(int64_t) * (n + 1), hipMemcpyHostToDevice,
                                     c->stream));
            int32_t* p = nullptr;
            if ((rc = dalloc(c, &p, (size_t)(o[t0 + n] - o[t0])))) return rc;
            part.push_back(p);
            hipLaunchKernelGGL(k_halo_pack, dim3((unsigned)n), dim3(kTile), 0, c->stream, tmp, cap, *off + t0, p);
            MF_HIP(c, hipGetLastError());
        }
        *total = o[nt];
        if (part.size() == 1) {
            *ids = part[0];
            part.clear();
        } else {
            if ((rc = dalloc(c, ids, (size_t)o[nt]))) return rc;
            for (size_t q = 0; q < part.size(); ++q) {
                const int64_t t0 = (int64_t)q * range, n = std::min(range, nt - t0);
                MF_HIP(c, hipMemcpyAsync(*ids + o[t0], part[q], sizeof(int32_t) * (o[t0 + n] - o[t0]),
                                         hipMemcpyDeviceToDevice, c->stream));
            }
        }
        *fits = true;
        return MF_OK;
    };
    int rc = body();
    const hipError_t e = hipStreamSynchronize(c->stream);  // nothing in flight reads the temporaries
    if (rc == MF_OK && e != hipSuccess) rc = hip_fail(c, e, "hipStreamSynchronize");
    dfree(tmp);
    dfree(count);
    for (int32_t* p : part) dfree(p);
    return rc;
}

static int build_tiles_a(mf_ctx* c, int64_t nt)
{
    const int64_t N = c->N;
    const int K = c->k;
    // phase A halo records: 6 doubles per node for Euler (state, v1, v2)
    const int rec = c->nvar == 4 ? 6 : c->nvar;
    const int cap = (int)(kTileLdsBytes / (rec * sizeof(double)));
    const int T = halo_table(cap);
    const size_t n_la = (size_t)nt * K * kTile;
    int rc;
    if ((rc = dalloc(c, &c->d_la, n_la)) || (rc = dalloc(c, &c->d_la_s, n_la))) return rc;
    auto launch = [&](int64_t t0, unsigned n, int32_t* ids, int32_t* count) {
        hipLaunchKernelGGL(k_halo_a, dim3(n), dim3(kTile), sizeof(int32_t) * T, c->stream, t0, N, K, c->d_idx, c->d_idx_s,
                           T, cap, ids, count, c->d_la, c->d_la_s);
    };
    bool fits;
    int hmax;
    if ((rc = collect_halos(c, nt, cap, launch, &c->d_ha_off, &c->d_ha_ids, &hmax, &c->ha_total, &fits))) return rc;
    if (!fits) {  // global-memory kernels
        dfree(c->d_la);
        dfree(c->d_la_s);
        c->d_la = c->d_la_s = nullptr;
        return MF_OK;
    }
    c->n_tiles = nt;
    c->ha_max = hmax;
    c->tiles_a = true;
    return MF_OK;
}

static int build_tiles_b(mf_ctx* c, int64_t nt, int rec_b)
{
    const int64_t N = c->N;
    const int cap = (int)(kTileLdsBytesB / (rec_b * sizeof(double)));
    const int T = halo_table(cap);
    const int64_t nsl = nt * kSlicesPerTile;
    int rc;
    if ((rc = dalloc(c, &c->d_rowb, (size_t)nt * kTile)) || (rc = dalloc(c, &c->d_sb_w, (size_t)nsl))) return rc;
    hipLaunchKernelGGL(k_rows_b, dim3((unsigned)nt), dim3(kTile), 0, c->stream, N, c->d_tdeg, c->d_rowb, c->d_sb_w);
    MF_HIP(c, hipGetLastError());
    std::vector<int32_t> sw(nsl);
    MF_HIP(c, hipMemcpyAsync(sw.data(), c->d_sb_w, sizeof(int32_t) * nsl, hipMemcpyDeviceToHost, c->stream));
    MF_HIP(c, hipStreamSynchronize(c->stream));
    std::vector<int64_t> soff(nsl + 1, 0);
    for (int64_t s = 0; s < nsl; ++s) soff[s + 1] = soff[s] + (int64_t)sw[s] * kSellC;
    const int64_t ne = soff[nsl];
    if ((rc = upload(c, &c->d_sb_off, soff)) || (rc = dalloc(c, &c->d_lb, (size_t)ne)) ||
        (rc = dalloc(c, &c->d_tb_src, (size_t)ne)))
        return rc;
    auto launch = [&](int64_t t0, unsigned n, int32_t* ids, int32_t* count) {
        hipLaunchKernelGGL(k_halo_b, dim3(n), dim3(kTile), sizeof(int32_t) * T, c->stream, t0, N, c->d_tdeg, c->d_sell_off,
                           c->d_trow, c->d_tsrc, c->d_rowb, c->d_sb_off, c->d_sb_w, T, cap, ids, count, c->d_lb,
                           c->d_tb_src);
    };
    bool fits;
    int hmax;
    if ((rc = collect_halos(c, nt, cap, launch, &c->d_hb_off, &c->d_hb_ids, &hmax, &c->hb_total, &fits))) return rc;
    if (!fits) return MF_OK;  // global-memory transposed gather
    if ((rc = dalloc(c, &c->d_twb, (size_t)ne)) || (rc = dalloc(c, &c->d_twb32, (size_t)ne))) return rc;
    hipLaunchKernelGGL(k_fill_tile_weights, dim3((unsigned)((ne + 255) / 256)), dim3(256), 0, c->stream, ne,
                       c->d_tb_src, c->d_wxy, c->d_twb, c->d_twb32);
    MF_HIP(c, hipGetLastError());
    MF_HIP(c, hipStreamSynchronize(c->stream));
    c->hb_max = hmax;
    c->nb_entries = ne;
    c->tiles_b = true;
    return MF_OK;
}

// rec_b: doubles per phase-B halo record (G: 2 nvar, L: nvar), which
// decides whether a tile's phase-B halo fits in LDS.  Phase B needs the
// global transpose.
int build_tiles(mf_ctx* c, bool want_b, int rec_b)
{
    const int64_t nt = (c->N + kTile - 1) / kTile;
    if (!c->tried_a) {
        free_tiles(c);
        c->tried_a = true;
        const int rc = build_tiles_a(c, nt);
        if (rc) return rc;
    }
    if (!want_b || !c->tiles_a || c->tried_b) return MF_OK;
    if (!c->have_T) return fail(c, MF_ERR_STATE, "tiles: no transposed operator");
    free_tiles_b(c);
    c->tried_b = true;
    c->tiles_b_rec = rec_b;
    return build_tiles_b(c, nt, rec_b);
}

}  // namespace mf
