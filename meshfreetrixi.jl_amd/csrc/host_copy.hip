// Transfers between the caller's arrays and the device through pinned chunks.
//
// hipMemcpy on pageable memory takes one call per field (12 of them, 3.8 us
// of device time each and as much again between them, around a small
// rhs!) and moves large arrays at about 10 GB/s, bound by one thread copying
// into (and faulting in) the caller's pages; the link does 57 GB/s.  Here
// small states cross in one kernel that reads or writes a pinned chunk
// directly, and large transfers run chunk by chunk, several threads copying
// between the chunks and the caller's pages while the link streams.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <exception>
#include <mutex>
#include <thread>
#include <vector>

#include "mf_device.h"

namespace mf {

constexpr size_t kChunkBytes = (size_t)2 << 20;
constexpr int kMaxChunks = 16;              // of the process, whatever its contexts
constexpr int kCopyThreads = 8;             // per large transfer, at most one per processor
constexpr size_t kDirectBytes = (size_t)1 << 20;   // states up to this size: read or written by the kernel
// Transfers by several threads, from these sizes.  To the host they also fault
// the caller's pages in, which one thread does at about 15 GB/s; towards the
// device the runtime reads pageable memory at 30 GB/s by itself and the threads
// gain only once they run for a while (us, runtime / threads, up: 8 MB 268 / 330,
// 17 MB 502 / 580, 34 MB 982 / 1039, 46 MB 1657 / 1374, 67 MB 2237 / 1900; down: 8
// MB 489 / 324, 17 MB 942 / 567, 67 MB 3755 / 1852).
constexpr size_t kThreadBytesUp = (size_t)40 << 20, kThreadBytesDown = (size_t)4 << 20;
constexpr size_t kGrowBytes = (size_t)8 << 20;     // allocating chunks for them from this size

// The process's pinned chunks: allocated as transfers need them, at most
// kMaxChunks, kept while any context lives and freed with the last one.  A
// transfer that finds too few copies the pageable memory itself: allocating
// a chunk takes about as long as that copy takes for a few MB.
struct Chunk {
    char* host = nullptr;
    hipEvent_t done = nullptr;  // of device `device`
    int device = -1;
};

static std::mutex g_pool_mu;
static std::vector<Chunk> g_pool_free;
static int g_pool_total = 0;
static int g_pool_users = 0;

void pinned_pool_open()
{
    std::lock_guard<std::mutex> lock(g_pool_mu);
    ++g_pool_users;
}

void pinned_pool_close()
{
    std::lock_guard<std::mutex> lock(g_pool_mu);
    if (--g_pool_users > 0) return;
    for (Chunk& k : g_pool_free) {
        if (k.done) (void)hipEventDestroy(k.done);
        (void)hipHostFree(k.host);
    }
    g_pool_total -= (int)g_pool_free.size();
    g_pool_free.clear();
}

// Borrowed chunks, returned when it goes out of scope; the borrower has
// waited for every transfer by then.
struct Borrowed {
    std::vector<Chunk> c;
    Borrowed(mf_ctx* ctx, int want, bool grow)
    {
        c.reserve(want);
        std::lock_guard<std::mutex> lock(g_pool_mu);
        g_pool_free.reserve(kMaxChunks);
        while ((int)c.size() < want) {
            Chunk k;
            if (!g_pool_free.empty()) {
                k = g_pool_free.back();
                g_pool_free.pop_back();
            } else {
                void* p = nullptr;
                if (!grow || g_pool_total >= kMaxChunks) break;
                if (hipHostMalloc(&p, kChunkBytes, hipHostMallocPortable) != hipSuccess) {
                    (void)hipGetLastError();
                    break;
                }
                k.host = static_cast<char*>(p);
                ++g_pool_total;
            }
            if (k.device != ctx->device) {  // an event belongs to the device it was created on
                if (k.done) (void)hipEventDestroy(k.done);
                k.device = -1;
                k.done = nullptr;
                if (hipEventCreateWithFlags(&k.done, hipEventDisableTiming) != hipSuccess) {
                    (void)hipGetLastError();
                    k.done = nullptr;
                    g_pool_free.push_back(k);
                    break;
                }
                k.device = ctx->device;
            }
            c.push_back(k);
        }
    }
    ~Borrowed()
    {
        std::lock_guard<std::mutex> lock(g_pool_mu);
        for (const Chunk& k : c) g_pool_free.push_back(k);
    }
    Borrowed(const Borrowed&) = delete;
    Borrowed& operator=(const Borrowed&) = delete;
};

// A contiguous device range against `fields` of `field_bytes` each, back to
// back: copies the part [at, at + n) of it between `fields` and p.
static void copy_part(const HostFields& f, size_t at, size_t n, char* p, bool to_host)
{
    while (n) {
        const size_t v = at / f.field_bytes, o = at % f.field_bytes, m = std::min(n, f.field_bytes - o);
        char* h = static_cast<char*>(f.fields[v]) + o;
        if (to_host)
            std::memcpy(h, p, m);
        else
            std::memcpy(p, h, m);
        at += m;
        p += m;
        n -= m;
    }
}

// Chunks first, first + step, ... of the range through one pinned chunk.
static hipError_t copy_chunks(int device, hipStream_t stream, const HostFields& f, char* d, size_t bytes, size_t first,
                              size_t step, const Chunk& k, bool to_host)
{
    hipError_t e = hipSetDevice(device);
    for (size_t q = first; e == hipSuccess && q * kChunkBytes < bytes; q += step) {
        const size_t at = q * kChunkBytes, n = std::min(kChunkBytes, bytes - at);
        if (!to_host) copy_part(f, at, n, k.host, false);
        e = to_host ? hipMemcpyAsync(k.host, d + at, n, hipMemcpyDeviceToHost, stream)
                    : hipMemcpyAsync(d + at, k.host, n, hipMemcpyHostToDevice, stream);
        if (e == hipSuccess) e = hipEventRecord(k.done, stream);
        if (e == hipSuccess) e = hipEventSynchronize(k.done);
        if (to_host && e == hipSuccess) copy_part(f, at, n, k.host, true);
    }
    return e;
}

// Whether some field is memory that the runtime knows (pinned, managed): it is
// copied from or to directly, at the link's rate, which the pinned chunks would
// only slow down (17 MB 374 us against 573).
static bool known_memory(const HostFields& f)
{
    for (int v = 0; v < f.count; ++v) {
        hipPointerAttribute_t at;
        if (hipPointerGetAttributes(&at, f.fields[v]) != hipSuccess)
            (void)hipGetLastError();
        else if (at.type != hipMemoryTypeUnregistered)
            return true;
    }
    return false;
}

// The range [d, d + count field_bytes) to or from the fields; the fields are
// complete on return, towards the device the stream may still be reading them.
int copy_fields(mf_ctx* c, void* d, const HostFields& f, bool to_host)
{
    const size_t bytes = f.field_bytes * (size_t)f.count;
    if (bytes == 0) return MF_OK;
    int want = 0;
    if (bytes >= (to_host ? kThreadBytesDown : kThreadBytesUp) && !known_memory(f))
        want = (int)std::min<size_t>((bytes + kChunkBytes - 1) / kChunkBytes,
                                     std::min<size_t>(kCopyThreads, std::thread::hardware_concurrency()));
    const Borrowed b(c, want, bytes >= kGrowBytes);
    char* dp = static_cast<char*>(d);
    const int T = (int)b.c.size();
    if (T < 2) {
        for (int v = 0; v < f.count; ++v)
            MF_HIP(c, to_host ? hipMemcpyAsync(f.fields[v], dp + v * f.field_bytes, f.field_bytes,
                                               hipMemcpyDeviceToHost, c->stream)
                              : hipMemcpyAsync(dp + v * f.field_bytes, f.fields[v], f.field_bytes,
                                               hipMemcpyHostToDevice, c->stream));
        if (to_host) MF_HIP(c, hipStreamSynchronize(c->stream));
        return MF_OK;
    }
    // this thread's own share, and one more thread per further chunk; where
    // no thread can be started its share stays here
    std::vector<hipError_t> err(T, hipSuccess);
    std::vector<std::thread> th;
    th.reserve(T);
    std::vector<int> mine(1, 0);
    mine.reserve(T);
    for (int t = 1; t < T; ++t) {
        try {
            th.emplace_back([&, t] {
                err[t] = copy_chunks(c->device, c->stream, f, dp, bytes, t, T, b.c[t], to_host);
            });
        } catch (const std::exception&) {  // no thread or no memory for one
            mine.push_back(t);
        }
    }
    for (int t : mine) err[t] = copy_chunks(c->device, c->stream, f, dp, bytes, t, T, b.c[t], to_host);
    for (std::thread& x : th) x.join();
    for (hipError_t e : err)
        if (e != hipSuccess) {
            (void)hipStreamSynchronize(c->stream);  // the chunks go back to the pool
            return hip_fail(c, e, "copy between host and device");
        }
    return MF_OK;
}

// One array of `bytes` bytes.
int copy_array(mf_ctx* c, void* d, const void* h, size_t bytes, bool to_host)
{
    HostFields f;
    f.count = 1;
    f.field_bytes = bytes;
    f.fields[0] = const_cast<void*>(h);
    return copy_fields(c, d, f, to_host);
}

// aos[p V + v] = field v of the caller's node uid[p] and back, the fields
// back to back.  For states of up to kDirectBytes the fields are a pinned
// chunk.
int upload_state(mf_ctx* c, double* d_dst, const double* const* fields)
{
    HostFields f;
    f.count = c->nvar;
    f.field_bytes = sizeof(double) * (size_t)c->N;
    for (int v = 0; v < c->nvar; ++v) f.fields[v] = const_cast<double*>(fields[v]);
    const size_t bytes = f.field_bytes * (size_t)c->nvar;
    int rc;
    if (bytes <= kDirectBytes) {
        const Borrowed b(c, 1, true);
        if (!b.c.empty()) {
            copy_part(f, 0, bytes, b.c[0].host, false);
            if ((rc = launch_soa_to_aos(c, reinterpret_cast<const double*>(b.c[0].host), d_dst, true))) return rc;
            MF_HIP(c, hipStreamSynchronize(c->stream));
            return MF_OK;
        }
    }
    rc = copy_fields(c, c->d_T, f, false);
    if (!rc) rc = launch_soa_to_aos(c, c->d_T, d_dst, false);
    if (rc) (void)hipStreamSynchronize(c->stream);  // the caller's arrays are read no more
    return rc;
}

int download_state(mf_ctx* c, const double* d_src, double* const* fields)
{
    HostFields f;
    f.count = c->nvar;
    f.field_bytes = sizeof(double) * (size_t)c->N;
    for (int v = 0; v < c->nvar; ++v) f.fields[v] = fields[v];
    const size_t bytes = f.field_bytes * (size_t)c->nvar;
    int rc;
    if (bytes <= kDirectBytes) {
        const Borrowed b(c, 1, true);
        if (!b.c.empty()) {
            rc = launch_aos_to_soa(c, d_src, reinterpret_cast<double*>(b.c[0].host));
            const hipError_t e = hipStreamSynchronize(c->stream);
            if (rc) return rc;
            if (e != hipSuccess) return hip_fail(c, e, "hipStreamSynchronize");
            copy_part(f, 0, bytes, b.c[0].host, true);
            return MF_OK;
        }
    }
    if ((rc = launch_aos_to_soa(c, d_src, c->d_T))) return rc;
    return copy_fields(c, c->d_T, f, true);
}

// u in, rhs!, du and u out, of states up to kDirectBytes: one wait for all.
// `run` enqueues the rhs!; *done tells whether this way was taken.
int rhs_through_pinned(mf_ctx* c, double* d_u, double* d_du, double* const* u, double* const* du,
                       const std::function<int()>& run, bool* done)
{
    *done = false;
    const size_t field = sizeof(double) * (size_t)c->N, bytes = field * (size_t)c->nvar;
    if (bytes > kDirectBytes) return MF_OK;
    const Borrowed b(c, 1, true);
    if (b.c.empty()) return MF_OK;
    *done = true;
    HostFields f;
    f.count = c->nvar;
    f.field_bytes = field;
    for (int v = 0; v < c->nvar; ++v) f.fields[v] = u[v];
    // the input and u's output share a half of the chunk, du has the other
    char *pu = b.c[0].host, *pdu = pu + kDirectBytes;
    copy_part(f, 0, bytes, pu, false);
    int rc = launch_soa_to_aos(c, reinterpret_cast<const double*>(pu), d_u, true);
    if (!rc) rc = run();
    if (!rc) rc = launch_aos_to_soa(c, d_du, reinterpret_cast<double*>(pdu));
    if (!rc) rc = launch_aos_to_soa(c, d_u, reinterpret_cast<double*>(pu));
    const hipError_t e = hipStreamSynchronize(c->stream);
    if (rc) return rc;
    if (e != hipSuccess) return hip_fail(c, e, "hipStreamSynchronize");
    HostFields fd = f;
    for (int v = 0; v < c->nvar; ++v) fd.fields[v] = du[v];
    copy_part(fd, 0, bytes, pdu, true);
    copy_part(f, 0, bytes, pu, true);
    return MF_OK;
}

}  // namespace mf
