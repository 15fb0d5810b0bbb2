// Runtime pieces of libmr_aha_c: backend identity, HIP error hook and the
// per-device cache of FFT twiddle tables.

#include "mr_hip.hpp"

#include <cmath>
#include <map>
#include <mutex>
#include <tuple>

void mr_backend_clear_error() { (void)hipGetLastError(); }

// "cuda" is the value that makes the reference's bindings treat every array
// argument as a device pointer (python/mr_aha/_lib.py:700-715); this library
// follows that device-pointer ABI on HIP devices.
extern "C" MR_EXPORT const char *mr_backend(void) { return "cuda"; }

namespace {
std::mutex g_tw_mu;
std::map<std::tuple<int, int, int>, void *> g_tw;  // (device, n, bytes per real) -> table
}  // namespace

template <typename R> int mr_fft_get(int n, mr_fft_len<R> *out)
{
    using V = typename cvec<R>::T;
    MR_REQUIRE(n >= 1, "FFT length %d must be >= 1", n);
    const size_t lds = ((size_t)n + 2 * (size_t)mr_fft_ns(n)) * sizeof(V);
    if (lds > 64 * 1024)
        MR_FAIL(MR_ERR_UNSUPPORTED, "FFT length %d exceeds the single-pencil LDS limit", n);
    out->n = n;
    out->nst = mr_fft_factor(n, out->radix);
    if (out->nst < 0) MR_FAIL(MR_ERR_UNSUPPORTED, "FFT length %d has too many factors", n);
    int dev = 0;
    MR_HIP_CHECK(hipGetDevice(&dev));
    std::lock_guard<std::mutex> lk(g_tw_mu);
    auto key = std::make_tuple(dev, n, (int)sizeof(R));
    auto it = g_tw.find(key);
    if (it == g_tw.end()) {
        std::vector<V> h(n);
        for (int q = 0; q < n; ++q) {
            // exact quadrant values, long double elsewhere
            const long double a = -2.0L * 3.14159265358979323846264338327950288L * q / n;
            h[q].x = (R)cosl(a);
            h[q].y = (R)sinl(a);
            if ((4LL * q) % n == 0) {
                const int quad = (int)((4LL * q) / n);
                const R cs[4] = {1, 0, -1, 0}, sn[4] = {0, -1, 0, 1};
                h[q].x = cs[quad];
                h[q].y = sn[quad];
            }
        }
        // stage-major copy: entry r * Ns + k - 1 of stage (R, Ns) is
        // w_n^(k r n / (Ns R)); the stages tile [0, n - 1)
        std::vector<V> hs(n, h[0]);
        int Ns = 1;
        for (int s = 0; s < out->nst; ++s) {
            const int rad = out->radix[s];
            const int stride = n / (Ns * rad);
            for (int r = 1; r < rad; ++r)
                for (int k = 0; k < Ns; ++k) hs[r * Ns + k - 1] = h[(long long)k * r * stride];
            Ns *= rad;
        }
        // Uploaded on a private non-blocking stream: a legacy-stream copy
        // would be ordered after every blocking stream, including one that
        // another thread is capturing into a graph.
        void *d = nullptr;
        hipStream_t up = nullptr;
        MR_HIP_CHECK(hipMalloc(&d, 2 * n * sizeof(V)));
        MR_HIP_CHECK(hipStreamCreateWithFlags(&up, hipStreamNonBlocking));
        hipError_t e = hipMemcpyAsync(d, h.data(), n * sizeof(V), hipMemcpyHostToDevice, up);
        if (e == hipSuccess)
            e = hipMemcpyAsync(reinterpret_cast<V *>(d) + n, hs.data(), n * sizeof(V),
                               hipMemcpyHostToDevice, up);
        if (e == hipSuccess) e = hipStreamSynchronize(up);
        (void)hipStreamDestroy(up);
        if (e != hipSuccess) {
            (void)hipFree(d);
            MR_FAIL(MR_ERR_CUDA, "uploading the twiddles of length %d failed: %s", n,
                    hipGetErrorString(e));
        }
        it = g_tw.emplace(key, d).first;
    }
    out->tw = reinterpret_cast<const V *>(it->second);
    out->tws = out->tw + n;
    mr_fft_fill_divs(out);
    return MR_SUCCESS;
}

template int mr_fft_get<float>(int, mr_fft_len<float> *);
template int mr_fft_get<double>(int, mr_fft_len<double> *);

void mr_fft_release_all()
{
    std::lock_guard<std::mutex> lk(g_tw_mu);
    for (auto &kv : g_tw) (void)hipFree(kv.second);
    g_tw.clear();
}

// ---------------------------------------------------------------------------
// Scratch blocks kept between calls (mr_hip.hpp). A block belongs to one
// caller from mr_ws_get to mr_ws_put, so threads and streams never share one;
// only the lists are guarded.
// ---------------------------------------------------------------------------
namespace {
struct ws_block {
    void *p;
    size_t bytes;
    int dev;
    unsigned long long tick;   // request count when it became idle
};
std::mutex g_ws_mu;
std::vector<ws_block> g_ws_used, g_ws_idle;
unsigned long long g_ws_tick = 0;

// Return the idle blocks picked by `gone` to their devices (lock held).
template <class F> bool ws_drop(F gone)
{
    int cur = -1;
    (void)hipGetDevice(&cur);
    bool any = false;
    for (size_t i = 0; i < g_ws_idle.size();) {
        if (!gone(g_ws_idle[i])) {
            ++i;
            continue;
        }
        const ws_block b = g_ws_idle[i];
        g_ws_idle.erase(g_ws_idle.begin() + (long)i);
        if (b.dev != cur) (void)hipSetDevice(b.dev);
        (void)hipFree(b.p);
        if (b.dev != cur) (void)hipSetDevice(cur);
        any = true;
    }
    return any;
}
}  // namespace

size_t mr_ws_idle_bytes(int dev)
{
    std::lock_guard<std::mutex> lk(g_ws_mu);
    size_t n = 0;
    for (const ws_block &b : g_ws_idle) n += (b.dev == dev) ? b.bytes : 0;
    return n;
}

hipError_t mr_dev_malloc(void **p, size_t bytes)
{
    hipError_t e = hipMalloc(p, bytes);
    if (e == hipSuccess) return e;
    int dev = -1;
    (void)hipGetDevice(&dev);
    bool any;
    {
        std::lock_guard<std::mutex> lk(g_ws_mu);
        any = ws_drop([&](const ws_block &b) { return b.dev == dev; });
    }
    if (!any) return e;
    (void)hipGetLastError();
    return hipMalloc(p, bytes);
}

void *mr_ws_get(size_t bytes)
{
    if (bytes == 0) bytes = 1;
    // whole megabytes above one, so that slightly different requests match
    if (bytes > (1u << 20)) bytes = (bytes + (1u << 20) - 1) & ~(size_t)((1u << 20) - 1);
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess) return nullptr;
    {
        std::lock_guard<std::mutex> lk(g_ws_mu);
        ++g_ws_tick;
        ws_drop([](const ws_block &b) { return g_ws_tick - b.tick > 64; });
        size_t best = g_ws_idle.size();
        for (size_t i = 0; i < g_ws_idle.size(); ++i) {
            const ws_block &b = g_ws_idle[i];
            if (b.dev == dev && b.bytes >= bytes && b.bytes <= 2 * bytes &&
                (best == g_ws_idle.size() || b.bytes < g_ws_idle[best].bytes))
                best = i;
        }
        if (best < g_ws_idle.size()) {
            g_ws_used.push_back(g_ws_idle[best]);
            g_ws_idle.erase(g_ws_idle.begin() + (long)best);
            return g_ws_used.back().p;
        }
    }
    void *p = nullptr;
    if (mr_dev_malloc(&p, bytes) != hipSuccess) return nullptr;
    std::lock_guard<std::mutex> lk(g_ws_mu);
    g_ws_used.push_back(ws_block{p, bytes, dev, 0});
    return p;
}

void mr_ws_put(void *p)
{
    if (!p) return;
    std::lock_guard<std::mutex> lk(g_ws_mu);
    for (size_t i = 0; i < g_ws_used.size(); ++i) {
        if (g_ws_used[i].p != p) continue;
        g_ws_idle.push_back(g_ws_used[i]);
        g_ws_idle.back().tick = g_ws_tick;
        g_ws_used.erase(g_ws_used.begin() + (long)i);
        break;
    }
    // over the limit: the blocks idle longest go first
    size_t total = 0;
    for (const ws_block &b : g_ws_idle) total += b.bytes;
    while (total > (size_t)MR_WS_MAX_IDLE) {
        const void *oldest = g_ws_idle.front().p;
        total -= g_ws_idle.front().bytes;
        ws_drop([&](const ws_block &b) { return b.p == oldest; });
    }
}

// ---------------------------------------------------------------------------
// Streaming copy: the attainable HBM bandwidth that the passes are measured
// against (read + write of `bytes`). 16-byte vector loads and stores with the
// non-temporal hint, eight per work-item in flight, a grid of a few
// workgroups per CU striding over the buffer.
// ---------------------------------------------------------------------------
namespace {
typedef unsigned int mr_cp_u4 __attribute__((ext_vector_type(4)));

__global__ void __launch_bounds__(256) mr_k_stream_copy(const mr_cp_u4 *__restrict__ src,
                                                         mr_cp_u4 *__restrict__ dst, long long n)
{
    constexpr int U = 8;
    const long long stride = (long long)gridDim.x * 256 * U;
    for (long long b = (long long)blockIdx.x * 256 * U + threadIdx.x; b < n; b += stride) {
        mr_cp_u4 v[U];
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (b + (long long)u * 256 < n) v[u] = __builtin_nontemporal_load(src + b + (long long)u * 256);
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (b + (long long)u * 256 < n) __builtin_nontemporal_store(v[u], dst + b + (long long)u * 256);
    }
}
}  // namespace

extern "C" MR_EXPORT int mr_stream_copy(const void *d_src, void *d_dst, int64_t bytes,
                                        void *stream)
{
    mr_clear_error();
    MR_REQUIRE(d_src != nullptr && d_dst != nullptr, "mr_stream_copy: NULL buffer");
    MR_REQUIRE(bytes >= 0 && bytes % 16 == 0, "mr_stream_copy: %lld bytes is not a multiple of 16",
               (long long)bytes);
    MR_REQUIRE(((uintptr_t)d_src & 15) == 0 && ((uintptr_t)d_dst & 15) == 0,
               "mr_stream_copy: buffers must be 16-byte aligned");
    if (bytes == 0) return MR_SUCCESS;
    int dev = 0, ncu = 0;
    MR_HIP_CHECK(hipGetDevice(&dev));
    MR_HIP_CHECK(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev));
    const long long n = bytes / 16;
    long long blocks = (n + 256 * 8 - 1) / (256 * 8);
    const long long cap = (long long)ncu * 8;
    if (blocks > cap) blocks = cap;
    hipLaunchKernelGGL(mr_k_stream_copy, dim3((unsigned)blocks), dim3(256), 0,
                       (hipStream_t)stream, (const mr_cp_u4 *)d_src, (mr_cp_u4 *)d_dst, n);
    MR_LAUNCH_CHECK("mr_k_stream_copy");
    return MR_SUCCESS;
}
