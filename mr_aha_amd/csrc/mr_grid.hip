// ES-kernel gridding on gfx950 (see mr_grid.hpp for the conventions).

#include "mr_grid.hpp"

#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <cmath>

void mr_grid_setup(mr_grid *g, int d, const int *M, double eps)
{
    g->d = d;
    int w = (int)std::ceil(std::log10(1.0 / eps)) + 1;
    if (w < 2) w = 2;
    if (w > MR_GRID_MAXW) w = MR_GRID_MAXW;
    g->w = w;
    g->beta = 2.30 * w;
    g->nfine = 1;
    g->nbins = 1;
    for (int a = 0; a < 3; ++a) {
        if (a < d) {
            const int bs = (d == 2) ? 8 : 4;
            int need = 2 * M[a];
            if (need < 2 * w) need = 2 * w;
            const int nf = bs * mr_fft_next_smooth((need + bs - 1) / bs);
            g->M[a] = M[a];
            g->nf[a] = nf;
            g->bs[a] = bs;
            g->nb[a] = nf / bs;
        } else {
            g->M[a] = 1;
            g->nf[a] = 1;
            g->bs[a] = 1;
            g->nb[a] = 1;
        }
        g->nfine *= g->nf[a];
        g->nbins *= g->nb[a];
    }
}

namespace {

// Quadrature of the kernel's transform: Gauss-Legendre nodes on [-1, 1] and
// their weights times the kernel's value there (2 w + 60 nodes).
struct mr_grid_quad {
    int n;
    double z[2 * MR_GRID_MAXW + 60], f[2 * MR_GRID_MAXW + 60];
};

// Newton iteration on P_n for the nodes z > 0 (the others mirror them).
mr_grid_quad mr_make_quad(int w, double beta)
{
    mr_grid_quad q;
    const int n = q.n = 2 * w + 60;   // even
    for (int i = 0; i < n / 2; ++i) {
        double z = std::cos(M_PI * (i + 0.75) / (n + 0.5)), dp = 1.0;
        for (int it = 0; it < 100; ++it) {
            double p0 = 1.0, p1 = z;
            for (int k = 2; k <= n; ++k) {
                const double p2 = ((2.0 * k - 1.0) * z * p1 - (k - 1.0) * p0) / k;
                p0 = p1;
                p1 = p2;
            }
            dp = n * (z * p1 - p0) / (z * z - 1.0);
            const double dz = p1 / dp;
            z -= dz;
            if (std::fabs(dz) < 1e-15) break;
        }
        const double wq = 2.0 / ((1.0 - z * z) * dp * dp);
        q.z[i] = z;
        q.z[n - 1 - i] = -z;
        q.f[i] = q.f[n - 1 - i] = wq * std::exp(beta * (std::sqrt(1.0 - z * z) - 1.0));
    }
    return q;
}

}  // namespace

// Deconvolution factors 1/phi_hat(delta) of one axis, natural order.
__global__ void mr_k_grid_deconv(mr_grid_quad q, int M, int nf, int w, double *dc)
{
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= M) return;
    const int delta = (j < M - M / 2) ? j : j - M;
    const double c = (double)delta * w / nf;
    double s = 0.0;
    for (int i = 0; i < q.n; ++i) s += q.f[i] * cospi(c * q.z[i]);
    dc[j] = 1.0 / (0.5 * w * s);
}

int mr_grid_deconv(const mr_grid &g, double **dc, hipStream_t stream)
{
    const mr_grid_quad q = mr_make_quad(g.w, g.beta);
    for (int a = 0; a < g.d; ++a) {
        MR_HIP_CHECK(mr_dev_malloc((void **)&dc[a], g.M[a] * sizeof(double)));
        hipLaunchKernelGGL(mr_k_grid_deconv, dim3((unsigned)mr_ceil_div(g.M[a], 64)), dim3(64), 0,
                           stream, q, g.M[a], g.nf[a], g.w, dc[a]);
        MR_LAUNCH_CHECK("mr_k_grid_deconv");
    }
    return MR_SUCCESS;
}

__device__ __forceinline__ double mr_es(double z, double beta)
{
    const double t = 1.0 - z * z;
    return (t > 0.0) ? exp(beta * (sqrt(t) - 1.0)) : 0.0;
}

__device__ __forceinline__ int mr_first_point(float x, int nf, int w, double *u_out)
{
    const double u = (double)x * (double)nf * (0.5 / M_PI);
    *u_out = u;
    return (int)ceil(u - 0.5 * w);
}

// Element e of the key array is sample r = e mod Nkx of readout s = e div Nkx
// (trajectory index m = s + Ntrajs r): a stable sort by bin alone then leaves
// every bin in (readout, position) order. Sorting 32-bit bins takes three
// digits where (bin, readout, position) keys of 64 bits took eight.
__global__ void mr_k_grid_keys(const float *traj, long long n, long long Ntrajs, long long Nkx,
                               mr_grid g, unsigned *keys, int *vals)
{
    const long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= n) return;
    const long long s = e / Nkx, r = e - s * Nkx, m = s + Ntrajs * r;
    long long bin = 0, mul = 1;
    for (int a = 0; a < g.d; ++a) {
        double u;
        int i0 = mr_first_point(traj[m + n * a], g.nf[a], g.w, &u);
        i0 %= g.nf[a];
        if (i0 < 0) i0 += g.nf[a];
        bin += mul * (i0 / g.bs[a]);
        mul *= g.nb[a];
    }
    keys[e] = (unsigned)bin;
    vals[e] = (int)m;
}

__global__ void mr_k_grid_fill(const float *traj, long long n, long long Ntrajs, mr_grid g,
                               const int *perm, int *i0o, int *rd, double *wt)
{
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const long long m = perm[i];
    for (int a = 0; a < g.d; ++a) {
        double u;
        const int i0 = mr_first_point(traj[m + n * a], g.nf[a], g.w, &u);
        int im = i0 % g.nf[a];
        if (im < 0) im += g.nf[a];
        i0o[i * 3 + a] = im;
        for (int k = 0; k < g.w; ++k)
            wt[(i * g.d + a) * g.w + k] = mr_es(2.0 * ((double)(i0 + k) - u) / g.w, g.beta);
    }
    for (int a = g.d; a < 3; ++a) i0o[i * 3 + a] = 0;
    rd[i] = (int)(m % Ntrajs);
}

// start[b] = first sorted sample of bin >= b, b = 0 .. nbins (empty bins
// included, so the samples of bins b0 .. b1 are start[b0] .. start[b1 + 1]).
__global__ void mr_k_grid_starts(const unsigned *keys, long long n, long long nbins, int *start)
{
    const long long b = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (b > nbins) return;
    long long lo = 0, hi = n;
    while (lo < hi) {
        const long long mid = (lo + hi) >> 1;
        if ((long long)keys[mid] < b) lo = mid + 1;
        else hi = mid;
    }
    start[b] = (int)lo;
}

// Candidate samples of a tile (one bin's points): the samples of the bins
// whose first points reach it, nbr bins back along every axis (each bin
// once, also where the grid has no more bins than that). Bins that neighbour
// along x are neighbours in the sorted order, so a row of them is one range,
// or two where it wraps. Range r of 2 * rows: row r / 2, piece r % 2.
__device__ __forceinline__ int mr_tile_rows(const mr_grid &g, int *n1, int *n2)
{
    const int k1 = (g.d > 1) ? (g.w - 1 + g.bs[1] - 1) / g.bs[1] + 1 : 1;
    const int k2 = (g.d > 2) ? (g.w - 1 + g.bs[2] - 1) / g.bs[2] + 1 : 1;
    *n1 = k1 < g.nb[1] ? k1 : g.nb[1];
    *n2 = k2 < g.nb[2] ? k2 : g.nb[2];
    return *n1 * *n2;
}

__device__ __forceinline__ void mr_tile_range(const mr_grid &g, const int *start, const int *t,
                                              int n1, int r, int *lo, int *hi)
{
    const int row = r >> 1;
    int b1 = t[1] - row % n1, b2 = t[2] - row / n1;
    if (b1 < 0) b1 += g.nb[1];
    if (b2 < 0) b2 += g.nb[2];
    const long long B = (long long)g.nb[0] * (b1 + (long long)g.nb[1] * b2);
    int k0 = (g.w - 1 + g.bs[0] - 1) / g.bs[0] + 1;
    if (k0 > g.nb[0]) k0 = g.nb[0];
    const int x0 = t[0] - k0 + 1;   // first bin of the row, negative when it wraps
    int f, l;                       // bins f .. l of this piece
    if ((r & 1) == 0) {
        f = x0 < 0 ? 0 : x0;
        l = t[0];
    } else {
        f = x0 < 0 ? x0 + g.nb[0] : 0;
        l = x0 < 0 ? g.nb[0] - 1 : -1;
    }
    *lo = (l < f) ? 0 : start[B + f];
    *hi = (l < f) ? 0 : start[B + l + 1];
}

__device__ __forceinline__ void mr_tile_of(const mr_grid &g, long long tile, int *t)
{
    t[0] = (int)(tile % g.nb[0]);
    t[1] = (int)((tile / g.nb[0]) % g.nb[1]);
    t[2] = (int)(tile / ((long long)g.nb[0] * g.nb[1]));
}

// ext[tile] = segments of MR_GRID_SEG candidates beyond the tile's first
__global__ void mr_k_grid_segments(mr_grid g, const int *start, int *ext)
{
    const long long tile = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (tile >= g.nbins) return;
    int t[3], n1, n2, cand = 0;
    mr_tile_of(g, tile, t);
    const int nr = 2 * mr_tile_rows(g, &n1, &n2);
    for (int r = 0; r < nr; ++r) {
        int lo, hi;
        mr_tile_range(g, start, t, n1, r, &lo, &hi);
        cand += hi - lo;
    }
    ext[tile] = cand > MR_GRID_SEG ? (cand + MR_GRID_SEG - 1) / MR_GRID_SEG - 1 : 0;
}

// ext_tile / ext_no of every extra segment, from the exclusive sums of ext
__global__ void mr_k_grid_ext_list(long long nbins, const int *ext, const int *base, int2 *list)
{
    const long long tile = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (tile >= nbins) return;
    for (int k = 0; k < ext[tile]; ++k) list[base[tile] + k] = make_int2((int)tile, k + 1);
}

void mr_grid_samples_free(mr_grid_samples *s, bool idle)
{
    if (!idle) (void)hipDeviceSynchronize();
    void *bufs[] = {s->i0, s->rd, s->wt, s->start, s->ext};
    for (void *p : bufs) mr_ws_put(p);
    *s = mr_grid_samples();
}

int mr_grid_samples_build(const mr_grid &g, const float *traj, long long Ntrajs, long long Nkx,
                          hipStream_t stream, mr_grid_samples *out)
{
    const long long n = Ntrajs * Nkx;
    MR_REQUIRE(n > 0 && n < 0x7fffffffLL, "gridding: %lld samples outside [1, 2^31)", n);
    MR_REQUIRE(g.nbins < 0x7fffffffLL, "gridding: too many bins (%lld)", g.nbins);
    mr_grid_samples s;
    s.n = n;
    unsigned *keys = nullptr, *keys2 = nullptr;
    int *vals = nullptr, *perm = nullptr, *ext = nullptr, *base = nullptr;
    void *tmp = nullptr;
    size_t sort_bytes = 0, scan_bytes = 0;
    hipError_t e = hipSuccess;
    int end_bit = 1;
    while (end_bit < 32 && (g.nbins >> end_bit) != 0) ++end_bit;
#define MR_GA(ptr, bytes)                                                       \
    if (e == hipSuccess && !((ptr) = (decltype(ptr))mr_ws_get(bytes)))         \
        e = hipErrorOutOfMemory
    MR_GA(keys, n * sizeof(unsigned));
    MR_GA(keys2, n * sizeof(unsigned));
    MR_GA(vals, n * sizeof(int));
    MR_GA(perm, n * sizeof(int));
    MR_GA(ext, (g.nbins + 1) * sizeof(int));
    MR_GA(base, (g.nbins + 1) * sizeof(int));
    MR_GA(s.i0, n * 3 * sizeof(int));
    MR_GA(s.rd, n * sizeof(int));
    MR_GA(s.wt, (size_t)n * g.d * g.w * sizeof(double));
    MR_GA(s.start, (g.nbins + 1) * sizeof(int));
    if (e == hipSuccess)
        e = hipcub::DeviceRadixSort::SortPairs(nullptr, sort_bytes, keys, keys2, vals, perm,
                                              (int)n, 0, end_bit, stream);
    if (e == hipSuccess)
        e = hipcub::DeviceScan::ExclusiveSum(nullptr, scan_bytes, ext, base, (int)g.nbins + 1,
                                             stream);
    const size_t tmp_bytes = sort_bytes > scan_bytes ? sort_bytes : scan_bytes;
    MR_GA(tmp, tmp_bytes ? tmp_bytes : 1);
    int rc = MR_SUCCESS;
    if (e != hipSuccess) {
        (void)hipGetLastError();
        mr_set_error("gridding: failed to allocate the sample tables for %lld samples", n);
        rc = MR_ERR_ALLOC;
    }
    if (rc == MR_SUCCESS) {
        const unsigned nblk = (unsigned)mr_ceil_div(n, 256);
        const unsigned bblk = (unsigned)mr_ceil_div(g.nbins + 1, 256);
        int total = 0;
        hipLaunchKernelGGL(mr_k_grid_keys, dim3(nblk), dim3(256), 0, stream, traj, n, Ntrajs, Nkx,
                           g, keys, vals);
        size_t bytes = sort_bytes;
        e = hipGetLastError();
        if (e == hipSuccess)
            e = hipcub::DeviceRadixSort::SortPairs(tmp, bytes, keys, keys2, vals, perm, (int)n, 0,
                                                  end_bit, stream);
        if (e == hipSuccess) {
            hipLaunchKernelGGL(mr_k_grid_fill, dim3(nblk), dim3(256), 0, stream, traj, n, Ntrajs,
                               g, perm, s.i0, s.rd, s.wt);
            hipLaunchKernelGGL(mr_k_grid_starts, dim3(bblk), dim3(256), 0, stream, keys2, n,
                               g.nbins, s.start);
            hipLaunchKernelGGL(mr_k_grid_segments, dim3(bblk), dim3(256), 0, stream, g, s.start,
                               ext);
            e = hipGetLastError();
        }
        bytes = scan_bytes;   // the sum over all tiles lands in base[nbins]
        if (e == hipSuccess)
            e = hipcub::DeviceScan::ExclusiveSum(tmp, bytes, ext, base, (int)g.nbins + 1, stream);
        if (e == hipSuccess)
            e = hipMemcpyAsync(&total, base + g.nbins, sizeof(int), hipMemcpyDeviceToHost, stream);
        if (e == hipSuccess) e = hipStreamSynchronize(stream);
        if (e == hipSuccess && total > 0) {
            s.next = total;
            s.ext = (int2 *)mr_ws_get((size_t)total * sizeof(int2));
            if (!s.ext) e = hipErrorOutOfMemory;
            if (e == hipSuccess) {
                hipLaunchKernelGGL(mr_k_grid_ext_list, dim3(bblk), dim3(256), 0, stream, g.nbins,
                                   ext, base, s.ext);
                e = hipGetLastError();
            }
            if (e == hipSuccess) e = hipStreamSynchronize(stream);
        }
        if (e != hipSuccess) {
            (void)hipGetLastError();
            mr_set_error("gridding: sample sort failed: %s", hipGetErrorString(e));
            rc = MR_ERR_CUFINUFFT;
        }
    }
    if (rc != MR_SUCCESS) (void)hipStreamSynchronize(stream);   // nothing in flight
    void *scratch[] = {tmp, keys, keys2, vals, perm, ext, base};
    for (void *p : scratch) mr_ws_put(p);
    if (rc != MR_SUCCESS) {
        mr_grid_samples_free(&s, true);
        return rc;
    }
    *out = s;
    return MR_SUCCESS;
}

// ---------------------------------------------------------------------------
// Type-1 gather spreading. One wavefront per segment of at most MR_GRID_SEG
// candidate samples of a tile (8x8 points in 2D, 4x4x4 in 3D; lane = fine
// point). The candidates are taken 64 at a time: lane i tests whether sample i
// reaches the tile and, if so, stages its kernel values at the tile's points
// along each axis (zero outside its support), so a lane's weight of a sample
// is a product of D values read from LDS with no test. With readout-constant
// strengths (PER_SAMPLE false) the weights of consecutive samples of one
// readout are summed first and the CB strengths applied once per run; the
// strengths of a key are contiguous and uniform over the wavefront, so they
// come through the scalar cache. Per-sample strengths would each wait for it, so
// they are staged in LDS with the kernel values (16 sets 215 -> 92 us). The
// first segment of a tile is stored to the fine grid, later ones to `part`,
// which mr_k_spread_sum adds in order.
//
// Once the work is even, a stack's pass is bound by writing the fine grids (2.4
// GB in 0.52 ms, 0.89 of the copy rate, VALU issue 42 %); in 2D and 3D a wavefront's
// serial work on its candidates is what is left (VALU 33 and 40 %, LDS 18 and 25 %,
// memory 0.6 and 0.5). A tile at the centre of radial samples has a thousand times the
// candidates of one at the edge, and with one wavefront per tile the whole
// pass waited for it. Measured, one wavefront per tile and now: 256x256 L=8
// (512 x 512 samples, 36 sets) 2.58 -> 0.25 ms, 192x192x32 L=8 (1152 sets)
// 26.9 -> 3.2 ms, of which the 10.9 GB of output take 2.0, 96^3 L=4 (4000 x
// 192 samples) 49.7 -> 4.7 ms (9.1 GB, 1.7 ms); per sample, 128 x 384 samples
// onto 384x384, 4 sets, 1.26 -> 0.09 ms.
// ---------------------------------------------------------------------------

// LDS of one wavefront: 64 samples' kernel values (the odd stride keeps the
// staging writes off each other's banks), their keys, and the tile's ranges.
// SC: strengths staged beside them.
template <int D, int SC = 0> struct mr_spread_lds {
    static constexpr int BS = (D == 2) ? 8 : 4;
    static constexpr int STR = D * BS + 1;
    double w[64 * STR];
    int key[64];
    int base[64], end[64];
    double2 c[SC > 0 ? 64 * SC : 1];   // [slot][set]
};

template <int D, int CB, bool PER_SAMPLE>
__global__ void __launch_bounds__(256, 4)
mr_k_spread(mr_grid g, const int *__restrict__ i0s, const int *__restrict__ rds,
            const double *__restrict__ wts, const int *__restrict__ start,
            const int2 *__restrict__ ext, long long next, const double2 *__restrict__ str, int qs,
            int q0, int Q, double2 *__restrict__ fine, double2 *__restrict__ part)
{
    using lds_t = mr_spread_lds<D, PER_SAMPLE ? CB : 0>;
    constexpr int BS = lds_t::BS, STR = lds_t::STR;
    __shared__ lds_t sh4[4];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    lds_t &sh = sh4[wave];
    const long long id = (long long)blockIdx.x * 4 + wave;
    if (id >= g.nbins + next) return;   // the wavefronts share nothing
    // extra segments first: they belong to the crowded tiles
    const int2 es = id < next ? ext[id] : make_int2((int)(id - next), 0);
    const int seg = __builtin_amdgcn_readfirstlane(es.y);
    const long long tile = __builtin_amdgcn_readfirstlane(es.x);
    int t[3], T0[3], p[3], n1, n2;
    mr_tile_of(g, tile, t);
    p[0] = lane % BS;
    p[1] = (lane / BS) % BS;
    p[2] = (D == 3) ? lane / (BS * BS) : 0;
#pragma unroll
    for (int a = 0; a < 3; ++a) T0[a] = t[a] * g.bs[a];
    const int w = g.w;
    const int qb = blockIdx.y * CB;

    // ranges of candidates, inclusive sums of their lengths (2 * rows <= 50)
    const int nr = 2 * mr_tile_rows(g, &n1, &n2);
    int lo = 0, hi = 0;
    if (lane < nr) mr_tile_range(g, start, t, n1, lane, &lo, &hi);
    int sum = hi - lo;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int v = __shfl_up(sum, o);
        if (lane >= o) sum += v;
    }
    sh.end[lane] = sum;
    sh.base[lane] = hi - sum;   // candidate k of range r is sample base[r] + k
    const int total = __builtin_amdgcn_readlane(sum, 63);
    const int k_end = (seg + 1) * MR_GRID_SEG < total ? (seg + 1) * MR_GRID_SEG : total;

    double2 acc[CB];
#pragma unroll
    for (int q = 0; q < CB; ++q) acc[q] = make_double2(0.0, 0.0);
    const double2 *strq = str + q0 + qb;

    for (int k0 = seg * MR_GRID_SEG; k0 < k_end; k0 += 64) {
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        const int k = k0 + lane;
        bool in = k < k_end;
        int i = 0, o0[D];
        if (in) {
            int r = 0;
#pragma unroll
            for (int b = 32; b > 0; b >>= 1)
                if (r + b <= 64 && sh.end[r + b - 1] <= k) r += b;
            i = sh.base[r] + k;
#pragma unroll
            for (int a = 0; a < D; ++a) {
                int o = T0[a] - i0s[(long long)i * 3 + a];
                if (o < 0) o += g.nf[a];
                o0[a] = o;
                in = in && (o < w || o + BS > g.nf[a]);
            }
        }
        const unsigned long long m = __ballot(in);
        const int cnt = __popcll(m);
        if (in) {
            const int slot = __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32),
                                                       __builtin_amdgcn_mbcnt_lo((unsigned)m, 0));
            double *ws = sh.w + slot * STR;
            sh.key[slot] = PER_SAMPLE ? i : rds[i];
            // all loads before the first LDS write: one wait instead of one per value
            // (256x256 L=8 0.33 -> 0.25 ms, 96^3 L=4 per chunk 1.84 -> 1.57)
            double v[D][BS];
#pragma unroll
            for (int a = 0; a < D; ++a) {
                const double *wt = wts + ((long long)i * D + a) * w;
#pragma unroll
                for (int b = 0; b < BS; ++b) {
                    int o = o0[a] + b;
                    if (o >= g.nf[a]) o -= g.nf[a];
                    v[a][b] = (o < w) ? wt[o] : 0.0;
                }
            }
#pragma unroll
            for (int a = 0; a < D * BS; ++a) ws[a] = v[a / BS][a % BS];
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        if constexpr (PER_SAMPLE) {
            // the strengths of the staged samples, all loads in flight at once
            double2 v[CB];
#pragma unroll
            for (int n = 0; n < CB; ++n) {
                const int f = lane + 64 * n, j = f / CB, q = f % CB;
                v[n] = j < cnt ? strq[(long long)sh.key[j] * qs + q] : make_double2(0.0, 0.0);
            }
#pragma unroll
            for (int n = 0; n < CB; ++n) sh.c[lane + 64 * n] = v[n];
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
        }
        const int key = sh.key[lane];
        auto weight = [&](int j) {
            const double *ws = sh.w + j * STR;
            double v = ws[p[0]] * ws[BS + p[1]];
            if (D == 3) v *= ws[2 * BS + p[2]];
            return v;
        };
        auto apply = [&](double wv, int ky) {   // ky: the slot, or the readout of a run
            const double2 *c = PER_SAMPLE ? sh.c + ky * CB : strq + (long long)ky * qs;
#pragma unroll
            for (int q = 0; q < CB; ++q) {
                const double2 v = c[q];
                acc[q].x += wv * v.x;
                acc[q].y += wv * v.y;
            }
        };
        // last sample of every run of one readout
        unsigned long long ends = ~0ULL;
        if (!PER_SAMPLE) {
            const int nxt = __shfl_down(key, 1);
            ends = __ballot(lane == cnt - 1 || nxt != key);
        }
        // eight weights at a time, so that their LDS reads overlap
        double wsum = 0.0;
        for (int j0 = 0; j0 < cnt; j0 += 8) {
            double wv[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) wv[j] = weight((j0 + j) & 63);
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                if (j0 + j >= cnt) break;
                wsum += wv[j];
                if ((ends >> (j0 + j)) & 1) {
                    apply(wsum, PER_SAMPLE ? j0 + j : __builtin_amdgcn_readlane(key, j0 + j));
                    wsum = 0.0;
                }
            }
        }
    }
    double2 *dst;
    long long qstride;
    if (id < next) {
        dst = part + id * 64 + lane;
        qstride = next * 64;
    } else {
        dst = fine + (T0[0] + p[0]) +
              (long long)g.nf[0] * ((T0[1] + p[1]) + (long long)g.nf[1] * (T0[2] + p[2]));
        qstride = g.nfine;
    }
#pragma unroll
    for (int q = 0; q < CB; ++q)
        if (qb + q < Q) dst[(long long)(qb + q) * qstride] = acc[q];
}

// Add the extra segments of every crowded tile to its first: the workgroup
// of a tile's first extra segment (number 1) takes them all, in order.
template <int D>
__global__ void __launch_bounds__(64)
mr_k_spread_sum(mr_grid g, const int2 *__restrict__ ext, long long next,
                const double2 *__restrict__ part, double2 *__restrict__ fine, int q0)
{
    constexpr int BS = mr_spread_lds<D>::BS;
    const long long e0 = blockIdx.x;
    const int2 es = ext[e0];
    if (es.y != 1) return;
    long long e1 = e0 + 1;
    while (e1 < next && ext[e1].x == es.x) ++e1;
    const int lane = threadIdx.x;
    int t[3];
    mr_tile_of(g, es.x, t);
    const long long gl = (t[0] * BS + lane % BS) +
                         (long long)g.nf[0] * ((t[1] * BS + (lane / BS) % BS) +
                                               (long long)g.nf[1] *
                                                   (D == 3 ? t[2] * BS + lane / (BS * BS) : 0));
    const long long q = q0 + (int)blockIdx.y;
    double2 *f = fine + q * g.nfine + gl;
    const double2 *s = part + q * next * 64 + lane;
    double2 a = *f;
#pragma unroll 8
    for (long long e = e0; e < e1; ++e) {
        const double2 v = s[e * 64];
        a.x += v.x;
        a.y += v.y;
    }
    *f = a;
}

template <int D, bool PER_SAMPLE>
static int mr_spread_launch(const mr_grid &g, const mr_grid_samples &s, const double2 *str, int qs,
                            int q0, int Q, double2 *fine, double2 *part, hipStream_t stream)
{
    // strengths per wavefront: the fewest that keep the number of chunks of 16
    // (of 8 where they are staged in LDS)
    constexpr int CMAX = PER_SAMPLE ? 8 : 16;
    const int chunks = (Q + CMAX - 1) / CMAX, per = (Q + chunks - 1) / chunks;
    const long long blocks = mr_ceil_div(g.nbins + s.next, 4);
#define MR_SPREAD(CB)                                                                             \
    do {                                                                                          \
        MR_GRID_CHECK(blocks, 256, "mr_k_spread");                                                \
        hipLaunchKernelGGL((mr_k_spread<D, CB, PER_SAMPLE>),                                      \
                           dim3((unsigned)blocks, (unsigned)((Q + CB - 1) / CB)), dim3(256), 0,   \
                           stream, g, s.i0, s.rd, s.wt, s.start, s.ext, s.next, str, qs, q0, Q,   \
                           fine, part);                                                           \
    } while (0)
    if (per <= 4) MR_SPREAD(4);
    else if (per <= 8) MR_SPREAD(8);
    else if constexpr (!PER_SAMPLE) {
        if (per <= 12) MR_SPREAD(12);
        else MR_SPREAD(16);
    }
#undef MR_SPREAD
    MR_LAUNCH_CHECK("mr_k_spread");
    // a set per grid.y, of which a launch has 65535 at most
    for (int y0 = 0; s.next > 0 && y0 < Q; y0 += 65535) {
        hipLaunchKernelGGL(mr_k_spread_sum<D>,
                           dim3((unsigned)s.next, (unsigned)std::min(Q - y0, 65535)), dim3(64), 0,
                           stream, g, s.ext, s.next, part, fine, y0);
        MR_LAUNCH_CHECK("mr_k_spread_sum");
    }
    return MR_SUCCESS;
}

int mr_grid_spread(const mr_grid &g, const mr_grid_samples &s, const double2 *str, int qs, int q0,
                   int Q, double2 *fine, double2 *part, hipStream_t stream)
{
    return g.d == 2 ? mr_spread_launch<2, false>(g, s, str, qs, q0, Q, fine, part, stream)
                    : mr_spread_launch<3, false>(g, s, str, qs, q0, Q, fine, part, stream);
}

int mr_grid_spread_samples(const mr_grid &g, const mr_grid_samples &s, const double2 *str, int Q,
                           double2 *fine, double2 *part, hipStream_t stream)
{
    return g.d == 2 ? mr_spread_launch<2, true>(g, s, str, Q, 0, Q, fine, part, stream)
                    : mr_spread_launch<3, true>(g, s, str, Q, 0, Q, fine, part, stream);
}

// Type-2 interpolation. Eight lanes share a sample and QT sets: lane k reads
// column k (and k + 8) of every row the sample touches, so a load of the
// wavefront takes eight runs of w values instead of 64 values of 64 lines,
// whose addresses bounded it; the sets share weights and addressing, and their
// loads overlap. The lanes' sums are added at the end. 128 x 384 samples onto
// 16 grids of 384 x 384, w = 7: 124 -> 37 us.
template <int D, int QT>
__global__ void __launch_bounds__(256)
mr_k_interp(mr_grid g, const int *__restrict__ i0s, const double *__restrict__ wts, long long n,
            const double2 *__restrict__ fine, int Q, double2 *__restrict__ out, long long base)
{
    const long long id = base * 256 + (long long)blockIdx.x * blockDim.x + threadIdx.x;
    const long long i = id >> 3;
    const int k = (int)id & 7, q0 = blockIdx.y * QT;
    if (i >= n) return;   // all eight lanes of a sample
    const int w = g.w;
    const double2 *f[QT];
#pragma unroll
    for (int q = 0; q < QT; ++q) f[q] = fine + (long long)(q0 + q < Q ? q0 + q : Q - 1) * g.nfine;
    const double *wx = wts + (i * D + 0) * w;
    const double *wy = wts + (i * D + 1) * w;
    const double *wz = (D == 3) ? wts + (i * D + 2) * w : nullptr;
    const int ix = i0s[i * 3], iy = i0s[i * 3 + 1], iz = i0s[i * 3 + 2];
    double2 a[QT];
#pragma unroll
    for (int q = 0; q < QT; ++q) a[q] = make_double2(0.0, 0.0);
    const int nz = (D == 3) ? w : 1;
    for (int kx = k; kx < w; kx += 8) {
        int gx = ix + kx;
        if (gx >= g.nf[0]) gx -= g.nf[0];
        const double fx = wx[kx];
        for (int kz = 0; kz < nz; ++kz) {
            int gz = 0;
            double fz = fx;
            if (D == 3) {
                gz = iz + kz;
                if (gz >= g.nf[2]) gz -= g.nf[2];
                fz = fx * wz[kz];
            }
#pragma unroll 2
            for (int ky = 0; ky < w; ++ky) {
                int gy = iy + ky;
                if (gy >= g.nf[1]) gy -= g.nf[1];
                const double wv = fz * wy[ky];
                const long long o = gx + (long long)g.nf[0] * (gy + (long long)g.nf[1] * gz);
#pragma unroll
                for (int q = 0; q < QT; ++q) {
                    const double2 v = f[q][o];
                    a[q].x += wv * v.x;
                    a[q].y += wv * v.y;
                }
            }
        }
    }
#pragma unroll
    for (int q = 0; q < QT; ++q) {
#pragma unroll
        for (int o = 1; o < 8; o <<= 1) {
            a[q].x += __shfl_xor(a[q].x, o);
            a[q].y += __shfl_xor(a[q].y, o);
        }
        if (k == q && q0 + q < Q) out[i * Q + q0 + q] = a[q];
    }
}

int mr_grid_interp(const mr_grid &g, const mr_grid_samples &s, const double2 *fine, int Q,
                   double2 *out, hipStream_t stream)
{
    constexpr int QT = 4;
    const long long blocks = mr_ceil_div(s.n, 32), step = mr_max_blocks(256);
    auto *fn = g.d == 2 ? mr_k_interp<2, QT> : mr_k_interp<3, QT>;
    for (long long b0 = 0; b0 < blocks; b0 += step) {   // a dispatch counts 2^32 work-items
        hipLaunchKernelGGL(fn, dim3((unsigned)std::min(step, blocks - b0), (unsigned)((Q + QT - 1) / QT)),
                           dim3(256), 0, stream, g, s.i0, s.wt, s.n, fine, Q, out, b0);
        MR_LAUNCH_CHECK("mr_k_interp");
    }
    return MR_SUCCESS;
}

int mr_grid_fft(const mr_grid &g, double2 *fine, double2 *, int Q, bool inverse,
                hipStream_t stream)
{
    mr_fft_len<double> f[3];
    for (int a = 0; a < g.d; ++a) MR_TRY(mr_fft_get<double>(g.nf[a], &f[a]));
    const long long nx = g.nf[0], ny = g.nf[1], nz = g.nf[2];
    if (!inverse) {
        MR_TRY((mr_fft_pass<double, false>(f[0], mr_ld_axis<double2, true>{fine, 1, (int)nx},
                                           mr_st_axis<double2, true>{fine, 1, (int)nx},
                                           ny * nz * Q, 0, 4, stream, "grid x")));
        MR_TRY((mr_fft_pass<double, false>(f[1], mr_ld_axis<double2, false>{fine, nx, (int)ny},
                                           mr_st_axis<double2, false>{fine, nx, (int)ny},
                                           nx * nz * Q, 0, 16, stream, "grid y")));
        if (g.d == 3)
            MR_TRY((mr_fft_pass<double, false>(
                f[2], mr_ld_axis<double2, false>{fine, nx * ny, (int)nz},
                mr_st_axis<double2, false>{fine, nx * ny, (int)nz}, nx * ny * Q, 0, 16, stream,
                "grid z")));
    } else {
        MR_TRY((mr_fft_pass<double, true>(f[0], mr_ld_axis<double2, true>{fine, 1, (int)nx},
                                          mr_st_axis<double2, true>{fine, 1, (int)nx},
                                          ny * nz * Q, 0, 4, stream, "grid x")));
        MR_TRY((mr_fft_pass<double, true>(f[1], mr_ld_axis<double2, false>{fine, nx, (int)ny},
                                          mr_st_axis<double2, false>{fine, nx, (int)ny},
                                          nx * nz * Q, 0, 16, stream, "grid y")));
        if (g.d == 3)
            MR_TRY((mr_fft_pass<double, true>(
                f[2], mr_ld_axis<double2, false>{fine, nx * ny, (int)nz},
                mr_st_axis<double2, false>{fine, nx * ny, (int)nz}, nx * ny * Q, 0, 16, stream,
                "grid z")));
    }
    return MR_SUCCESS;
}
