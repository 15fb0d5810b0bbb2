// Run-time-length axis passes (mr_axis_rt.hpp).
//
// A tile is 16 pencils, neighbours along the contiguous axis where the pass
// allows (one 128-byte line per row), held in LDS as [element][16]: a
// wavefront's accesses in every stage are whole rows. Workgroups are
// persistent; the next tile's rows are loaded into registers while the current
// one is transformed and stored, and nothing else of the loop loads from
// memory in between (the twiddles sit in LDS), so the loads stay in flight
// over the stages. Barriers wait for LDS traffic only.
//
// Against the one-tile kernels, whose loads, transform and stores run one after
// another, the bound moves towards memory. What decides is how many wavefronts
// a CU holds: with 32-bit offsets from uniform bases, unmasked loads and the
// work-item index hidden behind an empty asm, the kernels with 8 elements a
// work-item take 62 (y), 78 and 96 registers (outer, forward and inverse)
// instead of 111 to 128, and the inverse outer
// pass went from 3.93 to 2.05 ms at 256x256x48, L=16, 16 coils (6.9 GB). With 12
// elements (lengths 257 to 384) it is 78, 102 and 128, with the radices 11 and 13
// 71, 87 and 106 (94, 118 and 128 with 12 elements); of these the forward outer
// kernels keep 36 bytes of scratch a lane, the inverse one with 12 elements and a
// radix 11 or 13 68 bytes. Before
// -> now at that size: forward outer 3.62 -> 2.46, inverse 4.67 -> 2.05 ms;
// 240x216x40, L=6, 10 coils: outer 0.59 + 0.75 -> 0.39 + 0.35 ms, y (432) 1.22 +
// 1.20 -> 0.87 + 0.75 ms (3.0 GB each: 3.4 and 4.0 TB/s); an odd plane (143x134x54,
// L=3, 6 coils, one pencil per workgroup before) 0.87 + 0.80 -> 0.07 + 0.07 ms.

#include "mr_axis_form.hpp"
#include "mr_axis_rt.hpp"
#include "mr_xbd.hpp"
#include "mr_fft_ct.hpp"

namespace {

__device__ __forceinline__ unsigned d24_q(const mr_d24 &d, unsigned x)
{
    return __umul24(x, d.mul) >> d.shr;
}

// The work-item index, hidden behind an empty asm: what derives from it is
// recomputed where it is used, not held in registers over the tile loop.
__device__ __forceinline__ int fresh_tid()
{
    unsigned t = threadIdx.x;
    asm volatile("" : "+v"(t));
    return (int)t;
}

// One Stockham stage in place over [n][PT]: work-item f takes pencil f mod PT
// and butterfly f / PT; n <= KE NT / PT.
template <int RR, bool INV, int NT, int KE, int PT>
__device__ __forceinline__ void ax_stage(float2 *A, const float2 *tw, int m, int Ns,
                                         const mr_d24 &nd)
{
    constexpr int KMAX = (KE + RR - 1) / RR;
    const int nb = m * PT, tid = fresh_tid();
    float2 v[KMAX][RR];
#pragma unroll
    for (int k = 0; k < KMAX; ++k) {
        const int f = tid + k * NT;
        if (f < nb) {
            const float2 *a = A + f;   // (f / PT) * PT + f mod PT
#pragma unroll
            for (int r = 0; r < RR; ++r) v[k][r] = a[r * m * PT];
        }
    }
    mr_lds_barrier();
#pragma unroll
    for (int k = 0; k < KMAX; ++k) {
        const int f = tid + k * NT;
        if (f < nb) {
            const unsigned p = f & (PT - 1), j = f / PT;
            const unsigned jn = d24_q(nd, j), kk = j - jn * Ns;
            if (Ns > 1) {
                const float2 *w = tw + (Ns - 1 + kk);
#pragma unroll
                for (int r = 1; r < RR; ++r) {
                    const float2 wr = w[(r - 1) * Ns];
                    v[k][r] = INV ? cmulc(wr, v[k][r]) : cmul(wr, v[k][r]);
                }
            }
            bfly<RR, INV>(v[k]);
            float2 *b = A + (jn * (Ns * RR) + kk) * PT + p;
#pragma unroll
            for (int q = 0; q < RR; ++q) b[q * Ns * PT] = v[k][q];
        }
    }
    mr_lds_barrier();
}

// BIG: lengths with a radix 11 or 13, whose butterflies take twice the
// registers of the others (kernels of their own, at half the wavefronts).
template <bool INV, int NT, int KE, int PT, bool BIG>
__device__ __forceinline__ void ax_fft(float2 *A, const float2 *tw, const mr_rt_len &f)
{
    int Ns = 1;
    for (int s = 0; s < f.nst; ++s) {
        const int RR = f.radix[s], m = f.m[s];
        const mr_d24 nd = f.nd[s];
        switch (RR) {
#define AX_ST(R) case R: ax_stage<R, INV, NT, KE, PT>(A, tw, m, Ns, nd); break;
            AX_ST(2) AX_ST(3) AX_ST(4) AX_ST(5) AX_ST(6) AX_ST(7) AX_ST(10)
        case 11: if constexpr (BIG) ax_stage<11, INV, NT, KE, PT>(A, tw, m, Ns, nd); break;
        case 13: if constexpr (BIG) ax_stage<13, INV, NT, KE, PT>(A, tw, m, Ns, nd); break;
#undef AX_ST
        default: ax_stage<8, INV, NT, KE, PT>(A, tw, m, Ns, nd); break;
        }
        Ns *= RR;
    }
}

// The same at a compiled length: strides, divisors and round counts are
// constants, LDS offsets immediates. Inverse outer pass at 320 (160^3, L=8, 8
// coils) 1.59 -> 1.43 ms, at 384 (2D 192x192, L=8, 12 coils) 47 -> 44 us.
template <int N, int S, bool INV, int NT, int KE, int PT>
__device__ __forceinline__ void ax_fft_ct(float2 *A, const float2 *tw)
{
    constexpr mr_ct_fac F = mr_ct_factor(N);
    if constexpr (S < F.nst) {
        constexpr int RR = F.r[S], NS = F.ns[S];
        constexpr mr_d24 nd = mr_d24_make(NS);
        ax_stage<RR, INV, NT, KE, PT>(A, tw, N / RR, NS, nd);
        ax_fft_ct<N, S + 1, INV, NT, KE, PT>(A, tw);
    }
}

// Tiles of this workgroup: XCD x (blockIdx.x mod 8) owns a contiguous share of
// the tiles, its workgroups take them in turn, so tiles that share rows of x or
// S meet in one L2.
struct ax_share {
    int t, end, step;
};
__device__ __forceinline__ ax_share ax_tiles(int nt)
{
    const int G = gridDim.x, x = blockIdx.x % 8, g8 = G / 8, g8r = G % 8;
    const int cx = g8 + (x < g8r ? 1 : 0);
    const long long before = (long long)x * g8 + (x < g8r ? x : g8r);
    return ax_share{(int)((long long)nt * before / G) + (int)(blockIdx.x / 8),
                    (int)((long long)nt * (before + cx) / G), cx};
}

__device__ __forceinline__ void ax_twiddles(float2 *tw, const float2 *tws, int n)
{
    for (int i = threadIdx.x; i < n; i += blockDim.x) tw[i] = tws[i];
}

// Element `off` bytes past a wavefront-uniform base: the base stays in scalar
// registers, a lane holds 32 bits.
__device__ __forceinline__ float2 ax_ld(const float2 *base, unsigned off)
{
    return *reinterpret_cast<const float2 *>(reinterpret_cast<const char *>(base) + off);
}
__device__ __forceinline__ void ax_st(float2 *base, unsigned off, float2 v)
{
    *reinterpret_cast<float2 *>(reinterpret_cast<char *>(base) + off) = v;
}

// Loads take no masks: a lane without an element, row, position or coil reads
// a neighbour's (clamped) and puts zero in its place when the tile is written
// to LDS.
template <bool INV, int NT, int KE, int PT, bool BIG>
__global__ void __launch_bounds__(NT, ax_waves(AX_Y, KE, BIG))
mr_k_axis_y(mr_rt_len f, const float2 *tws, mr_ax_y a, mr_fdiv idiv, int npencil, int nt)
{
    constexpr int DE = NT / PT;
    extern __shared__ __align__(16) unsigned char mr_smem[];
    float2 *A = reinterpret_cast<float2 *>(mr_smem);
    float2 *tw = A + f.n * PT;
    const int n = f.n;
    const int I = (int)a.I;
    ax_twiddles(tw, tws, n);
    ax_share sh = ax_tiles(nt);
    float2 r[KE];
    // column of pencil p of tile t: base of the tile's first column (uniform)
    // and the lane's byte offset from it; rows I values apart
    auto column = [&](int t, int rows, int p, long long *first, unsigned *off) {
        const int p0 = t * PT;
        const int o = (int)mr_fdiv_q(idiv, (unsigned)p0);
        int i = p0 - o * I;
        *first = i + (long long)I * rows * o;
        int q = p;
        if (p0 + q >= npencil) q = npencil - 1 - p0;
        unsigned d = (unsigned)q;
        for (i += q; i >= I; i -= I) d += (unsigned)(I * (rows - 1));   // next plane
        *off = d * 8u;
    };
    auto load = [&](int t) {
        const int tid = fresh_tid(), p = tid & (PT - 1), e0 = tid / PT;
        long long first;
        unsigned off;
        column(t, a.n_in, p, &first, &off);
        const float2 *src = a.in + first;
#pragma unroll
        for (int k = 0; k < KE; ++k) {
            int s = e0 + k * DE + a.c_in;
            if (s >= n) s -= n;
            s = s < a.n_in ? s : a.n_in - 1;
            r[k] = ax_ld(src, off + (unsigned)(s * I) * 8u);
        }
    };
    if (sh.t < sh.end) load(sh.t);
    for (; sh.t < sh.end; sh.t += sh.step) {
        {
            const int tid = fresh_tid(), p = tid & (PT - 1), e0 = tid / PT;
#pragma unroll
            for (int k = 0; k < KE; ++k) {
                const int e = e0 + k * DE;
                int s = e + a.c_in;
                if (s >= n) s -= n;
                if (e < n) A[e * PT + p] = s < a.n_in ? r[k] : make_float2(0.f, 0.f);
            }
        }
        mr_lds_barrier();
        if (sh.t + sh.step < sh.end) load(sh.t + sh.step);
        ax_fft<INV, NT, KE, PT, BIG>(A, tw, f);
        const int tid = fresh_tid(), p = tid & (PT - 1), e0 = tid / PT;
        long long first;
        unsigned off;
        column(sh.t, a.n_out, p, &first, &off);
        float2 *dst = a.out + first;
        const bool pv = sh.t * PT + p < npencil;
#pragma unroll
        for (int k = 0; k < KE; ++k) {
            const int e = e0 + k * DE;
            int s = e + a.c_out;
            if (s >= n) s -= n;
            if (e < n && s < a.n_out && pv) ax_st(dst, off + (unsigned)(s * I) * 8u, A[e * PT + p]);
        }
        mr_lds_barrier();   // A is read out before the next tile is written
    }
}

// A work-item's place in a tile of an outer pass: pencil p = position xs, coil
// cs; first element e0.
struct ax_lane {
    int p, e0, xs, cs;
};
template <int PT> __device__ __forceinline__ ax_lane ax_lane_of(int lgxw)
{
    const int tid = fresh_tid(), p = tid & (PT - 1);
    return ax_lane{p, tid / PT, p & ((1 << lgxw) - 1), p >> lgxw};
}

// Outer passes. A tile is XW neighbouring plane positions of one rank times CW
// = PT / XW coils, and takes ceil(nc / CW) rounds over the coils. Tiles run
// over the ranks first, which share the rows of S.
template <int NT, int KE, int PT, bool BIG>
__global__ void __launch_bounds__(NT, ax_waves(AX_FO, KE, BIG))
mr_k_axis_fo(mr_rt_len f, const float2 *tws, mr_ax_z a, mr_fdiv ldiv, int lgxw, int nt)
{
    constexpr int DE = NT / PT;
    extern __shared__ __align__(16) unsigned char mr_smem[];
    float2 *A = reinterpret_cast<float2 *>(mr_smem);
    float2 *tw = A + f.n * PT;
    const int n = f.n, CW = PT >> lgxw;
    const unsigned row = (unsigned)a.plane * 8u;   // bytes
    ax_twiddles(tw, tws, n);
    ax_share sh = ax_tiles(nt);
    float2 sv[KE], xv[KE];
    // byte offset of image row z of the work-item's k-th element (clamped)
    auto zoff = [&](int e0, int k) {
        int z = e0 + k * DE + a.cz;
        if (z >= n) z -= n;
        return (unsigned)(z < a.nz ? z : a.nz - 1) * row;
    };
    auto xoff = [&](int xs, int xt) {   // of the lane's position in its tile (clamped)
        const int last = (int)a.plane - 1 - (xt << lgxw);
        return (unsigned)(xs < last ? xs : last) * 8u;
    };
    auto load_s = [&](int xt, int c0) {
        const ax_lane q = ax_lane_of<PT>(lgxw);
        const int c = c0 + q.cs < a.nc ? q.cs : a.nc - 1 - c0;
        const float2 *S = a.S + ((long long)xt << lgxw) + a.N * (a.coil0 + c0);
        const unsigned off = xoff(q.xs, xt) + (unsigned)(a.N * c) * 8u;
#pragma unroll
        for (int k = 0; k < KE; ++k) sv[k] = ax_ld(S, off + zoff(q.e0, k));
    };
    auto load_x = [&](int xt, int l) {
        const ax_lane q = ax_lane_of<PT>(lgxw);
        const float2 *x = a.x + ((long long)xt << lgxw) + a.N * l;
        const unsigned off = xoff(q.xs, xt);
#pragma unroll
        for (int k = 0; k < KE; ++k) xv[k] = ax_ld(x, off + zoff(q.e0, k));
    };
    if (sh.t < sh.end) {
        const int xt = (int)mr_fdiv_q(ldiv, (unsigned)sh.t);
        load_x(xt, sh.t - xt * a.L);
        load_s(xt, 0);
    }
    for (; sh.t < sh.end; sh.t += sh.step) {
        const int xt = (int)mr_fdiv_q(ldiv, (unsigned)sh.t), l = sh.t - xt * a.L;
        for (int c0 = 0; c0 < a.nc; c0 += CW) {
            const ax_lane q = ax_lane_of<PT>(lgxw);
#pragma unroll
            for (int k = 0; k < KE; ++k) {
                const int e = q.e0 + k * DE;
                int z = e + a.cz;
                if (z >= n) z -= n;
                if (e < n) A[e * PT + q.p] = z < a.nz ? cmul(sv[k], xv[k]) : make_float2(0.f, 0.f);
            }
            mr_lds_barrier();
            if (c0 + CW < a.nc) {
                load_s(xt, c0 + CW);
            } else if (sh.t + sh.step < sh.end) {
                const int t1 = sh.t + sh.step, xt1 = (int)mr_fdiv_q(ldiv, (unsigned)t1);
                load_x(xt1, t1 - xt1 * a.L);
                load_s(xt1, 0);
            }
            ax_fft<false, NT, KE, PT, BIG>(A, tw, f);
            float2 *dst = a.work + ((long long)xt << lgxw) +
                          a.plane * n * (l + (long long)a.L * c0);
            const ax_lane u = ax_lane_of<PT>(lgxw);
            const unsigned off = (unsigned)u.xs * 8u + (unsigned)(u.cs * a.L * n) * row;
            const bool pv = (xt << lgxw) + u.xs < a.plane && c0 + u.cs < a.nc;
#pragma unroll
            for (int k = 0; k < KE; ++k) {
                const int e = u.e0 + k * DE;
                if (e < n && pv) ax_st(dst, off + (unsigned)e * row, A[e * PT + u.p]);
            }
            mr_lds_barrier();
        }
    }
}

// N: a compiled length, or 0
template <int NT, int KE, int PT, bool BIG, int N = 0>
__global__ void __launch_bounds__(NT, ax_waves(AX_IO, KE, BIG))
mr_k_axis_io(mr_rt_len f, const float2 *tws, mr_ax_z a, mr_fdiv ldiv, int lgxw, int nt)
{
    constexpr int DE = NT / PT;
    extern __shared__ __align__(16) unsigned char mr_smem[];
    float2 *A = reinterpret_cast<float2 *>(mr_smem);
    float2 *tw = A + f.n * PT;
    const int n = N > 0 ? N : f.n, CW = PT >> lgxw;
    const unsigned row = (unsigned)a.plane * 8u;   // bytes
    ax_twiddles(tw, tws, n);
    ax_share sh = ax_tiles(nt);
    float2 r[KE], sv[KE], acc[KE];
    auto xoff = [&](int xs, int xt) {
        const int last = (int)a.plane - 1 - (xt << lgxw);
        return (unsigned)(xs < last ? xs : last) * 8u;
    };
    auto load = [&](int xt, int l, int c0) {
        const ax_lane q = ax_lane_of<PT>(lgxw);
        const int c = c0 + q.cs < a.nc ? q.cs : a.nc - 1 - c0;
        const float2 *src = a.work + ((long long)xt << lgxw) +
                            a.plane * n * (l + (long long)a.L * c0);
        const unsigned off = xoff(q.xs, xt) + (unsigned)(c * a.L * n) * row;
#pragma unroll
        for (int k = 0; k < KE; ++k) {
            const int e = q.e0 + k * DE;
            r[k] = ax_ld(src, off + (unsigned)(e < n ? e : n - 1) * row);
        }
    };
    if (sh.t < sh.end) {
        const int xt = (int)mr_fdiv_q(ldiv, (unsigned)sh.t);
        load(xt, sh.t - xt * a.L, 0);
    }
    for (; sh.t < sh.end; sh.t += sh.step) {
        const int xt = (int)mr_fdiv_q(ldiv, (unsigned)sh.t), l = sh.t - xt * a.L;
        for (int c0 = 0; c0 < a.nc; c0 += CW) {
            const ax_lane q = ax_lane_of<PT>(lgxw);
#pragma unroll
            for (int k = 0; k < KE; ++k) {
                const int e = q.e0 + k * DE;
                if (e < n) A[e * PT + q.p] = r[k];
            }
            mr_lds_barrier();
            // this round's S rows, then the next round's data: both are in
            // flight over the stages, the S rows are back first
            {
                const int c = c0 + q.cs < a.nc ? q.cs : a.nc - 1 - c0;
                const float2 *S = a.S + ((long long)xt << lgxw) + a.N * (a.coil0 + c0);
                const unsigned off = xoff(q.xs, xt) + (unsigned)(a.N * c) * 8u;
#pragma unroll
                for (int k = 0; k < KE; ++k) {
                    int z = q.e0 + k * DE + a.cz;
                    if (z >= n) z -= n;
                    sv[k] = ax_ld(S, off + (unsigned)(z < a.nz ? z : a.nz - 1) * row);
                }
            }
            if (c0 + CW < a.nc) {
                load(xt, l, c0 + CW);
            } else if (sh.t + sh.step < sh.end) {
                const int t1 = sh.t + sh.step, xt1 = (int)mr_fdiv_q(ldiv, (unsigned)t1);
                load(xt1, t1 - xt1 * a.L, 0);
            }
            if constexpr (N > 0) ax_fft_ct<N, 0, true, NT, KE, PT>(A, tw);
            else ax_fft<true, NT, KE, PT, BIG>(A, tw, f);
            const ax_lane w = ax_lane_of<PT>(lgxw);
#pragma unroll
            for (int k = 0; k < KE; ++k) {
                const int e = w.e0 + k * DE;
                const float2 v = cmulc(sv[k], A[(e < n ? e : n - 1) * PT + w.p]);
                if (CW == 1) {
                    acc[k] = (c0 == 0) ? v : cadd(acc[k], v);
                } else {
                    // the tile's coils in order (absent ones are not added)
                    for (int c = 0; c < CW && c0 + c < a.nc; ++c) {
                        const int lane = (threadIdx.x & (64 - PT)) + w.xs + (c << lgxw);
                        const float2 u = make_float2(__shfl(v.x, lane), __shfl(v.y, lane));
                        acc[k] = (c0 + c == 0) ? u : cadd(acc[k], u);
                    }
                }
            }
            mr_lds_barrier();
        }
        const ax_lane w = ax_lane_of<PT>(lgxw);
        if (w.cs != 0 || (xt << lgxw) + w.xs >= a.plane) continue;
        float2 *dst = a.out + ((long long)xt << lgxw) + a.N * l;
#pragma unroll
        for (int k = 0; k < KE; ++k) {
            const int e = w.e0 + k * DE;
            int z = e + a.cz;
            if (z >= n) z -= n;
            if (e < n && z < a.nz) {
                const unsigned off = (unsigned)w.xs * 8u + (unsigned)z * row;
                ax_st(dst, off, a.accumulate ? cadd(ax_ld(dst, off), acc[k]) : acc[k]);
            }
        }
    }
}

int ax_cus()
{
    static const int n = [] {
        int dev = 0, v = 0;
        if (hipGetDevice(&dev) != hipSuccess ||
            hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
            v <= 0)
            v = 256;
        return v;
    }();
    return n;
}

bool ax_ok(const mr_fft_len<float> &f, mr_rt_len *rt, bool *big)
{
    *big = false;
    if (f.n > MR_AX_NMAX || mr_env_ll("MR_AHA_HIP_AXRT", 1) == 0) return false;
    for (int s = 0; s < f.nst; ++s) {
        const bool b = f.radix[s] == 11 || f.radix[s] == 13;
        if (!mr_fft_unrolled(f.radix[s]) && !b) return false;
        *big = *big || b;
    }
    return mr_rt_len_make(f, rt);
}

template <class K, class... Args>
int ax_launch(K kernel, const ax_form &fm, ax_kind kind, bool big, int n, long long nt,
              hipStream_t s, const char *name, Args... args)
{
    const int NT = fm.nt;
    const size_t lds = (size_t)ax_lds(fm, n);
    if (lds > 65536)
        MR_HIP_CHECK(hipFuncSetAttribute((const void *)kernel,
                                         hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    const long long most = (long long)ax_cus() * ax_per_cu(kind, fm, big, n);
    const long long grid = nt < most ? nt : most;
    hipLaunchKernelGGL(kernel, dim3((unsigned)grid), dim3(NT), lds, s, args..., (int)nt);
    MR_LAUNCH_CHECK(name);
    return MR_SUCCESS;
}

}  // namespace

// The forms of ax_pick: the narrow one is for outer passes, the wide one for y
#define AX_EACH_Y(CALL)                                                                          \
    if (fm.nt == 128) CALL(128, 8, 16);                                                          \
    else if (fm.nt == 256) CALL(256, 8, 16);                                                     \
    else if (fm.nt == 1024) CALL(1024, 8, 16);                                                   \
    else if (fm.ke == 12) CALL(512, 12, 16);                                                     \
    else CALL(512, 8, 16);
#define AX_EACH_Z(CALL)                                                                          \
    if (fm.nt == 128) CALL(128, 8, 16);                                                          \
    else if (fm.nt == 256) CALL(256, 8, 16);                                                     \
    else if (fm.pt == 8) CALL(512, 8, 8);                                                        \
    else if (fm.ke == 12) CALL(512, 12, 16);                                                     \
    else CALL(512, 8, 16);

#define AX_Y1(INV, NT, KE, PT, BIG)                                                              \
    ax_launch(mr_k_axis_y<INV, NT, KE, PT, BIG>, fm, AX_Y, BIG, f.n, nt, s, "mr_k_axis_y", rt,    \
              f.tws, a, idiv, (int)npencil)
#define AX_YF(NT, KE, PT)                                                                        \
    *rc = inverse ? (big ? AX_Y1(true, NT, KE, PT, true) : AX_Y1(true, NT, KE, PT, false))        \
                  : (big ? AX_Y1(false, NT, KE, PT, true) : AX_Y1(false, NT, KE, PT, false))

int mr_axis_rt_y(const mr_fft_len<float> &f, bool inverse, const mr_ax_y &a, long long npencil,
                  hipStream_t s, int *rc)
{
    mr_rt_len rt;
    bool big;
    if (!ax_ok(f, &rt, &big)) return 0;
    // 32-bit pencil numbers and byte offsets within a tile's columns
    if (npencil >= 0x7fffff00LL || a.I * 8 * (f.n + 1) * 17 >= 0xffffffffLL) return 0;
    const mr_fdiv idiv = mr_fdiv_make((unsigned)a.I);
    const ax_form fm = ax_pick(f.n, false, false);
    const long long nt = mr_ceil_div(npencil, fm.pt);
    AX_EACH_Y(AX_YF)
    return fm.pt;
}

#define AX_Z1(K, KIND, NT, KE, PT, BIG)                                                          \
    ax_launch(K<NT, KE, PT, BIG>, fm, KIND, BIG, f.n, nt, s, #K, rt, f.tws, a, ldiv, lgxw)
#define AX_ZF(NT, KE, PT)                                                                        \
    *rc = inverse ? (big ? AX_Z1(mr_k_axis_io, AX_IO, NT, KE, PT, true)                          \
                         : AX_Z1(mr_k_axis_io, AX_IO, NT, KE, PT, false))                        \
                  : (big ? AX_Z1(mr_k_axis_fo, AX_FO, NT, KE, PT, true)                          \
                         : AX_Z1(mr_k_axis_fo, AX_FO, NT, KE, PT, false))

int mr_axis_rt_z(const mr_fft_len<float> &f, bool inverse, const mr_ax_z &a, hipStream_t s, int *rc)
{
    mr_rt_len rt;
    bool big;
    if (!ax_ok(f, &rt, &big)) return 0;
    // whole lines (16 positions) where that gives every CU two tiles, else
    // narrower tiles that take several coils at once
    const ax_form fm = ax_pick(f.n, true, mr_ceil_div(a.plane, 16) * a.L < 2 * ax_cus());
    int lgxw = fm.pt == 16 ? 4 : 3;
    while (lgxw > 2 && mr_ceil_div(a.plane, 1LL << lgxw) * a.L < 2 * ax_cus() &&
           (fm.pt >> lgxw) < a.nc)
        --lgxw;
    const long long nt = mr_ceil_div(a.plane, 1LL << lgxw) * a.L;
    // 32-bit tile numbers and byte offsets within a tile's coils
    const long long cw = fm.pt >> lgxw;
    if (nt >= 0x7fffff00LL || a.plane * 8 * (f.n + 1) * (1 + (cw - 1) * a.L) >= 0xffffffffLL ||
        a.N * 8 * cw >= 0xffffffffLL)
        return 0;
    const mr_fdiv ldiv = mr_fdiv_make((unsigned)a.L);
    if (inverse) {
        switch (f.n * 100 + fm.pt) {
#define AX_ZN(N, NT, KE, PT)                                                                     \
    case N * 100 + PT:                                                                           \
        *rc = ax_launch(mr_k_axis_io<NT, KE, PT, false, N>, fm, AX_IO, false, f.n, nt, s,          \
                        "mr_k_axis_io", rt, f.tws, a, ldiv, lgxw);                               \
        return fm.pt;
            AX_ZN(256, 512, 8, 16) AX_ZN(320, 512, 8, 8) AX_ZN(320, 512, 12, 16)
            AX_ZN(384, 512, 8, 8) AX_ZN(384, 512, 12, 16) AX_ZN(512, 512, 8, 8)
#undef AX_ZN
        default: break;
        }
    }
    AX_EACH_Z(AX_ZF)
    return fm.pt;
}
