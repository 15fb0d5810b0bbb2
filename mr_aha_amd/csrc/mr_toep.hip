// Toeplitz kernel build on gfx950 (mr_calc_toep, mr_calc_toep_from_psf).
//
//   phi2_toep[kappa, t] = (1/prod M_tr) sum_delta psf_t[delta] e^{+2 pi i kappa.delta/M}
//   psf_t[delta]        = sum_m c_{t,m} e^{-i delta.x_m}
// (reference: src/cuda/mr_calc_toep.cu:10-24, 171-200, 498-643). Transformed
// axes: x, y for 2D and stack (every kz plane its own component, no shift
// and no scaling along z), x, y, z for 3D.
//
// MI355X pipeline per chunk of components q = z + Nkz * t:
//   1. gather-spread (FP64) of the readout-constant strengths onto the
//      2x fine grid (mr_grid_spread: no atomics, one strength multiply per
//      readout run of each bin),
//   2. per axis, in one pass over the pencils (mr_k_toep_axis): forward FFT of
//      the fine pencil (FP64, sign -1), crop to the M modes and deconvolution
//      by the ES kernel's transform, inverse FFT over the M modes (sign +1),
//      centered store; the last axis scales by 1/prod M and stores FP32 (or
//      gathers the mask).
// A mode count with a prime factor that has no unrolled butterfly takes step 2
// as separate passes: FFTs of the fine axes, deconvolution, inverse FFTs of
// the mode axes, shifted store.

#include "mr_grid.hpp"

#include <chrono>
#include <cstring>

// c[s * Q + q] = packed element t of the Gram block of readout s and kz
// plane z (q = z + Nkz t, Q of them: a readout's strengths are contiguous, as
// the spreading reads them); phi2 is [Ntrajs, Nkz, L, L] column-major
// (src/cuda/mr_kernels.cu:307-333 packing).
__global__ void mr_k_pack_strengths(const float2 *phi2, long long Ntrajs, int Nkz, int L,
                                    int upper, int T, double2 *c)
{
    const long long id = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    const long long total = (long long)T * Nkz * Ntrajs;
    if (id >= total) return;
    const long long s = id % Ntrajs;
    const long long q = id / Ntrajs;
    const int z = (int)(q % Nkz);
    const int t = (int)(q / Nkz);
    // packed offset t -> (i, j): walk columns
    int i = 0, j = 0, acc = 0;
    for (j = 0; j < L; ++j) {
        const int len = upper ? j + 1 : L - j;
        if (t < acc + len) {
            i = upper ? (t - acc) : j + (t - acc);
            break;
        }
        acc += len;
    }
    const float2 v = phi2[s + Ntrajs * (z + (long long)Nkz * (i + (long long)L * j))];
    c[s * T * Nkz + q] = make_double2((double)v.x, (double)v.y);
}

// nat[j + Ptr*q] = fine[(delta mod nf) + nfine*q] * dc0[jx] dc1[jy] dc2[jz]
__global__ void mr_k_deconv(const double2 *fine, mr_grid g, long long Ptr, int Qc,
                            const double *dc0, const double *dc1, const double *dc2, double2 *nat)
{
    const long long id = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (id >= Ptr * Qc) return;
    const long long q = id / Ptr;
    const long long j = id - q * Ptr;
    const int jx = (int)(j % g.M[0]);
    const int jy = (int)((j / g.M[0]) % g.M[1]);
    const int jz = (int)(j / ((long long)g.M[0] * g.M[1]));
    int f[3];
    const int jj[3] = {jx, jy, jz};
    for (int a = 0; a < 3; ++a) {
        const int M = g.M[a];
        int dlt = (jj[a] < M - M / 2) ? jj[a] : jj[a] - M;
        if (dlt < 0) dlt += g.nf[a];
        f[a] = dlt;
    }
    const long long fl = f[0] + (long long)g.nf[0] * (f[1] + (long long)g.nf[1] * f[2]);
    const double s = dc0[jx] * dc1[jy] * (dc2 ? dc2[jz] : 1.0);
    const double2 v = fine[fl + g.nfine * q];
    nat[id] = make_double2(v.x * s, v.y * s);
}

// centered psf [Ptr, Qc] (float) -> natural-order double
__global__ void mr_k_psf_to_nat(const float2 *psf, int m0, int m1, int m2, int s0, int s1, int s2,
                                long long Ptr, int Qc, double2 *nat)
{
    const long long id = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (id >= Ptr * Qc) return;
    const long long q = id / Ptr;
    const long long j = id - q * Ptr;
    int k0 = (int)(j % m0) + s0; if (k0 >= m0) k0 -= m0;
    int k1 = (int)((j / m0) % m1) + s1; if (k1 >= m1) k1 -= m1;
    int k2 = (int)(j / ((long long)m0 * m1)) + s2; if (k2 >= m2) k2 -= m2;
    const float2 v = psf[k0 + (long long)m0 * (k1 + (long long)m1 * k2) + Ptr * q];
    nat[id] = make_double2((double)v.x, (double)v.y);
}

// Natural -> centered, scale, FP32 store of components q0 .. q0+Qc-1.
// Unmasked: out[k + Ptr*q]. Masked: out[row + nm*t] for row = inv[k + Ptr*z].
__global__ void mr_k_toep_store(const double2 *nat, int m0, int m1, int m2, int s0, int s1, int s2,
                                long long Ptr, int Qc, long long q0, int Nkz, double scale,
                                const int *inv, long long nm, float2 *out)
{
    const long long id = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (id >= Ptr * Qc) return;
    const long long qq = id / Ptr;
    const long long k = id - qq * Ptr;
    int j0 = (int)(k % m0) - s0; if (j0 < 0) j0 += m0;
    int j1 = (int)((k / m0) % m1) - s1; if (j1 < 0) j1 += m1;
    int j2 = (int)(k / ((long long)m0 * m1)) - s2; if (j2 < 0) j2 += m2;
    const double2 v = nat[j0 + (long long)m0 * (j1 + (long long)m1 * j2) + Ptr * qq];
    const float2 o = make_float2((float)(v.x * scale), (float)(v.y * scale));
    const long long q = q0 + qq;
    if (!inv) {
        out[k + Ptr * q] = o;
        return;
    }
    const long long z = q % Nkz, t = q / Nkz;
    const int row = inv[k + Ptr * z];
    if (row >= 0) out[row + nm * t] = o;
}

// ---------------------------------------------------------------------------
// One axis of the build in one pass. The forward transform of the fine axis,
// the crop with its deconvolution weights and the inverse transform of the
// mode axis act on one axis each, so they commute with those of the other
// axes and an axis can be finished before the next: a pencil of nf values is
// read, becomes M centered values in LDS and is written back over its own
// first M places (the pitch stays that of the fine grid, no second buffer).
// Later axes then run over M instead of nf values of the finished ones.
//
// What counts is memory traffic: 2D moves 16 nf^2 read, 8 nf^2 written and read, 2 nf^2
// written bytes (and the spread's 16 nf^2) where the separate passes moved
// three times that. Measured, all separate passes and these: 256x256 L=8 (36
// components, nf 1024) 1.42 -> 0.55 ms, 192x192x32 L=8 (1152, nf 768) 27.3 ->
// 9.8 ms, 96^3 L=4 (10, nf 384) 27.1 -> 8.3 ms; 2.7 to 3.2 TB/s along x, 1.8 to
// 2.8 along y and z. Neither memory nor VALU issue (47 to 58 %) is saturated: a
// workgroup loads, transforms and stores one after another, and a CU holds two. The
// pencils of a workgroup share 8 NT values of LDS (72 KB at 512 work-items); along y and z they are neighbours in
// x, 64 bytes at nf = 1024, and the tiles that share a line are neighbours on
// one XCD.
// ---------------------------------------------------------------------------

#define MR_TA_MAXTX 32

// LDS place of element e: one spare value per 8, so that the radix-8 writes
// (8 values apart) of neighbouring lanes fall in different banks.
__host__ __device__ inline int mr_ta_at(int e) { return e + (e >> 3); }

// Pencil p = i + n0 (j + n1 o) starts at s0 i + s1 j + s2 o, elements `es`
// apart; M of them replace the nf read.
struct mr_ta_axis {
    double2 *data;
    long long n0, n1, s0, s1, s2, es;
    int shift;   // centering: mode j is stored at (j + shift) mod M
};
// Where the last axis stores: value k along it of pencil (i, j, o = q) is
// centered element i + c1 j + cs k of component q0 + o.
struct mr_ta_out {
    float2 *out;
    const int *inv;   // mask rows, or null
    long long c1, cs, Ptr, q0, nm;
    int Nkz;
    double scale;
};

// One in-place stage over tp pencils of length n (mr_stage_reg with the padded
// places). CROP: the first inverse stage, whose inputs are the cropped modes of
// the fine pencil (length nf) times their deconvolution weights. A butterfly
// loads its first twiddle and forms the others as products of two lower ones
// (three roundings deep at most): the texture unit would bind the stage with
// seven 16-byte twiddle loads beside eight LDS reads.
template <int RR, bool INV, bool CROP, int NT>
__device__ __forceinline__ void mr_ta_stage(double2 *A, const double2 *tws, const double *dc,
                                            int nf, int n, int ns, int tp, int Ns,
                                            const mr_fdiv &mdv, const mr_fdiv &nsdv)
{
    constexpr int EMAX = CROP ? 4 * NT : 8 * NT;   // a crop keeps at most half the pencil
    constexpr int KMAX = (EMAX / RR + NT - 1) / NT;
    const int m = n / RR, nb = tp * m, pos = n - n / 2;
    double2 v[KMAX][RR];
#pragma unroll
    for (int k = 0; k < KMAX; ++k) {
        const int f = threadIdx.x + k * NT;
        if (f < nb) {
            const int p = (int)mr_fdiv_q(mdv, (unsigned)f), j = f - p * m;
            const double2 *a = A + p * ns;
#pragma unroll
            for (int r = 0; r < RR; ++r) {
                const int e = j + r * m;
                if (CROP) {
                    const double w = dc[e];
                    const double2 x = a[mr_ta_at(e < pos ? e : e + nf - n)];
                    v[k][r] = make_double2(x.x * w, x.y * w);
                } else {
                    v[k][r] = a[mr_ta_at(e)];
                }
            }
        }
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < KMAX; ++k) {
        const int f = threadIdx.x + k * NT;
        if (f < nb) {
            const int p = (int)mr_fdiv_q(mdv, (unsigned)f), j = f - p * m;
            const int jn = (int)mr_fdiv_q(nsdv, (unsigned)j), kk = j - jn * Ns;
            if constexpr (RR > 1) {
                if (Ns > 1) {
                    double2 w[RR];
                    w[1] = tws[Ns + kk - 1];
#pragma unroll
                    for (int r = 2; r < RR; ++r) w[r] = cmul(w[r / 2], w[r - r / 2]);
#pragma unroll
                    for (int r = 1; r < RR; ++r) v[k][r] = INV ? cmulc(w[r], v[k][r]) : cmul(w[r], v[k][r]);
                }
                bfly<RR, INV>(v[k]);
            }
            double2 *b = A + p * ns;
            const int o = jn * Ns * RR + kk;
#pragma unroll
            for (int q = 0; q < RR; ++q) b[mr_ta_at(o + q * Ns)] = v[k][q];
        }
    }
    __syncthreads();
}

template <bool INV, bool CROP, int NT>
__device__ __forceinline__ void mr_ta_stages(double2 *A, const mr_fft_len<double> &f,
                                             const double *dc, int nf, int s0, int s1, int ns,
                                             int tp)
{
    int Ns = 1;
    for (int s = 0; s < s1; ++s) {
        const int RR = f.radix[s];
        const mr_fdiv &md = f.mdiv[s], &nd = f.nsdiv[s];
#define MR_TA_ST(R)                                                                               \
    case R: mr_ta_stage<R, INV, CROP, NT>(A, f.tws, dc, nf, f.n, ns, tp, Ns, md, nd); break;
        if (s >= s0) {
            switch (RR) {
                MR_TA_ST(2) MR_TA_ST(3) MR_TA_ST(4) MR_TA_ST(5) MR_TA_ST(6) MR_TA_ST(7)
                MR_TA_ST(8) MR_TA_ST(10)
            default: break;
            }
        }
#undef MR_TA_ST
        Ns *= RR;
    }
}

// FAST: a pencil's elements are contiguous (es = 1). LAST: store to `o`.
template <bool FAST, bool LAST, int NT>
__global__ void __launch_bounds__(NT, 4)
mr_k_toep_axis(mr_fft_len<double> fn, mr_fft_len<double> fm, mr_ta_axis ax, mr_ta_out o,
               const double *__restrict__ dc, long long npencil, int TX, mr_fdiv txdiv,
               long long pbase)
{
    extern __shared__ __align__(16) unsigned char mr_smem[];
    double2 *A = reinterpret_cast<double2 *>(mr_smem);
    __shared__ long long base[MR_TA_MAXTX], cbase[MR_TA_MAXTX], comp[MR_TA_MAXTX];
    __shared__ int cz[MR_TA_MAXTX];
    const int nf = fn.n, M = fm.n, ns = mr_ta_at(nf) + 1;
    const long long p0 = pbase + mr_xcd_block(blockIdx.x, gridDim.x) * TX;
    const int tp = (int)((npencil - p0 < TX) ? (npencil - p0) : TX);
    if (threadIdx.x < tp) {
        const long long p = p0 + threadIdx.x;
        const long long r = p / ax.n0, i = p - r * ax.n0;
        const long long q = r / ax.n1, j = r - q * ax.n1;
        base[threadIdx.x] = ax.s0 * i + ax.s1 * j + ax.s2 * q;
        if (LAST) {
            const long long qq = o.q0 + q;
            cz[threadIdx.x] = (int)(qq % o.Nkz);
            cbase[threadIdx.x] = i + o.c1 * j + (o.inv ? 0 : o.Ptr * qq);
            comp[threadIdx.x] = qq / o.Nkz;
        }
    }
    __syncthreads();
    // all of a thread's loads before its LDS writes
    double2 t[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        const int q = threadIdx.x + k * NT;
        const int hi = (int)mr_fdiv_q(FAST ? fn.ndiv : txdiv, (unsigned)q);
        const int lo = q - hi * (FAST ? nf : TX);
        const int p = FAST ? hi : lo, e = FAST ? lo : hi;
        const bool in = p < tp && e < nf;
        t[k] = in ? ax.data[base[p] + (FAST ? e : ax.es * e)] : make_double2(0.0, 0.0);
    }
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        const int q = threadIdx.x + k * NT;
        const int hi = (int)mr_fdiv_q(FAST ? fn.ndiv : txdiv, (unsigned)q);
        const int lo = q - hi * (FAST ? nf : TX);
        const int p = FAST ? hi : lo, e = FAST ? lo : hi;
        if (p < tp && e < nf) A[p * ns + mr_ta_at(e)] = t[k];
    }
    __syncthreads();
    mr_ta_stages<false, false, NT>(A, fn, dc, nf, 0, fn.nst, ns, tp);
    if (fm.nst > 0) mr_ta_stages<true, true, NT>(A, fm, dc, nf, 0, 1, ns, tp);
    else mr_ta_stage<1, true, true, NT>(A, fm.tws, dc, nf, 1, ns, tp, 1, mr_fdiv{1, 0, 0},
                                        mr_fdiv{1, 0, 0});
    mr_ta_stages<true, false, NT>(A, fm, dc, nf, 1, fm.nst, ns, tp);
    auto put = [&](int p, int e) {
        int k = e + ax.shift;
        if (k >= M) k -= M;
        const double2 v = A[p * ns + mr_ta_at(e)];
        if (!LAST) {
            ax.data[base[p] + (FAST ? k : ax.es * k)] = v;
            return;
        }
        const float2 w = make_float2((float)(v.x * o.scale), (float)(v.y * o.scale));
        const long long c = cbase[p] + o.cs * k;
        if (!o.inv) {
            o.out[c] = w;
        } else {
            const int row = o.inv[c + o.Ptr * cz[p]];
            if (row >= 0) o.out[row + o.nm * comp[p]] = w;
        }
    };
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int q = threadIdx.x + k * NT;
        const int hi = (int)mr_fdiv_q(FAST ? fm.ndiv : txdiv, (unsigned)q);
        const int lo = q - hi * (FAST ? M : TX);
        const int p = FAST ? hi : lo, e = FAST ? lo : hi;
        if (p < tp && e < M) put(p, e);
    }
}

// inv[centered linear index] = mask row, -1 elsewhere
__global__ void mr_k_mask_rows(int *inv, long long P, const int64_t *mask, long long nm)
{
    const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= nm) return;
    const long long k = mask[t];
    if (k >= 0 && k < P) inv[k] = (int)t;
}
__global__ void mr_k_fill_i32(int *p, long long n, int v)
{
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

// Bytes of gridding scratch a build aims at per chunk of components.
#define MR_TOEP_CHUNK_BYTES (2LL << 30)

namespace {

struct toep_geom {
    int d;        // transformed axes
    int M[3];     // transformed grid (1 beyond d)
    int shift[3]; // centering shift per transformed axis
    long long Ptr;
    int Nkz;
    double scale;
};

toep_geom mr_toep_geom(const mr_config *cfg)
{
    toep_geom g;
    const bool three = cfg->traj_type == MR_TRAJ_3D;
    g.d = three ? 3 : 2;
    g.M[0] = cfg->phi2_dim[0];
    g.M[1] = cfg->phi2_dim[1];
    g.M[2] = three ? cfg->phi2_dim[2] : 1;
    for (int a = 0; a < 3; ++a) g.shift[a] = g.M[a] / 2;
    g.Ptr = (long long)g.M[0] * g.M[1] * g.M[2];
    g.Nkz = (cfg->traj_type == MR_TRAJ_STACK) ? cfg->phi2_dim[2] : 1;
    g.scale = 1.0 / (double)g.Ptr;
    return g;
}

// Inverse FFT over the transformed M grid of Qc natural-order volumes.
int mr_toep_ifft(const toep_geom &tg, double2 *nat, int Qc, hipStream_t s)
{
    mr_fft_len<double> f[3];
    for (int a = 0; a < tg.d; ++a) MR_TRY(mr_fft_get<double>(tg.M[a], &f[a]));
    const long long m0 = tg.M[0], m1 = tg.M[1], m2 = tg.M[2];
    MR_TRY((mr_fft_pass<double, true>(f[0], mr_ld_axis<double2, true>{nat, 1, (int)m0},
                                      mr_st_axis<double2, true>{nat, 1, (int)m0},
                                      m1 * m2 * Qc, 0, 4, s, "toep ifft x")));
    MR_TRY((mr_fft_pass<double, true>(f[1], mr_ld_axis<double2, false>{nat, m0, (int)m1},
                                      mr_st_axis<double2, false>{nat, m0, (int)m1},
                                      m0 * m2 * Qc, 0, 16, s, "toep ifft y")));
    if (tg.d == 3)
        MR_TRY((mr_fft_pass<double, true>(f[2], mr_ld_axis<double2, false>{nat, m0 * m1, (int)m2},
                                          mr_st_axis<double2, false>{nat, m0 * m1, (int)m2},
                                          m0 * m1 * Qc, 0, 16, s, "toep ifft z")));
    return MR_SUCCESS;
}

// Scratch of one call; its work on `s` has ended, or is waited for, before
// the blocks go back.
struct toep_bufs {
    hipStream_t s;
    bool done = false;
    mr_grid_samples smp;
    double2 *c = nullptr, *fine = nullptr, *nat = nullptr, *part = nullptr;
    double *dc[3] = {nullptr, nullptr, nullptr};
    int *inv = nullptr;
    explicit toep_bufs(hipStream_t st) : s(st) {}
    toep_bufs(const toep_bufs &) = delete;
    ~toep_bufs()
    {
        if (!done) (void)hipStreamSynchronize(s);
        void *bufs[] = {c, fine, nat, part, inv};
        for (void *p : bufs) mr_ws_put(p);
        for (double *p : dc) if (p) (void)hipFree(p);
        mr_grid_samples_free(&smp, true);
    }
};

int mr_build_mask_rows(const mr_config *cfg, const int64_t *mask, hipStream_t s, int **inv)
{
    const long long P = mr_pad_size(cfg), nm = cfg->num_masked;
    *inv = (int *)mr_ws_get(P * sizeof(int));
    if (!*inv) MR_FAIL(MR_ERR_ALLOC, "failed to allocate the mask rows of %lld locations", P);
    hipLaunchKernelGGL(mr_k_fill_i32, dim3((unsigned)mr_ceil_div(P, 256)), dim3(256), 0, s, *inv,
                       P, -1);
    MR_LAUNCH_CHECK("mr_k_fill_i32");
    hipLaunchKernelGGL(mr_k_mask_rows, dim3((unsigned)mr_ceil_div(nm, 256)), dim3(256), 0, s,
                       *inv, P, mask, nm);
    MR_LAUNCH_CHECK("mr_k_mask_rows");
    return MR_SUCCESS;
}

// Every axis of qn fine grids in place, then the store of components q0 ...
int mr_toep_axes(const toep_geom &tg, const mr_grid &g, double2 *fine, double *const *dc, int qn,
                 long long q0, const int *inv, long long nm, float2 *out, hipStream_t s)
{
    const long long nx = g.nf[0], ny = g.nf[1], nz = g.nf[2];
    const long long m0 = tg.M[0], m1 = tg.M[1];
    for (int a = 0; a < tg.d; ++a) {
        mr_fft_len<double> fn, fm;
        MR_TRY(mr_fft_get<double>(g.nf[a], &fn));
        MR_TRY(mr_fft_get<double>(tg.M[a], &fm));
        mr_ta_axis ax{fine, 0, 0, 0, 0, 0, 1, tg.shift[a]};
        long long np = 0;
        if (a == 0) {
            np = ny * nz * qn;
            ax.n0 = np; ax.n1 = 1; ax.s0 = nx;
        } else if (a == 1) {
            np = m0 * nz * qn;
            ax.n0 = m0; ax.n1 = nz; ax.s0 = 1; ax.s1 = nx * ny; ax.s2 = nx * ny * nz; ax.es = nx;
        } else {
            np = m0 * m1 * qn;
            ax.n0 = m0; ax.n1 = m1; ax.s0 = 1; ax.s1 = nx; ax.s2 = nx * ny * nz; ax.es = nx * ny;
        }
        const mr_ta_out o{out, inv, m0, a == 2 ? m0 * m1 : m0, tg.Ptr, q0, nm, tg.Nkz, tg.scale};
        const bool last = a == tg.d - 1;
        // 8 NT values per workgroup: 256 threads where whole pencils fill them
        // (more, smaller workgroups overlap their phases), else 512; along y
        // and z 512 threads for wider rows
        const int nf = g.nf[a];
        const bool small = a == 0 && 2048 / nf * nf >= 1740;
        const int NT = small ? 256 : 512;
        int TX = 8 * NT / nf;
        if (TX > MR_TA_MAXTX) TX = MR_TA_MAXTX;
        if (a > 0) TX = mr_pow2_floor(TX);
        const size_t lds = (size_t)TX * (mr_ta_at(nf) + 1) * sizeof(double2);
        auto fn_k = a == 0 ? (small ? mr_k_toep_axis<true, false, 256>
                                    : mr_k_toep_axis<true, false, 512>)
                           : last ? mr_k_toep_axis<false, true, 512>
                                  : mr_k_toep_axis<false, false, 512>;
        if (lds > 65536)
            MR_HIP_CHECK(hipFuncSetAttribute((const void *)fn_k,
                                             hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
        const long long blocks = mr_ceil_div(np, TX), maxb = mr_max_blocks(NT);
        for (long long b0 = 0; b0 < blocks; b0 += maxb) {
            const long long nb = blocks - b0 < maxb ? blocks - b0 : maxb;
            hipLaunchKernelGGL(fn_k, dim3((unsigned)nb), dim3(NT), lds, s, fn, fm, ax, o, dc[a], np,
                               TX, mr_fdiv_make((unsigned)TX), b0 * TX);
            MR_LAUNCH_CHECK("mr_k_toep_axis");
        }
    }
    return MR_SUCCESS;
}

// The same by separate passes, through the natural-order grids b.nat.
int mr_toep_separate(const toep_geom &tg, const mr_grid &g, const toep_bufs &b, int qn,
                     long long q0, long long nm, float2 *out, hipStream_t s)
{
    MR_TRY(mr_grid_fft(g, b.fine, nullptr, qn, false, s));
    MR_GRID_CHECK(mr_ceil_div(tg.Ptr * qn, 256), 256, "mr_k_deconv");
    hipLaunchKernelGGL(mr_k_deconv, dim3((unsigned)mr_ceil_div(tg.Ptr * qn, 256)), dim3(256), 0, s,
                       b.fine, g, tg.Ptr, qn, b.dc[0], b.dc[1], b.dc[2], b.nat);
    MR_LAUNCH_CHECK("mr_k_deconv");
    MR_TRY(mr_toep_ifft(tg, b.nat, qn, s));
    hipLaunchKernelGGL(mr_k_toep_store, dim3((unsigned)mr_ceil_div(tg.Ptr * qn, 256)), dim3(256), 0,
                       s, b.nat, tg.M[0], tg.M[1], tg.M[2], tg.shift[0], tg.shift[1], tg.shift[2],
                       tg.Ptr, qn, q0, tg.Nkz, tg.scale, b.inv, nm, out);
    MR_LAUNCH_CHECK("mr_k_toep_store");
    return MR_SUCCESS;
}

}  // namespace

int mr_calc_toep_impl(const mr_config *cfg, const mr_complex *d_phi2, const float *d_traj,
                      int64_t Ntrajs, int64_t Nkx, const int64_t *d_mask, mr_complex *d_out)
{
    hipStream_t s = (hipStream_t)cfg->stream;
    const toep_geom tg = mr_toep_geom(cfg);
    const int T = (int)mr_num_tri(cfg->L);
    const long long Q = (long long)T * tg.Nkz;

    mr_grid g;
    mr_grid_setup(&g, tg.d, tg.M, cfg->eps);
    toep_bufs b(s);
    mr_grid_samples &smp = b.smp;
    MR_TRY(mr_grid_samples_build(g, d_traj, Ntrajs, Nkx, s, &smp));

    b.c = (double2 *)mr_ws_get((Q * Ntrajs + MR_GRID_STR_PAD) * sizeof(double2));
    if (!b.c) MR_FAIL(MR_ERR_ALLOC, "failed to allocate the strengths of %lld components", Q);
    hipLaunchKernelGGL(mr_k_pack_strengths, dim3((unsigned)mr_ceil_div(Q * Ntrajs, 256)),
                       dim3(256), 0, s, reinterpret_cast<const float2 *>(d_phi2), (long long)Ntrajs,
                       tg.Nkz, cfg->L, cfg->triangulation == MR_TRI_UPPER ? 1 : 0, T, b.c);
    MR_LAUNCH_CHECK("mr_k_pack_strengths");
    MR_TRY(mr_grid_deconv(g, b.dc, s));
    if (cfg->is_masked) MR_TRY(mr_build_mask_rows(cfg, d_mask, s, &b.inv));

    // the one-pass axes need unrolled butterflies for the mode counts (the
    // fine counts always have them)
    bool onepass = true;
    for (int a = 0; a < tg.d; ++a)
        onepass = onepass && mr_fft_smooth(tg.M[a]) && g.nf[a] <= 4096;

    // Chunk of components: fine grids (and natural-order grids for the
    // separate passes) within budget.
    size_t budget = 0;
    MR_TRY(mr_mem_budget(cfg, &budget));
    const size_t per_q = ((size_t)g.nfine + (onepass ? 0 : (size_t)tg.Ptr) +
                          (size_t)smp.part_elems(1)) * sizeof(double2);
    long long Qc = (long long)(budget / 2 / per_q);
    // A chunk beyond a few GB gains nothing (192x192x32 L=8: 15.2 ms with 1.2 GB
    // chunks, 15.4 with all 10.9 GB), and giving that much memory back stalls
    // the call now and then (250 ms for 9 GB and more). Below four components a
    // spread has too few strengths for the weights it forms (96^3 L=4, 0.9 GB
    // each: 28 ms one at a time, 22.5 in twos, 19.4 in fours).
    long long fit = (long long)(MR_TOEP_CHUNK_BYTES / per_q);
    if (fit < 4) fit = 4;
    if (Qc > fit) Qc = mr_ceil_div(Q, mr_ceil_div(Q, fit));   // even chunks
    const long long cap = mr_env_ll("MR_AHA_TOEP_MAX_CHUNK", 0);
    if (cap > 0 && Qc > cap) Qc = cap;
    if (Qc > Q) Qc = Q;
    if (Qc > 65535LL * 16) Qc = 65535LL * 16;
    if (Qc < 1) Qc = 1;
    b.fine = (double2 *)mr_ws_get((size_t)g.nfine * Qc * sizeof(double2));
    if (!onepass) b.nat = (double2 *)mr_ws_get((size_t)tg.Ptr * Qc * sizeof(double2));
    if (smp.next > 0)
        b.part = (double2 *)mr_ws_get((size_t)smp.part_elems(Qc) * sizeof(double2));
    if (!b.fine || (!onepass && !b.nat) || (smp.next > 0 && !b.part)) {
        (void)hipGetLastError();
        MR_FAIL(MR_ERR_ALLOC,
                "failed to allocate the calc_toep chunk buffers (chunk = %lld); lower "
                "mr_config.mem_fraction or the upsampled grid size",
                Qc);
    }
    for (long long q0 = 0; q0 < Q; q0 += Qc) {
        const int qn = (int)((Q - q0 < Qc) ? Q - q0 : Qc);
        MR_TRY(mr_grid_spread(g, smp, b.c, (int)Q, (int)q0, qn, b.fine, b.part, s));
        if (onepass)
            MR_TRY(mr_toep_axes(tg, g, b.fine, b.dc, qn, q0, b.inv, (long long)cfg->num_masked,
                                reinterpret_cast<float2 *>(d_out), s));
        else
            MR_TRY(mr_toep_separate(tg, g, b, qn, q0, (long long)cfg->num_masked,
                                    reinterpret_cast<float2 *>(d_out), s));
        if (cfg->verbose)
            printf("[mr_aha] calc_toep: components %lld-%lld of %lld issued\n", q0, q0 + qn - 1, Q);
    }
    MR_HIP_CHECK(hipStreamSynchronize(s));
    b.done = true;
    return MR_SUCCESS;
}

extern "C" MR_EXPORT int mr_calc_toep(const mr_config *cfg, const mr_complex *d_phi2,
                                      const float *d_traj, int64_t Ntrajs, int64_t Nkx,
                                      const int64_t *d_mask, mr_complex *d_phi2_toep)
{
    mr_clear_error();
    MR_REQUIRE(cfg != nullptr, "mr_calc_toep: cfg is NULL");
    MR_REQUIRE(d_phi2 != nullptr, "mr_calc_toep: d_phi2 is NULL");
    MR_REQUIRE(d_traj != nullptr, "mr_calc_toep: d_traj is NULL");
    MR_REQUIRE(d_phi2_toep != nullptr, "mr_calc_toep: d_phi2_toep is NULL");
    MR_REQUIRE(Ntrajs > 0, "mr_calc_toep: Ntrajs = %lld must be > 0", (long long)Ntrajs);
    MR_REQUIRE(Nkx > 0, "mr_calc_toep: Nkx = %lld must be > 0", (long long)Nkx);
    if (cfg->is_masked)
        MR_REQUIRE(d_mask != nullptr, "mr_calc_toep: d_mask is required when is_masked is set");
    MR_TRY(mr_config_validate(cfg));
    int prev = -1;
    int rc = mr_push_device(cfg, &prev);
    if (rc == MR_SUCCESS)
        rc = mr_calc_toep_impl(cfg, d_phi2, d_traj, Ntrajs, Nkx, d_mask, d_phi2_toep);
    mr_pop_device(prev);
    return rc;
}

static int mr_calc_toep_from_psf_impl(const mr_config *cfg, const mr_complex *d_psf, int64_t t0,
                                      int64_t n_comp, const int64_t *d_mask, mr_complex *d_out)
{
    hipStream_t s = (hipStream_t)cfg->stream;
    const toep_geom tg = mr_toep_geom(cfg);
    const long long Qc = n_comp * tg.Nkz;
    toep_bufs b(s);
    if (cfg->is_masked) MR_TRY(mr_build_mask_rows(cfg, d_mask, s, &b.inv));
    b.nat = (double2 *)mr_ws_get((size_t)tg.Ptr * Qc * sizeof(double2));
    if (!b.nat) {
        (void)hipGetLastError();
        MR_FAIL(MR_ERR_ALLOC, "failed to allocate %lld scratch elements for mr_calc_toep_from_psf",
                tg.Ptr * Qc);
    }
    MR_GRID_CHECK(mr_ceil_div(tg.Ptr * Qc, 256), 256, "mr_k_psf_to_nat");
    hipLaunchKernelGGL(mr_k_psf_to_nat, dim3((unsigned)mr_ceil_div(tg.Ptr * Qc, 256)), dim3(256),
                       0, s, reinterpret_cast<const float2 *>(d_psf), tg.M[0], tg.M[1], tg.M[2],
                       tg.shift[0], tg.shift[1], tg.shift[2], tg.Ptr, (int)Qc, b.nat);
    MR_LAUNCH_CHECK("mr_k_psf_to_nat");
    MR_TRY(mr_toep_ifft(tg, b.nat, (int)Qc, s));
    hipLaunchKernelGGL(mr_k_toep_store, dim3((unsigned)mr_ceil_div(tg.Ptr * Qc, 256)), dim3(256),
                       0, s, b.nat, tg.M[0], tg.M[1], tg.M[2], tg.shift[0], tg.shift[1],
                       tg.shift[2], tg.Ptr, (int)Qc, (long long)t0 * tg.Nkz, tg.Nkz, tg.scale,
                       b.inv, (long long)cfg->num_masked, reinterpret_cast<float2 *>(d_out));
    MR_LAUNCH_CHECK("mr_k_toep_store");
    MR_HIP_CHECK(hipStreamSynchronize(s));
    b.done = true;
    return MR_SUCCESS;
}

extern "C" MR_EXPORT int mr_calc_toep_from_psf(const mr_config *cfg, const mr_complex *d_psf,
                                               int64_t t0, int64_t n_comp, const int64_t *d_mask,
                                               mr_complex *d_phi2_toep)
{
    mr_clear_error();
    MR_REQUIRE(cfg != nullptr, "mr_calc_toep_from_psf: cfg is NULL");
    MR_REQUIRE(d_psf != nullptr, "mr_calc_toep_from_psf: d_psf is NULL");
    MR_REQUIRE(d_phi2_toep != nullptr, "mr_calc_toep_from_psf: d_phi2_toep is NULL");
    MR_TRY(mr_config_validate(cfg));
    const int64_t ntri = mr_num_tri(cfg->L);
    MR_REQUIRE(t0 >= 0 && n_comp >= 1 && t0 + n_comp <= ntri,
               "mr_calc_toep_from_psf: components [%lld, %lld) outside [0, %lld)", (long long)t0,
               (long long)(t0 + n_comp), (long long)ntri);
    if (cfg->is_masked)
        MR_REQUIRE(d_mask != nullptr,
                   "mr_calc_toep_from_psf: d_mask is required when is_masked is set");
    int prev = -1;
    int rc = mr_push_device(cfg, &prev);
    if (rc == MR_SUCCESS) rc = mr_calc_toep_from_psf_impl(cfg, d_psf, t0, n_comp, d_mask, d_phi2_toep);
    mr_pop_device(prev);
    return rc;
}
