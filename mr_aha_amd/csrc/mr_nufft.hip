// method = MR_OP_NUFFT engine: per coil a type-2 NUFFT (sign -1), the
// per-readout Gram multiply k'_l = sum_j k_j B(j, l), and a type-1 NUFFT
// (sign +1) back (reference: src/cuda/mr_nufft_op.cu:613-700,
// python/mr_aha/nufft.py:473-552). For a stack the image is modulated by
// zmod(z) = exp(2 pi i floor(Nz/2) z / Nz), transformed along z with the
// unnormalised DFT pair, and kz plane K uses the Gram blocks of plane K.
//
// MI355X realisation: FP64 ES gridding of mr_grid.hip (the same sorted
// sample table serves the type-2 interpolation and the type-1 gather
// spreading), FP64 fine-grid FFTs of the project FFT engine. The L (x Nkz)
// transforms of several coils go through every stage in one launch: a 2D
// operator's coil alone is ten launches of 5 to 90 us that leave most of the
// chip idle. Padding, deconvolution and the sensitivity product are part of the
// first transform pass, cropping of the last ones, and the passes skip the
// lines that are zero or not kept. 192x192 L=4, 4 coils, 128 x 384 samples:
// apply
// 876 -> 450 us, 222 us with the gridding's part (mr_grid.hip).

#include "mr_grid.hpp"

#include <algorithm>
#include <new>

// Work memory of one launch's coils. Enough to fill the chip (a 2D coil takes 10
// to 100 MB); a coil that needs more runs alone, as in any size before.
#define MR_NU_BATCH_MB 1024

struct mr_nufft_eng {
    mr_config cfg;
    hipStream_t s;
    mr_grid g;
    mr_grid_samples smp;
    int d;          // NUFFT dimensions
    int Nkz;        // kz planes (stack) or 1
    int Q;          // transforms per coil: L * Nkz
    int nb;         // coils per launch
    long long Nimg; // image voxels
    long long Ntrajs, Nkx, Mnu;
    float2 *phi2;   // Gram blocks [Ntrajs, Nkz, L, L]
    double *dc[3];
    double2 *img;   // [Nimg, L, nb] (z fastest after x, y): image-side work
    double2 *acc;   // [Nimg, L] coil sum (several batches of coils)
    double2 *fine;  // [Q nb, nfine]
    double2 *tmp;   // k1 and k2, or the half-transformed grids
    double2 *k1;    // [Mnu (sorted samples)][Q nb]
    double2 *k2;    // [Mnu][Q nb], plus the spare entries of a strength array
    double2 *part;  // scratch of the spreading
    mr_fft_len<double> fz;
};

// Buffers whose size goes with the coils per launch
static void mr_nufft_free_batch(mr_nufft_eng *e)
{
    double2 **bufs[] = {&e->img, &e->acc, &e->fine, &e->tmp, &e->part};
    for (double2 **p : bufs) {
        if (*p) (void)hipFree(*p);
        *p = nullptr;
    }
}

static void mr_nufft_free(mr_nufft_eng *e)
{
    mr_grid_samples_free(&e->smp, false);
    for (double *p : e->dc) if (p) (void)hipFree(p);
    if (e->phi2) (void)hipFree(e->phi2);
    mr_nufft_free_batch(e);
    delete e;
}

void mr_nufft_eng_destroy(mr_nufft_eng *e)
{
    if (e) mr_nufft_free(e);
}

// The host side alone (see mr_aha_plan_abandon).
void mr_nufft_eng_abandon(mr_nufft_eng *e) { delete e; }

int mr_nufft_eng_create(const mr_config *cfg, const mr_complex *d_phi2, const float *d_traj,
                        int64_t Ntrajs, int64_t Nkx, double upsampfac, mr_nufft_eng **out)
{
    *out = nullptr;
    if (upsampfac != 0.0 && upsampfac != 2.0)
        MR_FAIL(MR_ERR_UNSUPPORTED, "mr_op_create: nufft_upsampfac = %g; this build grids with 2.0",
                upsampfac);
    mr_nufft_eng *e = new (std::nothrow) mr_nufft_eng();
    if (!e) MR_FAIL(MR_ERR_ALLOC, "failed to allocate the NUFFT engine");
    e->cfg = *cfg;
    e->s = (hipStream_t)cfg->stream;
    const bool three = cfg->traj_type == MR_TRAJ_3D;
    e->d = three ? 3 : 2;
    e->Nkz = (cfg->traj_type == MR_TRAJ_STACK) ? cfg->n_dim[2] : 1;
    e->Q = cfg->L * e->Nkz;
    e->Nimg = mr_image_size(cfg);
    e->Ntrajs = Ntrajs;
    e->Nkx = Nkx;
    e->Mnu = Ntrajs * Nkx;
    int modes[3] = {cfg->n_dim[0], cfg->n_dim[1], three ? cfg->n_dim[2] : 1};
    mr_grid_setup(&e->g, e->d, modes, cfg->eps);
    int rc = mr_grid_samples_build(e->g, d_traj, Ntrajs, Nkx, e->s, &e->smp);
    if (rc != MR_SUCCESS) { mr_nufft_free(e); return rc; }
    const size_t phi2_bytes = (size_t)Ntrajs * e->Nkz * cfg->L * cfg->L * sizeof(float2);
    // values per coil: image, fine grids, samples (twice) or the grids with
    // their last axis still at image size, partial tiles
    const long long Q = e->Q, nhalf = e->g.nfine / e->g.nf[e->d - 1] * e->g.M[e->d - 1];
    const long long tmp = std::max(2 * Q * e->Mnu, Q * nhalf);
    const long long per = e->Nimg * cfg->L + Q * e->g.nfine + tmp + e->smp.part_elems(Q);
    // coils per launch: as many as fit MR_NU_BATCH_MB
    // (MR_AHA_HIP_NU_MB overrides it) and the memory budget, evened out; sets are
    // counted in grid.y. Fewer where the device has no room for them after all.
    size_t budget = 0;
    rc = mr_mem_budget(cfg, &budget);
    if (rc != MR_SUCCESS) { mr_nufft_free(e); return rc; }
    const long long most = std::min<long long>(mr_env_ll("MR_AHA_HIP_NU_MB", MR_NU_BATCH_MB) * (1LL << 20),
                                               (long long)budget);
    const size_t img_bytes = (size_t)e->Nimg * cfg->L * sizeof(double2);
    long long nb = std::min<long long>(most / (16 * per), 65535 / Q);
    nb = std::max(1LL, std::min<long long>(nb, cfg->n_coils));
    hipError_t he = mr_dev_malloc((void **)&e->phi2, phi2_bytes);
    for (; he == hipSuccess; nb /= 2) {
        nb = mr_ceil_div(cfg->n_coils, mr_ceil_div(cfg->n_coils, nb));
        e->nb = (int)nb;
        he = mr_dev_malloc((void **)&e->img, img_bytes * nb);
        if (he == hipSuccess && nb < cfg->n_coils) he = mr_dev_malloc((void **)&e->acc, img_bytes);
        if (he == hipSuccess)
            he = mr_dev_malloc((void **)&e->fine, (size_t)(nb * Q * e->g.nfine) * sizeof(double2));
        if (he == hipSuccess)
            he = mr_dev_malloc((void **)&e->tmp, (size_t)(nb * tmp + MR_GRID_STR_PAD) * sizeof(double2));
        if (he == hipSuccess && e->smp.next > 0)
            he = mr_dev_malloc((void **)&e->part, (size_t)e->smp.part_elems(nb * Q) * sizeof(double2));
        if (he == hipSuccess || nb == 1) break;
        (void)hipGetLastError();
        mr_nufft_free_batch(e);
        he = hipSuccess;
    }
    e->k1 = e->tmp;
    e->k2 = e->tmp + nb * Q * e->Mnu;
    if (he == hipSuccess) {
        rc = mr_grid_deconv(e->g, e->dc, e->s);
        if (rc != MR_SUCCESS) { mr_nufft_free(e); return rc; }
    }
    if (he == hipSuccess)
        he = hipMemcpyAsync(e->phi2, d_phi2, phi2_bytes, hipMemcpyDeviceToDevice, e->s);
    if (he == hipSuccess) he = hipStreamSynchronize(e->s);
    if (he != hipSuccess) {
        (void)hipGetLastError();
        mr_nufft_free(e);
        MR_FAIL(MR_ERR_ALLOC, "failed to allocate the NUFFT engine buffers: %s", hipGetErrorString(he));
    }
    if (e->Nkz > 1) {
        rc = mr_fft_get<double>(e->Nkz, &e->fz);
        if (rc != MR_SUCCESS) { mr_nufft_free(e); return rc; }
    }
    *out = e;
    return MR_SUCCESS;
}

// Stack: img[i + Nimg (l + L c)] = S_c[i] x_l[i] zmod(z), `n` values
__global__ void mr_k_nu_img(const float2 *x, const float2 *S, long long Nimg, long long NxNy, int L,
                            int Nz, long long n, double2 *img)
{
    const long long id = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (id >= n) return;
    const long long v = id / Nimg, i = id - v * Nimg;
    const int c = (int)(v / L);
    const float2 xv = x[i + Nimg * (v - (long long)c * L)], sv = S[i + Nimg * c];
    const double re = (double)sv.x * xv.x - (double)sv.y * xv.y;
    const double im = (double)sv.x * xv.y + (double)sv.y * xv.x;
    const long long z = i / NxNy;
    double sn, cs;
    sincospi(2.0 * (double)((Nz / 2) * z % Nz) / Nz, &sn, &cs);
    img[id] = make_double2(re * cs - im * sn, re * sn + im * cs);
}

// Pixel weights: the product of the axes' deconvolution factors at centered
// image coordinates (iy, iz); along x at element s of the row.
struct mr_nu_row {
    int N[3];
    const double *dc[3];   // natural order; null beyond the transformed axes
    __device__ double axis(int a, int i) const
    {
        if (!dc[a]) return 1.0;
        int j = i - N[a] / 2;
        if (j < 0) j += N[a];
        return dc[a][j];
    }
};

// First pass of the type-2 transform, along x: pencil p = image row (y, z) of
// transform q, element e of nf = image column (e + N/2) mod nf times the
// deconvolution weights, zero outside. PROD: the image is S_c x_l (q = l + L c),
// else `img` holds it.
template <bool PROD> struct mr_nu_ld_x {
    static constexpr bool kElemFast = true;
    struct PB {
        long long x, S;
        double w;
    };
    mr_nu_row r;
    int nf, L;
    long long Nvol;
    const float2 *x, *S;
    const double2 *img;
    __device__ int nsub() const { return 1; }
    __device__ PB pencil(long long p, int) const
    {
        const long long rows = (long long)r.N[1] * r.N[2], q = p / rows;
        const int row = (int)(p - q * rows), z = row / r.N[1], y = row - z * r.N[1];
        PB b;
        const long long c = PROD ? q / L : 0;
        b.x = (long long)r.N[0] * row + Nvol * (q - c * L);
        b.S = (long long)r.N[0] * row + Nvol * c;
        b.w = r.axis(1, y) * r.axis(2, z);
        return b;
    }
    __device__ double2 get(const PB &b, int e) const
    {
        int s = e + r.N[0] / 2;
        if (s >= nf) s -= nf;
        if (s >= r.N[0]) return make_double2(0.0, 0.0);
        const double w = r.axis(0, s) * b.w;
        if constexpr (PROD) {
            const float2 xv = x[b.x + s], sv = S[b.S + s];
            return make_double2(((double)sv.x * xv.x - (double)sv.y * xv.y) * w,
                                ((double)sv.x * xv.y + (double)sv.y * xv.x) * w);
        } else {
            const double2 v = img[b.x + s];
            return make_double2(v.x * w, v.y * w);
        }
    }
};

// Last pass of the type-1 transform, along x: the kept columns of image row
// (y, z), weighted, to img[q].
struct mr_nu_st_x {
    static constexpr bool kElemFast = true;
    struct PB {
        long long o;
        double w;
    };
    mr_nu_row r;
    int nf;
    long long Nvol;
    double2 *img;
    __device__ PB pencil(long long p, int) const
    {
        const long long rows = (long long)r.N[1] * r.N[2], q = p / rows;
        const int row = (int)(p - q * rows), z = row / r.N[1], y = row - z * r.N[1];
        PB b;
        b.o = (long long)r.N[0] * row + Nvol * q;
        b.w = r.axis(1, y) * r.axis(2, z);
        return b;
    }
    __device__ void put(const PB &b, int, int e, int, double2 v, double2 *) const
    {
        int s = e + r.N[0] / 2;
        if (s >= nf) s -= nf;
        if (s >= r.N[0]) return;
        const double w = r.axis(0, s) * b.w;
        img[b.o + s] = make_double2(v.x * w, v.y * w);
    }
    __device__ void flush(long long, int, double2 *) const {}
};

// k2[i, K + Nkz (l + L c)] = sum_j k1[i, K + Nkz (j + L c)] B_{rd(i),K}(j, l)
__global__ void mr_k_nu_gram(const double2 *k1, const float2 *phi2, const int *rd, long long n,
                             long long Ntrajs, int Nkz, int L, int nc, double2 *k2)
{
    const long long id = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (id >= n) return;   // (K, c, i), K fastest
    const long long ic = id / Nkz, i = ic / nc;
    const int K = (int)(id - ic * Nkz);
    const float2 *B = phi2 + rd[i] + Ntrajs * (long long)K;  // entry (j,l) at + Ntrajs*Nkz*(j + L*l)
    const long long bs = Ntrajs * Nkz, row = ic * Nkz * L + K;
    for (int l = 0; l < L; ++l) {
        double re = 0.0, im = 0.0;
        for (int j = 0; j < L; ++j) {
            const double2 v = k1[row + (long long)Nkz * j];
            const float2 b = B[bs * (j + (long long)L * l)];
            re += v.x * b.x - v.y * b.y;
            im += v.x * b.y + v.y * b.x;
        }
        k2[row + (long long)Nkz * l] = make_double2(re, im);
    }
}

// Coil sum of conj(S_c zmod) img_c over nc coils in order, on top of acc unless
// `first`; to `out` when the last coil is in, else to acc.
__global__ void mr_k_nu_acc(const double2 *img, const float2 *S, long long Nimg, long long NxNy, int L,
                            int Nz, int stack, int nc, int first, double2 *acc, float2 *out)
{
    const long long id = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (id >= Nimg * L) return;
    const long long i = id % Nimg;
    double sn = 0.0, cs = 1.0;
    if (stack) sincospi(2.0 * (double)((Nz / 2) * (i / NxNy) % Nz) / Nz, &sn, &cs);
    double2 a = first ? make_double2(0.0, 0.0) : acc[id];
    for (int c = 0; c < nc; ++c) {
        const float2 sv = S[i + Nimg * c];
        double sr = sv.x, si = sv.y;
        if (stack) {
            const double r2 = sr * cs - si * sn, i2 = sr * sn + si * cs;
            sr = r2;
            si = i2;
        }
        const double2 v = img[id + Nimg * L * c];
        a.x += sr * v.x + si * v.y;
        a.y += sr * v.y - si * v.x;
    }
    if (out) out[id] = make_float2((float)a.x, (float)a.y);
    else acc[id] = a;
}

static int mr_nu_zfft(mr_nufft_eng *e, int nc, bool inverse)
{
    const long long NxNy = (long long)e->cfg.n_dim[0] * e->cfg.n_dim[1];
    const int Nz = e->Nkz;
    mr_ld_axis<double2, false> ld{e->img, NxNy, Nz};
    mr_st_axis<double2, false> st{e->img, NxNy, Nz};
    if (inverse)
        return mr_fft_pass<double, true>(e->fz, ld, st, NxNy * e->cfg.L * nc, 0, 16, e->s, "nufft z");
    return mr_fft_pass<double, false>(e->fz, ld, st, NxNy * e->cfg.L * nc, 0, 16, e->s, "nufft z");
}

// Fine-grid transforms of QB sets, image (S x, or e->img of a stack) -> fine:
// each axis is padded as it is transformed, so the passes along x and y run over
// image-sized remaining axes only.
static int mr_nu_forward(mr_nufft_eng *e, const mr_nu_row &r, const float2 *x, const float2 *S,
                         long long Nvol, bool prod, int QB)
{
    const mr_grid &g = e->g;
    const long long fx = g.nf[0], fy = g.nf[1], n1 = r.N[1], n2 = r.N[2];
    mr_fft_len<double> f[3];
    for (int a = 0; a < g.d; ++a) MR_TRY(mr_fft_get<double>(g.nf[a], &f[a]));
    // the halfway grids alternate so that the last pass ends in fine
    double2 *tx = g.d == 2 ? e->tmp : e->fine;
    const mr_st_axis<double2, true> sx{tx, 1, (int)fx};
    if (prod)
        MR_TRY((mr_fft_pass<double, false>(f[0], mr_nu_ld_x<true>{r, (int)fx, e->cfg.L, Nvol, x, S, nullptr},
                                           sx, n1 * n2 * QB, 0, 4, e->s, "nufft x")));
    else
        MR_TRY((mr_fft_pass<double, false>(f[0], mr_nu_ld_x<false>{r, (int)fx, 1, Nvol, nullptr, nullptr, e->img},
                                           sx, n1 * n2 * QB, 0, 4, e->s, "nufft x")));
    double2 *ty = g.d == 2 ? e->fine : e->tmp;
    MR_TRY((mr_fft_pass<double, false>(
        f[1], mr_ld_pad<double2, false>{tx, fx, (int)fy, (int)n1, (int)n1 / 2},
        mr_st_axis<double2, false>{ty, fx, (int)fy}, fx * n2 * QB, 0, 16, e->s, "nufft y")));
    if (g.d == 3)
        MR_TRY((mr_fft_pass<double, false>(
            f[2], mr_ld_pad<double2, false>{ty, fx * fy, g.nf[2], (int)n2, (int)n2 / 2},
            mr_st_axis<double2, false>{e->fine, fx * fy, g.nf[2]}, fx * fy * QB, 0, 16, e->s,
            "nufft z")));
    return MR_SUCCESS;
}

// The same back: fine -> e->img, each axis cropped as it is transformed.
static int mr_nu_inverse(mr_nufft_eng *e, const mr_nu_row &r, long long Nvol, int QB)
{
    const mr_grid &g = e->g;
    const long long fx = g.nf[0], fy = g.nf[1], n1 = r.N[1], n2 = r.N[2];
    mr_fft_len<double> f[3];
    for (int a = 0; a < g.d; ++a) MR_TRY(mr_fft_get<double>(g.nf[a], &f[a]));
    double2 *ty = g.d == 2 ? e->fine : e->tmp, *tx = g.d == 2 ? e->tmp : e->fine;
    if (g.d == 3)
        MR_TRY((mr_fft_pass<double, true>(
            f[2], mr_ld_axis<double2, false>{e->fine, fx * fy, g.nf[2]},
            mr_st_crop<double2, false>{ty, fx * fy, g.nf[2], (int)n2, (int)n2 / 2}, fx * fy * QB, 0,
            16, e->s, "nufft z")));
    MR_TRY((mr_fft_pass<double, true>(
        f[1], mr_ld_axis<double2, false>{ty, fx, (int)fy},
        mr_st_crop<double2, false>{tx, fx, (int)fy, (int)n1, (int)n1 / 2}, fx * n2 * QB, 0, 16, e->s,
        "nufft y")));
    return mr_fft_pass<double, true>(f[0], mr_ld_axis<double2, true>{tx, 1, (int)fx},
                                     mr_nu_st_x{r, (int)fx, Nvol, e->img}, n1 * n2 * QB, 0, 4, e->s,
                                     "nufft x");
}

int mr_nufft_eng_execute(mr_nufft_eng *e, const mr_complex *d_x, const mr_complex *d_SEs,
                         mr_complex *d_out)
{
    const mr_config &c = e->cfg;
    const int L = c.L;
    const bool stack = e->Nkz > 1 || c.traj_type == MR_TRAJ_STACK;
    const long long NxNy = (long long)c.n_dim[0] * c.n_dim[1];
    const long long Nvol = stack ? NxNy : e->Nimg;
    const auto *x = reinterpret_cast<const float2 *>(d_x);
    const auto *S = reinterpret_cast<const float2 *>(d_SEs);
    mr_nu_row r;
    for (int a = 0; a < 3; ++a) {
        r.N[a] = e->g.M[a];
        r.dc[a] = a < e->d ? e->dc[a] : nullptr;
    }
    for (int c0 = 0; c0 < c.n_coils; c0 += e->nb) {
        const int nc = std::min(e->nb, c.n_coils - c0), QB = e->Q * nc;
        const float2 *Sc = S + e->Nimg * c0;
        if (stack) {
            const long long n = e->Nimg * L * nc;
            hipLaunchKernelGGL(mr_k_nu_img, dim3((unsigned)mr_ceil_div(n, 256)), dim3(256), 0, e->s,
                               x, Sc, e->Nimg, NxNy, L, c.n_dim[2], n, e->img);
            MR_LAUNCH_CHECK("mr_k_nu_img");
            if (e->Nkz > 1) MR_TRY(mr_nu_zfft(e, nc, false));
        }
        MR_TRY(mr_nu_forward(e, r, x, Sc, Nvol, !stack, QB));
        MR_TRY(mr_grid_interp(e->g, e->smp, e->fine, QB, e->k1, e->s));
        const long long ng = e->Mnu * e->Nkz * nc;
        hipLaunchKernelGGL(mr_k_nu_gram, dim3((unsigned)mr_ceil_div(ng, 256)), dim3(256), 0, e->s,
                           e->k1, e->phi2, e->smp.rd, ng, e->Ntrajs, e->Nkz, L, nc, e->k2);
        MR_LAUNCH_CHECK("mr_k_nu_gram");
        MR_TRY(mr_grid_spread_samples(e->g, e->smp, e->k2, QB, e->fine, e->part, e->s));
        MR_TRY(mr_nu_inverse(e, r, Nvol, QB));
        if (e->Nkz > 1) MR_TRY(mr_nu_zfft(e, nc, true));
        hipLaunchKernelGGL(mr_k_nu_acc, dim3((unsigned)mr_ceil_div(e->Nimg * L, 256)), dim3(256), 0,
                           e->s, e->img, Sc, e->Nimg, NxNy, L, c.n_dim[2], stack ? 1 : 0, nc,
                           c0 == 0 ? 1 : 0, e->acc,
                           c0 + nc == c.n_coils ? reinterpret_cast<float2 *>(d_out) : nullptr);
        MR_LAUNCH_CHECK("mr_k_nu_acc");
    }
    return MR_SUCCESS;
}
