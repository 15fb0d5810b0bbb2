// Fused x pass for any smooth x grid length (radices 2 .. 8 and 10) and any
// rank up to 16: the shapes without a kernel of mr_xbd_ct.hip. The rank is a
// template parameter (the block walks keep their outputs in registers), the
// length is not.
//
// When the outer axes are transformed on the image side first, the x axis is
// the last one: for one k-space row r = (ky, kz) (natural order) the forward
// x-FFT, the block multiply of the row's Mx locations and the inverse x-FFT
// need nothing outside the row. One workgroup takes the row for a group of up
// to G coils of Y [Nx, R, V] (R = My*Mz rows, V = L * coils):
//   load   the L*G pencils of Nx image columns, zero-padded to Mx in natural
//          order (pad map of src/cuda/mr_kernels.cu:111-128)
//   FFT    forward, radix stages in LDS
//   block  v <- v B(k) at each of the Mx locations; the row's T*Mx kernel
//          entries are read coalesced (centered kx runs contiguously except at
//          the one wrap point) and shared, through L2, by the G coils and by
//          the coil groups of the row, which are consecutive workgroups of
//          one XCD (src/cuda/mr_kernels_bd.cu:74-139 for the walk)
//   IFFT   inverse
//   store  the Nx image columns back in place (crop of mr_kernels.cu:158-165)
// Padded k-space never reaches HBM: per row and coil the pass moves 2*L*Nx
// values plus the kernel row.
//
// What it spends its time on is VALU and LDS issue, one phase after another (55 and
// 36 % of its cycles at 240x216x40, 15 points of the latter bank conflicts), so
// it takes over what it can of the compiled-length kernels: the coil-pair walks
// with two entries per 16-byte load (unmasked kernels), the half-empty first stage
// and the cropped last one where the image fills the
// centred half of the pencil, divisions as one full-rate 24-bit multiply,
// 16-byte image loads and stores. Every twiddle is read from the table (the
// compiled kernels form powers of one, which is a little less exact). What stays is
// an add per LDS access (the butterfly strides are not immediates). Measured against
// the kernel before it (one coil per walk, 8-byte entries, all eight inputs read): 240x216x40,
// grid 480x432x40, L=6, 10 coils, masked 5.66 -> 3.11 ms (5.1 GB, 1.6 TB/s);
// 225x198, grid 450x396, L=5, 7 coils 91 -> 65 us. Ranks 14 to 16 spill 4 to 36
// registers (20 to 96 bytes of scratch a lane) and are faster all the same: 112x96x12, 8
// coils, L=14, 15, 16: 731 -> 539, 792 -> 574, 867 -> 693 us.

#pragma once

#include "mr_xbd.hpp"
#include "mr_fft_ct.hpp"
#include "mr_xbd_rt.hpp"

namespace {

__device__ __forceinline__ unsigned mr_d24_q(const mr_d24 &d, unsigned x)
{
    return __umul24(x, d.mul) >> d.shr;
}

// One Stockham stage in place over tp pencils of length N (stride N), as
// mr_ct_stage: phase 1 reads every butterfly input and twiddle of the thread
// into registers, phase 2 (after the barrier) writes the outputs; rounds are
// skipped per wavefront, lanes past the last butterfly repeat it.
// PR = 1: the first forward stage (radix 8) of a centred half-filled pencil,
// inputs 2 .. 5 zero and not read; PR = 2: the last inverse stage of one,
// outputs in the dropped middle half not stored.
template <int RR, bool INV, int PR, int NT>
__device__ __forceinline__ void mr_rt_stage(float2 *A, const mr_tw_buf &tw, int N, int tp, int wave,
                                            int m, int Ns, const mr_d24 &md, const mr_d24 &nd)
{
    static_assert(PR != 1 || RR == 8, "padded first stage");
    constexpr int KMAX = (MR_RT_EPT + RR - 1) / RR;   // N * tp <= MR_RT_EPT * NT
    const int nb = tp * m;
    const unsigned tid = threadIdx.x;
    float2 v[KMAX][RR];
#pragma unroll
    for (int k = 0; k < KMAX; ++k) {
        if (k * NT + wave * 64 < nb) {
            const unsigned f = min(tid + k * NT, (unsigned)(nb - 1));
            const unsigned p = mr_d24_q(md, f), j = f - p * m;
            const float2 *a = A + p * N + j;
#pragma unroll
            for (int r = 0; r < RR; ++r)
                if (PR != 1 || r < 2 || r > 5) v[k][r] = a[r * m];
        }
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < KMAX; ++k) {
        if (k * NT + wave * 64 < nb) {
            const unsigned f = min(tid + k * NT, (unsigned)(nb - 1));
            const unsigned p = mr_d24_q(md, f), j = f - p * m;
            const unsigned jn = mr_d24_q(nd, j), kk = j - jn * Ns;
            if (PR != 1 && Ns > 1) {
                float2 w[RR];
#pragma unroll
                for (int r = 1; r < RR; ++r) w[r] = tw.get(Ns - 1 + kk, (unsigned)((r - 1) * Ns));
#pragma unroll
                for (int r = 1; r < RR; ++r)
                    v[k][r] = INV ? cmulc(w[r], v[k][r]) : cmul(w[r], v[k][r]);
            }
            if constexpr (PR == 1) bfly8_ends<INV>(v[k]);
            else bfly<RR, INV>(v[k]);
            float2 *b = A + p * N + jn * (Ns * RR) + kk;
            if (RR % 2 == 0 && PR != 2 && Ns == 1) {
                // RR adjacent outputs (N is even, so they are 16-byte aligned)
#pragma unroll
                for (int q = 0; q + 1 < RR; q += 2)
                    *reinterpret_cast<mr_u32x4_ct *>(b + q) = mr_u32x4_ct{
                        __float_as_uint(v[k][q].x), __float_as_uint(v[k][q].y),
                        __float_as_uint(v[k][q + 1].x), __float_as_uint(v[k][q + 1].y)};
            } else {
#pragma unroll
                for (int q = 0; q < RR; ++q)
                    if (PR != 2 || !(4 * q >= RR && 4 * (q + 1) <= 3 * RR)) b[q * Ns] = v[k][q];
            }
        }
    }
    __syncthreads();
}

// The transform; TRIM: the image fills the centred half of the pencil (first
// radix 8, more than one stage).
template <bool INV, int NT>
__device__ __forceinline__ void mr_rt_fft(float2 *A, const mr_tw_buf &tw, const mr_rt_len &f, int tp,
                                          int wave, bool trim)
{
    int s = 0, Ns = 1, end = f.nst;
    if (!INV && trim) {
        mr_rt_stage<8, false, 1, NT>(A, tw, f.n, tp, wave, f.m[0], 1, f.md[0], f.nd[0]);
        s = 1;
        Ns = 8;
    }
    if (INV && trim) --end;
    for (; s < end; ++s) {
        const int RR = f.radix[s], m = f.m[s];
        const mr_d24 md = f.md[s], nd = f.nd[s];
        switch (RR) {
#define MR_RT_ST(R)                                                                       \
    case R: mr_rt_stage<R, INV, 0, NT>(A, tw, f.n, tp, wave, m, Ns, md, nd); break;
            MR_RT_ST(2) MR_RT_ST(3) MR_RT_ST(4) MR_RT_ST(5) MR_RT_ST(6) MR_RT_ST(7) MR_RT_ST(10)
#undef MR_RT_ST
        default: mr_rt_stage<8, INV, 0, NT>(A, tw, f.n, tp, wave, m, Ns, md, nd); break;
        }
        Ns *= RR;
    }
    if (INV && trim) {
        const int m = f.m[s];
        const mr_d24 md = f.md[s], nd = f.nd[s];
        switch (f.radix[s]) {
#define MR_RT_ST(R)                                                                       \
    case R: mr_rt_stage<R, INV, 2, NT>(A, tw, f.n, tp, wave, m, Ns, md, nd); break;
            MR_RT_ST(2) MR_RT_ST(3) MR_RT_ST(4) MR_RT_ST(5) MR_RT_ST(6) MR_RT_ST(7) MR_RT_ST(10)
#undef MR_RT_ST
        default: mr_rt_stage<8, INV, 2, NT>(A, tw, f.n, tp, wave, m, Ns, md, nd); break;
        }
    }
}

template <int L, bool MASKED, int NT>
__global__ void __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(4)))
mr_k_xbd_rt(float2 *__restrict__ Y, const float2 *__restrict__ ker, const int *__restrict__ inv,
            long long kstride, mr_dims d, mr_rt_len f, const float2 *tws, long long R, int G,
            int ncoil, int ncg)
{
    constexpr int NW = NT / 64;
    extern __shared__ __align__(16) unsigned char mr_smem[];
    float2 *A = reinterpret_cast<float2 *>(mr_smem);
    const int Nx = d.n[0], N = f.n, cnx = d.c_n[0];
    const long long q = mr_xcd_block(blockIdx.x, gridDim.x);
    const long long r = q / ncg;
    const int c0 = (int)(q - r * ncg) * G;
    const int gn = (ncoil - c0 < G) ? ncoil - c0 : G;
    const int tp = gn * L;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const mr_tw_buf twb{mr_rsrc(tws, (unsigned)N * 8u)};
    // pencil pl = g*L + l of the workgroup is volume v = L*c0 + pl; every
    // wavefront loads and stores whole pencils, so a pencil's base is uniform
    const float2 *Yr = Y + (long long)Nx * r + (long long)Nx * R * L * c0;
    const long long pstride = (long long)Nx * R;
    const unsigned rowbytes = (unsigned)Nx * 8u;
    // two points per lane where the pencils and their slots pair up (Nx a
    // multiple of 4, so Nx, cnx = Nx/2 and N are even; 16-byte aligned rows)
    const bool px = (Nx & 3) == 0 && (cnx & 1) == 0 && (N & 1) == 0 &&
                    ((unsigned long long)Y & 15) == 0;
    const bool trim = f.nst >= 2 && f.radix[0] == 8 && 2 * Nx == N && 4 * cnx == N;
    for (int pl = wave; pl < tp; pl += NW) {
        const __amdgpu_buffer_rsrc_t rs = mr_rsrc(Yr + pstride * pl, rowbytes);
        float2 *Ap = A + pl * N;
        if (px) {
            for (int s0 = 0; s0 < Nx; s0 += 512) {
                mr_u32x4_ct v[4];
#pragma unroll
                for (int c = 0; c < 4; ++c)
                    if (s0 + c * 128 < Nx)
                        v[c] = __builtin_amdgcn_raw_buffer_load_b128(
                            rs, (s0 + c * 128 + 2 * lane) * 8, 0, 0);
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    const int s = s0 + c * 128 + 2 * lane;
                    int e = s - cnx;
                    if (e < 0) e += N;
                    if (s < Nx) *reinterpret_cast<mr_u32x4_ct *>(Ap + e) = v[c];
                }
            }
        } else {
            for (int s0 = 0; s0 < Nx; s0 += 256) {
                float2 v[4];
#pragma unroll
                for (int c = 0; c < 4; ++c)
                    if (s0 + c * 64 < Nx) v[c] = mr_bload(rs, (unsigned)(s0 + c * 64 + lane) * 8u);
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    const int s = s0 + c * 64 + lane;
                    int e = s - cnx;
                    if (e < 0) e += N;
                    if (s < Nx) Ap[e] = v[c];
                }
            }
        }
        if (!trim)
            for (int i = lane; i < N - Nx; i += 64) {
                int e = Nx + i - cnx;
                if (e >= N) e -= N;
                if (e < 0) e += N;
                Ap[e] = make_float2(0.f, 0.f);
            }
    }
    __syncthreads();
    mr_rt_fft<false, NT>(A, twb, f, tp, wave, trim);

    // block step: a wavefront per 64 locations of a coil pair (an odd last
    // coil walks alone)
    const int My = d.m[1];
    const int jy = (int)(r % My), jz = (int)(r / My);
    int ky = jy + d.c_m[1]; if (ky >= My) ky -= My;
    int kz = jz + d.c_m[2]; if (kz >= d.m[2]) kz -= d.m[2];
    const long long rowc = (long long)N * (ky + (long long)My * kz);
    const int nblk = (N + 63) >> 6;
    // entries two per 16-byte load (mr_bd_walk_pair_x2): unmasked, N and the
    // kx centering shift even (a pair of adjacent locations has adjacent
    // entries from an even index on), whole 64-location blocks
    const bool x2 = !MASKED && (N & 1) == 0 && (d.c_m[0] & 1) == 0 &&
                    ((unsigned long long)ker & 15) == 0;
    for (int t = wave; t < ((gn + 1) >> 1) * nblk; t += NW) {
        const int pq = t / nblk, e0 = (t - pq * nblk) * 64;
        const bool full = x2 && e0 + 64 <= N;
        const bool two = 2 * pq + 1 < gn;
        const int hi = lane >> 5;
        const int e = e0 + (full ? ((lane & 31) << 1) + hi : lane);
        if (e >= N) continue;
        long long b;
        if (MASKED) {
            b = inv[e + (long long)N * r];
        } else {
            int kx = e + d.c_m[0];
            if (kx >= N) kx -= N;
            b = rowc + kx;
        }
        float2 *a0 = A + 2 * pq * L * N + e, *a1 = a0 + L * N;
        const unsigned bo = (unsigned)(b * 8);
        if (MASKED && b < 0) {
#pragma unroll
            for (int l = 0; l < L; ++l) {
                a0[l * N] = make_float2(0.f, 0.f);
                if (two) a1[l * N] = make_float2(0.f, 0.f);
            }
        } else if (!MASKED && full) {
            const unsigned bp = (unsigned)((b - hi) * 8 + (hi ? kstride * 8 : 0));
            if (two) {
                if (d.tri_upper) mr_bd_walk_pair_x2<L, true, 4>(a0, a1, N, ker, kstride, bp, bo);
                else if constexpr (L % 2 == 0) mr_bd_walk_pair_x2c<L, 4>(a0, a1, N, ker, kstride, bp, bo);
                else mr_bd_walk_pair_x2<L, false, 4>(a0, a1, N, ker, kstride, bp, bo);
            } else {
                if (d.tri_upper) mr_bd_walk_pair_x2<L, true, 8, 1>(a0, a0, N, ker, kstride, bp, bo);
                else if constexpr (L % 2 == 0) mr_bd_walk_pair_x2c<L, 8, 1>(a0, a0, N, ker, kstride, bp, bo);
                else mr_bd_walk_pair_x2<L, false, 8, 1>(a0, a0, N, ker, kstride, bp, bo);
            }
        } else if (two) {
            if (d.tri_upper) mr_bd_walk_pair<L, true, (L > 8 ? 8 : 16)>(a0, a1, N, ker, kstride, bo);
            else mr_bd_walk_pair<L, false, (L > 8 ? 8 : 16)>(a0, a1, N, ker, kstride, bo);
        } else {
            if (d.tri_upper) mr_bd_walk_g<L, true>(a0, N, ker, kstride, bo);
            else mr_bd_walk_g<L, false>(a0, N, ker, kstride, bo);
        }
    }
    __syncthreads();
    mr_rt_fft<true, NT>(A, twb, f, tp, wave, trim);

    for (int pl = wave; pl < tp; pl += NW) {
        const __amdgpu_buffer_rsrc_t rs = mr_rsrc(Yr + pstride * pl, rowbytes);
        const float2 *Ap = A + pl * N;
        if (px) {
            for (int s = 2 * lane; s < Nx; s += 128) {
                int e = s - cnx;
                if (e < 0) e += N;
                __builtin_amdgcn_raw_buffer_store_b128(*reinterpret_cast<const mr_u32x4_ct *>(Ap + e),
                                                       rs, s * 8, 0, 0);
            }
        } else {
            for (int s = lane; s < Nx; s += 64) {
                int e = s - cnx;
                if (e < 0) e += N;
                mr_bstore(rs, (unsigned)s * 8u, Ap[e]);
            }
        }
    }
}

template <bool MASKED, int NT> mr_xbd_rt_fn mr_rt_pick(int L)
{
    switch (L) {
#define MR_XBD_CASE(n) case n: return mr_k_xbd_rt<n, MASKED, NT>;
        MR_XBD_CASE(1) MR_XBD_CASE(2) MR_XBD_CASE(3) MR_XBD_CASE(4)
        MR_XBD_CASE(5) MR_XBD_CASE(6) MR_XBD_CASE(7) MR_XBD_CASE(8)
        MR_XBD_CASE(9) MR_XBD_CASE(10) MR_XBD_CASE(11) MR_XBD_CASE(12)
        MR_XBD_CASE(13) MR_XBD_CASE(14) MR_XBD_CASE(15) MR_XBD_CASE(16)
#undef MR_XBD_CASE
    default: return nullptr;
    }
}

}  // namespace
