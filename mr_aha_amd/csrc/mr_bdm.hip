// Block multiply of ranks 17 .. 80 on the matrix cores, in place over the
// padded k-space grids of the separate-pass route: at every grid location
// y_o = sum_r v_r A_ro with A Hermitian from its packed triangle, for each
// coil (src/cuda/mr_kernels_bdt.cu:218-416). K is [P, L, ncoil] in natural
// order, the kernel [T, kstride] centered (or [T, num_masked] with the inverse
// mask map).
//
// Per location this is a (coils) x L by L x L product in FP32, done with
// v_mfma_f32_16x16x4_f32: rows are coils, columns 16 outputs, 4 rows r of the
// block at a time. A workgroup owns 8 (or 16) consecutive locations and as many
// wavefronts; a wavefront computes one location, its inputs and all its outputs
// in registers.
//  * The inputs and then the kernel stream through two LDS buffers in tiles of
//    16 x 16: read once, coalesced over locations, and each wavefront reads its
//    own location's tile back as operands. The next two tiles are in flight in
//    registers meanwhile, and there is one barrier per tile.
//  * A tile (rows R, columns C) of the stored triangle is used twice while it
//    is in LDS: as is for the outputs C, conjugated and transposed for the
//    outputs R. So the kernel is read once.
//  * Odd LDS strides (locations, tile rows) spread the operand reads, plain and
//    transposed, over the banks.
//  * Complex products: from 9 coils on the 16 rows are coils, with the real and
//    imaginary inputs as two operands and two accumulators per output tile.
//    Up to 8 coils the rows are (coil, part), the second operand holds
//    (-imaginary, real), and one accumulator receives both products.
//
// Bound: memory, then the staging. 640x640 grid, L = 72, 12 coils moves 14.3 GB
// (kernel 8.6, inputs and outputs 5.7) in 3.92 ms, 3.6 TB/s, where the tiled
// kernel took 7.45 ms (whole 320x320 apply 10.7 -> 7.37 ms); without the kernel
// loads it takes 2.8 ms, its matrix instructions alone 1.9 ms.
// Why ranks up to 80: a wavefront holds 8 registers of inputs and 8 (4 up to 8
// coils) of outputs per 16 ranks, 80 of its 128 at rank 80.
#include "mr_xbd.hpp"
#include "mr_fft_ct.hpp"

#include <algorithm>
#include <utility>

namespace {

typedef float mr_f4 __attribute__((ext_vector_type(4)));

constexpr int BDM_S = 17;     // LDS stride of tile rows, in tile entries
constexpr int BDM_MAXL = 80;

template <class F, int... I>
__device__ __forceinline__ void bdm_each(F &&f, std::integer_sequence<int, I...>)
{
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F> __device__ __forceinline__ void bdm_for(F &&f)
{
    bdm_each(f, std::make_integer_sequence<int, N>{});
}

// Tile n of the triangle's tiles in the order (0,0), (1,0), (1,1), (2,0), ...
constexpr int bdm_row(int n)
{
    int r = 0;
    while (n > r) n -= ++r;
    return r;
}
constexpr int bdm_col(int n)
{
    int r = 0;
    while (n > r) n -= ++r;
    return n;
}

// NT: tiles of 16 ranks, NM: 8 coils per operand row set (1: up to 8, 2: up to
// 16), TP: locations and wavefronts per workgroup
template <int NT, int NM, int TP, bool MASKED>
__global__ void __launch_bounds__(64 * TP, NT == 2 ? 8 : 4)
mr_k_bdm(float2 *__restrict__ K, const float2 *__restrict__ ker, const int *__restrict__ inv,
         long long kstride, mr_dims d, int ncoil, int nbat, long long tile0)
{
    constexpr int NC = 8 * NM, NB = NT * (NT + 1) / 2, NI = NT + NB, NV = NC / 4;
    constexpr int PD = 2;   // tiles in flight; 3 to 5 measured no better at any rank
    constexpr int E = TP + 1, BUF = 16 * BDM_S * E;   // LDS stride of tile entries, tile
    __shared__ float2 lds[2][BUF];
    const int L = d.L;
    const bool upper = d.tri_upper != 0;
    const long long P = d.pad_size;
    const long long lb = mr_xcd_block(blockIdx.x, gridDim.x);
    const long long tq = lb / nbat, tile = tile0 + tq;
    const int cb = (int)(lb - tq * nbat) * NC;
    const int nb = ncoil - cb < NC ? ncoil - cb : NC;
    // staging: location p, row or coil q1 (+ 4 i, uniform in a wavefront), column or rank q0
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int p = threadIdx.x % TP, q0 = (threadIdx.x / TP) & 15, q1 = w * 4 / TP;
    const long long loc = tile * TP + p;
    long long kb = -1;
    if (loc < P) kb = MASKED ? (long long)inv[loc] : mr_nat_to_cent_lin(loc, d);
    // inputs and outputs of this location
    float2 *kv = K + (loc < P ? loc : P - 1) + P * (long long)L * cb;
    if (MASKED && !__syncthreads_or(kb >= 0)) {
        if (loc < P)
            for (int e = threadIdx.x / TP; e < nb * L; e += 64) kv[P * e] = make_float2(0.f, 0.f);
        return;
    }
    const float2 *kp = ker + (kb >= 0 ? kb : 0);

    const int flip = upper ? (int)0x80000000 : 0;
    float2 pre[PD][4];
    // This work-item's share of item `it` (input tile `it`, then the kernel's):
    // a wavefront's loads differ in a wave-uniform row (coil), so one 64-bit
    // lane offset serves all four. Unconditional loads, the last entry (coil)
    // in place of one that does not exist, and nothing done to the values
    // before they are staged: a branch or a sign here made the compiler wait
    // for every load by itself.
    auto load = [&](auto I) {
        constexpr int it = decltype(I)::value;
        if constexpr (it < NT) {
            const int r = it < NT - 1 || 16 * it + q0 < L ? 16 * it + q0 : L - 1;
            const float2 *v = kv + P * r;
#pragma unroll
            for (int i = 0; i < NV; ++i) {
                const int c = q1 + 4 * i < nb ? q1 + 4 * i : nb - 1;
                pre[it % PD][i] = v[P * L * c];
            }
        } else if constexpr (it < NI) {
            constexpr int R = bdm_row(it - NT), C = bdm_col(it - NT);
            const int c = C < NT - 1 || 16 * C + q0 < L ? 16 * C + q0 : L - 1;
            const float2 *a = kp + kstride * (upper ? c : c * L - c * (c + 1) / 2);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int rr = 16 * R + q1 + 4 * i;
                const int r = R < NT - 1 || rr < L ? rr : L - 1;
                pre[it % PD][i] = a[kstride * (upper ? r * (r + 1) / 2 : r)];
            }
        }
    };

    const int lane = threadIdx.x & 63;
    const int li = lane & 15, lg = lane >> 4;
    float u0[4 * NT], u1[4 * NT];
    mr_f4 acc[NM][NT];
#pragma unroll
    for (int m = 0; m < NM; ++m)
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[m][t] = mr_f4{0.f, 0.f, 0.f, 0.f};
    // outputs of tile O += inputs of rows (4 ks + lg) of tile V times x + i y
    auto mul = [&](int O, int u, float x, float y) {
        acc[0][O] = __builtin_amdgcn_mfma_f32_16x16x4f32(u0[u], x, acc[0][O], 0, 0, 0);
        if constexpr (NM == 1) {
            acc[0][O] = __builtin_amdgcn_mfma_f32_16x16x4f32(u1[u], y, acc[0][O], 0, 0, 0);
        } else {
            acc[1][O] = __builtin_amdgcn_mfma_f32_16x16x4f32(u0[u], y, acc[1][O], 0, 0, 0);
            acc[0][O] = __builtin_amdgcn_mfma_f32_16x16x4f32(u1[u], -y, acc[0][O], 0, 0, 0);
            acc[1][O] = __builtin_amdgcn_mfma_f32_16x16x4f32(u1[u], x, acc[1][O], 0, 0, 0);
        }
    };

    bdm_for<PD>(load);
    bdm_for<NI>([&](auto I) {
        constexpr int it = decltype(I)::value;
        float2 *b = lds[it & 1];
        if constexpr (it < NT) {
#pragma unroll
            for (int i = 0; i < NV; ++i)
                b[((q1 + 4 * i) * BDM_S + q0) * E + p] =
                    it < NT - 1 || 16 * it + q0 < L ? pre[it % PD][i] : make_float2(0.f, 0.f);
        } else {
            constexpr int R = bdm_row(it - NT);
            constexpr bool diag = R == bdm_col(it - NT);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int r = q1 + 4 * i;
                float2 a = pre[it % PD][i];
                if (R == NT - 1 && 16 * R + r >= L) a = make_float2(0.f, 0.f);
                // the upper triangle stores A_cr = conj(A_rc)
                if (!diag || r != q0) a.y = __int_as_float(__float_as_int(a.y) ^ flip);
                if (!diag || q0 <= r) b[(r * BDM_S + q0) * E + p] = a;
                if (diag && q0 < r) b[(q0 * BDM_S + r) * E + p] = make_float2(a.x, -a.y);
            }
        }
        load(std::integral_constant<int, it + PD>{});
        mr_lds_barrier();
        if constexpr (it < NT) {
            const int c = NM == 1 ? li >> 1 : li;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const float2 v = b[(c * BDM_S + 4 * k + lg) * E + w];
                u0[4 * it + k] = NM == 1 && (li & 1) ? v.y : v.x;
                u1[4 * it + k] = NM == 2 ? v.y : (li & 1) ? v.x : -v.y;
            }
        } else {
            constexpr int R = bdm_row(it - NT), C = bdm_col(it - NT);
            float2 a[4], h[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                a[k] = b[((4 * k + lg) * BDM_S + li) * E + w];
                if constexpr (R != C) h[k] = b[(li * BDM_S + 4 * k + lg) * E + w];
            }
#pragma unroll
            for (int k = 0; k < 4; ++k)
                if (R < NT - 1 || 16 * R + 4 * k < L) mul(C, 4 * R + k, a[k].x, a[k].y);
            if constexpr (R != C) {
#pragma unroll
                for (int k = 0; k < 4; ++k) mul(R, 4 * C + k, h[k].x, -h[k].y);
            }
        }
    });
    // outputs back through LDS, a tile of 16 ranks at a time; the indexes are
    // formed anew behind an empty asm instead of held through the tiles
    unsigned ot = threadIdx.x;
    asm volatile("" : "+v"(ot));
    const int op = ot % TP, o0 = (ot / TP) & 15;
    const long long oloc = tile * TP + op;
    const bool keep = oloc < P && (!MASKED || inv[oloc] >= 0);
    float2 *ov = K + oloc + P * (long long)L * cb;
    bdm_for<NT>([&](auto T) {
        constexpr int t = decltype(T)::value;
        float2 *b = lds[(NI + t) & 1];
        if constexpr (NM == 1) {
#pragma unroll
            for (int j = 0; j < 2; ++j)
                b[((2 * lg + j) * BDM_S + li) * E + w] =
                    make_float2(acc[0][t][2 * j], acc[0][t][2 * j + 1]);
        } else {
#pragma unroll
            for (int j = 0; j < 4; ++j)
                b[((4 * lg + j) * BDM_S + li) * E + w] = make_float2(acc[0][t][j], acc[1][t][j]);
        }
        mr_lds_barrier();
        const int r = 16 * t + o0;
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            const int c = q1 + 4 * i;
            if (oloc < P && r < L && c < nb)
                ov[P * ((long long)L * c + r)] =
                    keep ? b[(c * BDM_S + o0) * E + op] : make_float2(0.f, 0.f);
        }
    });
}

typedef void (*mr_bdm_fn)(float2 *, const float2 *, const int *, long long, mr_dims, int, int,
                          long long);

template <int NM, int TP, bool MASKED> mr_bdm_fn bdm_fn(int nt)
{
    switch (nt) {
    case 2: return mr_k_bdm<2, NM, TP, MASKED>;
    case 3: return mr_k_bdm<3, NM, TP, MASKED>;
    case 4: return mr_k_bdm<4, NM, TP, MASKED>;
    default: return mr_k_bdm<5, NM, TP, MASKED>;
    }
}

template <int NM> mr_bdm_fn bdm_fn_wide(int nt)
{
    return nt == 4 ? mr_k_bdm<4, NM, 16, false> : mr_k_bdm<5, NM, 16, false>;
}

}  // namespace

// Launch the matrix-core block multiply over K [P, L, nc], or return false
// where the tiled kernel (mr_bdt.hip) takes the call. *rc receives the status
// of a launch.
//
// The products on padding (ranks up to a multiple of 16, coils up to 8 or 16)
// decide: with a fifth of the products useful or more this kernel is faster.
// Measured, tiled -> this (us; useful part): L=72 C=2 at 512x512 2309 -> 2177
// (0.20), L=65 C=3 at 384x384 1318 -> 852 (0.25), L=17 C=16 at 512x512 567 ->
// 558 (0.28), L=20 C=8 at 400x400 208 -> 185 (0.39), L=48 C=16 at 384x384 1489
// -> 813 (1); below, L=17 C=4 at 400x400 110 -> 158 (0.14), L=33 C=2 at 320x320
// 173 -> 204 (0.12).
bool mr_bdm_launch(const mr_dims &d, float2 *K, const float2 *ker, const int *inv,
                   long long kstride, int nc, bool masked, hipStream_t s, int *rc)
{
    if (d.L <= 16 || d.L > BDM_MAXL || nc < 1) return false;
    const int nt = (d.L + 15) / 16;
    const int nm = nc > 8 ? 2 : 1;
    const int nbat = (int)mr_ceil_div(nc, 8 * nm);
    if (5LL * d.L * d.L * nc < 256LL * nt * nt * 8 * nm * nbat) return false;
    // Kernel entries 2 MB (a multiple) apart fall in the same sets of the
    // caches, which lose the other half of a line before the workgroup next
    // door has read it: whole lines of 16 locations there (512x512 L=72: 12
    // coils 3.77 -> 3.45 ms, 2 coils 2.77 -> 2.18 ms). Elsewhere two
    // workgroups of 8 per CU are better, one loads while the other multiplies
    // (640x640 L=72, 12 coils 4.15 -> 3.92 ms, 384x384 L=65 0.90 -> 0.85 ms).
    const bool lines = !masked && nt >= 4 && kstride % (1 << 18) == 0;
    const int TP = lines ? 16 : 8;
    mr_bdm_fn fn;
    if (lines) fn = nm == 2 ? bdm_fn_wide<2>(nt) : bdm_fn_wide<1>(nt);
    else if (nm == 2) fn = masked ? bdm_fn<2, 8, true>(nt) : bdm_fn<2, 8, false>(nt);
    else fn = masked ? bdm_fn<1, 8, true>(nt) : bdm_fn<1, 8, false>(nt);
    const long long tiles = mr_ceil_div(d.pad_size, TP);
    // a dispatch counts its work-items in 32 bits: chunks of whole tiles
    const long long step = std::max(1LL, mr_max_blocks(64 * TP) / nbat);
    *rc = [&]() -> int {
        for (long long t0 = 0; t0 < tiles; t0 += step) {
            const long long blocks = std::min(step, tiles - t0) * nbat;
            hipLaunchKernelGGL(fn, dim3((unsigned)blocks), dim3(64 * TP), 0, s, K, ker, inv,
                               kstride, d, nc, nbat, t0);
            MR_LAUNCH_CHECK("mr_k_bdm");
        }
        return MR_SUCCESS;
    }();
    return true;
}
