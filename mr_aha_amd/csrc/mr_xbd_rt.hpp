// Fused x pass at a run-time x length (mr_xbd_rt.hip).
#pragma once

#include "mr_hip.hpp"

// LDS values per work-item of a workgroup: 512 work-items hold 80 KB of
// pencils (two workgroups per CU), 1024 have room for 160 KB (one) and are given
// up to 128 KB (MR_XBD_EMAX values).
#define MR_RT_EPT 20
#define MR_RT_MAXST 16

// x / D for x < 2^15 as (x * mul) >> shr with mul = ceil(2^shr / D),
// shr = 15 + ceil(log2 D): the excess x (mul D - 2^shr) / (D 2^shr) stays below
// 2^-ceil(log2 D) <= 1 / D, so the floor is exact, and x * mul < 2^32 comes
// from one 24-bit multiply (mul <= 2^16).
struct mr_d24 {
    unsigned mul, shr;
};
__host__ __device__ inline constexpr mr_d24 mr_d24_make(unsigned d)
{
    unsigned l = 0;
    while ((1u << l) < d) ++l;
    const unsigned k = 15 + l;
    return mr_d24{(unsigned)(((1ull << k) + d - 1) / d), k};
}

// Per-length plan, by value in the kernel arguments.
struct mr_rt_len {
    int n, nst;
    int radix[MR_RT_MAXST], m[MR_RT_MAXST];   // radix and n / radix of each stage
    mr_d24 md[MR_RT_MAXST], nd[MR_RT_MAXST];  // division by m and by the earlier radices' product
};
bool mr_rt_len_make(const mr_fft_len<float> &fx, mr_rt_len *f);

typedef void (*mr_xbd_rt_fn)(float2 *, const float2 *, const int *, long long, mr_dims, mr_rt_len,
                             const float2 *, long long, int, int, int);
// Kernel for rank L (1 .. 16) with nt = 512 or 1024 work-items, or nullptr.
mr_xbd_rt_fn mr_xbd_rt_pick(int L, bool masked, int nt);
