// Axis passes of the x-last pipeline at run-time lengths (mr_axis_rt.hip): the
// y transforms and the outer transforms with the sensitivity product or the
// coil sum, for any length up to MR_AX_NMAX made of the radices 2 .. 8, 10, 11
// and 13, any pencil stride and any alignment.
#pragma once

#include "mr_hip.hpp"
#include "mr_xbd_rt.hpp"

#define MR_AX_NMAX 512

// y pass: pencil p = i + I o; element e reads row (e + c_in) mod n of a column
// of n_in rows (zero past them) and is written to row (e + c_out) mod n of a
// column of n_out rows (dropped past them).
struct mr_ax_y {
    const float2 *in;
    float2 *out;
    long long I;
    int n_in, c_in, n_out, c_out;
};

// Outer passes: plane positions i < plane, ranks l < L, coils coil0 .. + nc - 1.
// Forward: element e = S_c x_l at image row z = (e + cz) mod n (zero for
// z >= nz), transformed, to work[i + plane (e + n v)], v = l + L c.
// Inverse: the transform of work, element e -> image row z, times conj(S_c),
// summed over the coils in order, to out[i + plane z + N l] (added to it when
// `accumulate`).
struct mr_ax_z {
    const float2 *x, *S;
    float2 *work, *out;
    long long plane, N;
    int nz, cz, L, nc, coil0, accumulate;
};

// Launch the pass and return the pencils of its tiles, or return 0 when the
// length is not one of these (or MR_AHA_HIP_AXRT=0). *rc receives the status of
// a launched pass.
int mr_axis_rt_y(const mr_fft_len<float> &f, bool inverse, const mr_ax_y &a, long long npencil,
                  hipStream_t s, int *rc);
int mr_axis_rt_z(const mr_fft_len<float> &f, bool inverse, const mr_ax_z &a, hipStream_t s, int *rc);
