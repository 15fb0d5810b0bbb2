// Non-uniform gridding shared by the Toeplitz kernel build (type-1, sign -1)
// and the NUFFT operator (type-1 / type-2): exponential-of-semicircle (ES)
// kernel of Barnett, Magland and af Klinteberg, "A parallel non-uniform fast
// Fourier transform library based on an exponential of semicircle kernel",
// SIAM J. Sci. Comput. 41(5) (2019): width w = ceil(log10(1/eps)) + 1,
// phi(z) = exp(beta (sqrt(1 - z^2) - 1)), beta = 2.30 w, upsampling 2.
//
// Sample m at angle x (radians) sits at fine-grid coordinate u = x nf/(2 pi);
// it touches the w points i0 .. i0+w-1 with i0 = ceil(u - w/2) (mod nf) and
// weight phi(2 (i - u) / w). The fine grid is cut into bins of bs points per
// axis (bs divides nf); a sample belongs to the bin of its first point i0.
#pragma once

#include "mr_hip.hpp"

#define MR_GRID_MAXW 16

struct mr_grid {
    int d;           // transformed dimensions (2 or 3)
    int nf[3];       // fine grid, 1 beyond d
    int M[3];        // modes per axis, 1 beyond d
    int bs[3];       // bin size per axis
    int nb[3];       // bins per axis
    int w;           // kernel width
    double beta;
    long long nfine; // prod nf
    long long nbins; // prod nb
};

// Fill the geometry for `d` transformed axes with mode counts M[0..d-1].
void mr_grid_setup(mr_grid *g, int d, const int *M, double eps);

// Deconvolution factors 1/phi_hat(delta) of the modes of every transformed
// axis a < d in natural order (index j <-> delta = j or j - M), into dc[a]
// allocated here (the caller frees it), on `stream`. dc[a] of the other axes
// stays as it is: their only mode has factor one.
int mr_grid_deconv(const mr_grid &g, double **dc, hipStream_t stream);

// Candidate samples per segment of mr_k_spread: a wavefront's share of a tile.
// Large enough that few tiles are split (each extra segment costs a partial
// tile per strength set in memory), small enough that the last wavefront ends
// with the others (1024: the per-sample launch of a 192x192 comparator takes
// 0.31 ms instead of 0.09, a 256x256 L=8 build's 0.53 instead of 0.34).
#define MR_GRID_SEG 256

// Strength rows are read in chunks of up to this many sets, also past the
// last set of a row: the strength array ends with as many spare entries.
#define MR_GRID_STR_PAD 16

// Per-sample geometry, sorted by (bin, readout, readout position).
struct mr_grid_samples {
    long long n = 0;        // samples
    int *i0 = nullptr;      // [n * 3] first fine point per axis (mod nf), sorted order
    int *rd = nullptr;      // [n] readout of each sorted sample
    double *wt = nullptr;   // [n * d * w] weights per axis, sorted order
    int *start = nullptr;   // [nbins + 1] first sorted sample of bin >= b
    long long next = 0;     // segments beyond the first of their tile
    int2 *ext = nullptr;    // [next] (tile, segment number >= 1), ascending
    // scratch values (double2) that spreading Q sets needs for them
    long long part_elems(long long Q) const { return next * 64 * Q; }
};

// Build the sorted sample table from a [Ntrajs, Nkx, ndim] trajectory
// (first `g.d` coordinates used) on `stream`. Synchronous.
int mr_grid_samples_build(const mr_grid &g, const float *traj, long long Ntrajs, long long Nkx,
                          hipStream_t stream, mr_grid_samples *out);
// Give the tables back to the kept scratch; unless `idle` (no work that uses
// them is pending) the device is waited for first, as hipFree would.
void mr_grid_samples_free(mr_grid_samples *s, bool idle);

// Type-1 spreading of Q strength sets (strength of a sample of readout s, set
// q: str[s * qs + q0 + q], i.e. constant along a readout) onto Q fine
// grids fine[q * nfine + g], complex double. Gather formulation: every fine
// point sums the samples of the bins that can reach it; no atomics. `part`
// holds part_elems(Q) values.
int mr_grid_spread(const mr_grid &g, const mr_grid_samples &s, const double2 *str, int qs, int q0,
                   int Q, double2 *fine, double2 *part, hipStream_t stream);

// Same with per-sample strengths str[i * Q + q] of sorted sample i.
int mr_grid_spread_samples(const mr_grid &g, const mr_grid_samples &s, const double2 *str,
                           int Q, double2 *fine, double2 *part, hipStream_t stream);

// Type-2 interpolation: out[i * Q + q] = sum_points fine[q][p] weight of
// sorted sample i.
int mr_grid_interp(const mr_grid &g, const mr_grid_samples &s, const double2 *fine, int Q,
                   double2 *out, hipStream_t stream);

// Forward or inverse FFT of Q fine grids in place (double precision).
int mr_grid_fft(const mr_grid &g, double2 *fine, double2 *scratch, int Q, bool inverse,
                hipStream_t stream);
