// Forms of the run-time-length axis passes (mr_axis_rt.hip) and how many of
// their workgroups a CU holds. No device code: the rules run on the host alone.
#pragma once

// Work-items, elements per work-item (the tile's registers) and pencils of a
// tile of length n. Up to 256 every form keeps 8 elements and 16 pencils (whole
// lines), so that short lengths do not leave lanes of a butterfly round idle. Up
// to 384, 512 work-items with 12 elements: two workgroups per CU overlap their
// phases, where 1024 with 8 leave one (320 along z of 160^3, L=8, 8 coils:
// inverse 1.57 against 2.50 ms; 288 along y of 144^3: 1.34 against 1.66). Up to
// 512 the y passes take 1024 work-items (432: 0.87 and 0.75 ms, 512 with 16
// elements 0.89 and 0.78). The outer passes take 8 pencils there, and also below
// when whole lines would give a CU fewer than two tiles (2D: 225x198, 396 along
// y, inverse 40 us against 51 with 16 pencils). Beyond 512 the one-tile kernels
// are as fast or faster (2D 640: inverse 56 us against 73).
struct ax_form {
    int nt, ke, pt;
};
constexpr ax_form ax_pick(int n, bool outer, bool few)
{
    if (n <= 64) return {128, 8, 16};
    if (n <= 128) return {256, 8, 16};
    if (n <= 256) return {512, 8, 16};
    if (outer && (few || n > 384)) return {512, 8, 8};
    if (n <= 384) return {512, 12, 16};
    return {1024, 8, 16};
}

enum ax_kind { AX_Y, AX_FO, AX_IO };   // y passes, forward and inverse outer passes

// Wavefronts per SIMD of a kernel: its launch bound, so the registers allow
// them. `big`: the kernels with radices 11 and 13.
constexpr int ax_waves(ax_kind k, int ke, bool big)
{
    if (k == AX_Y) return ke > 8 ? (big ? 5 : 6) : big ? 7 : 8;
    if (k == AX_FO) return ke > 8 ? 4 : big ? 5 : 6;
    return ke > 8 || big ? 4 : 5;
}

constexpr int AX_LDS = 163840;
constexpr int ax_lds(const ax_form &f, int n) { return n * (f.pt + 1) * 8; }

// Workgroups per CU, by registers (four SIMDs) and LDS. The tiles are dealt out
// to the workgroups when they start, so a workgroup that only starts once
// another has ended does its share alone at the end: with three workgroups per
// CU where the registers hold two, the forward outer pass of 81x81x150, L=6, 5
// coils (length 300) took 268 us instead of 225, with four y workgroups instead
// of three 300 along y of 150x150x12, L=8, 8 coils 113 instead of 106 us.
constexpr int ax_per_cu(ax_kind k, const ax_form &f, bool big, int n)
{
    const int by_regs = 4 * ax_waves(k, f.ke, big) * 64 / f.nt, by_lds = AX_LDS / ax_lds(f, n);
    const int per = by_regs < by_lds ? by_regs : by_lds;
    return per < 1 ? 1 : per;
}
