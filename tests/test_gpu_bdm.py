"""The matrix-core block multiply (ranks 17 .. 80) at the edges of its tiles:
ranks around the multiples of 16 and the last rank it takes, coil counts around
its row sets of 8 and 16, grids that are not whole tiles of 16 locations, masks
that leave whole tiles out, both triangles, complex diagonals, and the form for
kernel rows 2 MB apart, against the FP64 five-stage apply.

Tolerance: an output sums 2 L <= 160 products in FP32, sqrt(160) roundings of
6e-8 in the mean square (7.6e-7), and the transforms add about 3e-7: 2e-6.
"""

import numpy as np
import pytest

from conftest import rel

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

CASES = [(17, (12, 10), 1), (31, (11, 9), 8), (32, (16, 12), 9), (33, (11, 7), 16),
         (48, (9, 8), 17), (49, (8, 7), 8), (64, (8, 6), 16), (65, (7, 6), 10), (79, (7, 5), 2),
         (80, (8, 5), 12), (81, (6, 5), 9),
         # few coils: the tiled kernel on the other side of the rule
         (17, (12, 10), 4), (33, (9, 8), 2)]


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


@pytest.mark.parametrize("L,n,C", CASES)
@pytest.mark.parametrize("masked", [False, True])
def test_matrix_core_block_multiply(L, n, C, masked):
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    import mr_aha_amd as mr
    from oracle import conventions as cv
    from oracle import toeplitz

    rng = np.random.default_rng(L + 100 * C)
    g = cv.make_geometry("2D", n, L, C)
    mask = None
    if masked:   # the middle third of the grid and a few others: tiles wholly outside
        keep = rng.random(g.P) < 0.05
        keep[g.P // 3: 2 * g.P // 3] = True
        keep[: g.P // 8] = False
        mask = np.flatnonzero(keep).astype(np.int64)
    cplx = lambda s: (rng.standard_normal(s) + 1j * rng.standard_normal(s)).astype(np.complex64)  # noqa: E731
    K = cplx((g.T, mask.size) if masked else (g.T,) + g.grid_shape())
    x, S = cplx((L,) + g.img_shape()), cplx((C,) + g.img_shape())
    for tri in ("lower", "upper"):
        print(f"[bdm] L={L} n={n} C={C} masked={masked} {tri}", flush=True)
        cfg = mr.make_config("2D", n, L, n_coils=C, triangulation=tri, is_masked=masked,
                             num_masked=int(mask.size) if masked else 0)
        ref = toeplitz.apply(g, x, S, K.astype(np.complex128), upper=(tri == "upper"), mask=mask)
        y = mr.aha_toeplitz(cfg, dev(x), dev(S), dev(K), dev(mask) if masked else None)
        e = rel(y.cpu().numpy(), ref)
        print(f"[bdm]   vs FP64 {e:.2e}", flush=True)
        assert e < 2e-6


@pytest.mark.parametrize("L,C", [(50, 9), (72, 3)])
def test_kernel_rows_two_megabytes_apart(L, C):
    """A 512x512 grid: workgroups of 16 locations."""
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    import mr_aha_amd as mr

    n, M = 256, 512
    rng = np.random.default_rng(L)
    cfg = mr.make_config("2D", (n, n), L, n_coils=C)
    T = L * (L + 1) // 2
    g = torch.Generator(device="cuda").manual_seed(L)
    K = torch.randn((T, M, M, 2), generator=g, device="cuda")
    K = torch.view_as_complex(K)
    cplx = lambda s: (rng.standard_normal(s) + 1j * rng.standard_normal(s)).astype(np.complex64)  # noqa: E731
    x, S = dev(cplx((L, n, n))), dev(cplx((C, n, n)))
    y = mr.aha_toeplitz(cfg, x, S, K)
    ref = torch.zeros((L, n, n), dtype=torch.complex128, device="cuda")
    for c in range(C):
        v = torch.zeros((L, M, M), dtype=torch.complex128, device="cuda")
        v[:, M // 4:3 * M // 4, M // 4:3 * M // 4] = S[c] * x
        v = torch.fft.fftshift(torch.fft.fft2(torch.fft.ifftshift(v, dim=(1, 2))), dim=(1, 2))
        o, t = torch.zeros_like(v), 0
        for j in range(L):
            for i in range(j, L):
                a = K[t].to(torch.complex128)
                o[j] += a * v[i]
                if i != j:
                    o[i] += a.conj() * v[j]
                t += 1
        o = torch.fft.fftshift(torch.fft.ifft2(torch.fft.ifftshift(o, dim=(1, 2)), norm="forward"), dim=(1, 2))
        ref += S[c].conj() * o[:, M // 4:3 * M // 4, M // 4:3 * M // 4]
    e = float((y - ref).abs().square().sum().sqrt() / ref.abs().square().sum().sqrt())
    print(f"[bdm] L={L} C={C} 512x512 vs FP64 {e:.2e}", flush=True)
    assert e < 2e-6
