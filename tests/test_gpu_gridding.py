"""Gridding of the kernel build and of the NUFFT comparator at the sizes where
the tiles go wrong, against the exact sums.

Shapes: a grid of a single tile and of two (every neighbour wraps onto it), a
tile with several segments of candidate samples (all readouts cross the
centre), no sample in most tiles, strength chunks of every width with and
without a remainder, narrow and wide kernels.

Tolerance: ten times the gridding tolerance (the kernels' own error is below
the requested one per axis) plus the rounding of the complex64 result.
"""

import numpy as np
import pytest

from conftest import rel

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def mr():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    import mr_aha_amd
    return mr_aha_amd


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _problem(tt, n, L, spokes, nkx, seed):
    from oracle import conventions as cv
    rng = np.random.default_rng(seed)
    g = cv.make_geometry(tt, n, L, 2)
    nd = 3 if tt == "3D" else 2
    d = rng.standard_normal((nd, spokes))
    d /= np.sqrt((d ** 2).sum(0))
    r = np.pi * (2.0 * np.arange(nkx) / nkx - 1.0)
    traj = (r[None, :, None] * d[:, None, :]).astype(np.float32)
    planes = (n[2],) if tt == "stack" else ()
    a = rng.standard_normal((L,) + planes + (spokes,)) + 1j * rng.standard_normal((L,) + planes + (spokes,))
    phi2 = (a[None] * np.conj(a[:, None])).astype(np.complex64)
    return g, traj, phi2


CASES = [
    # one tile / two tiles an axis
    ("2D", (2, 3), 2, 3, 5, 1e-2),
    ("2D", (4, 4), 3, 9, 16, 1e-6),
    # most tiles empty, one readout
    ("2D", (40, 31), 1, 1, 7, 1e-6),
    # several segments at the centre; strengths 4, 8, 12, 16 wide with remainders
    ("2D", (24, 20), 2, 600, 24, 1e-6),
    ("2D", (24, 20), 3, 300, 48, 1e-6),
    ("2D", (21, 16), 4, 300, 40, 1e-4),
    ("2D", (16, 18), 5, 200, 36, 1e-6),
    ("2D", (16, 18), 6, 200, 36, 1e-12),
    ("stack", (14, 16, 5), 3, 150, 32, 1e-6),
    ("3D", (8, 10, 6), 2, 400, 20, 1e-6),
    ("3D", (10, 8, 9), 4, 200, 20, 1e-3),
    ("3D", (12, 12, 12), 3, 40, 24, 1e-12),
]


@pytest.mark.parametrize("tt,n,L,spokes,nkx,eps", CASES)
def test_kernel_build_tiles(mr, tt, n, L, spokes, nkx, eps):
    from oracle import toeplitz
    print(f"[gridding] {tt} {n} L={L} {spokes}x{nkx} eps={eps}", flush=True)
    g, traj, phi2 = _problem(tt, n, L, spokes, nkx, 17 * L + spokes)
    cfg = mr.make_config(tt, n, L, n_coils=2, eps=eps)
    K = mr.calc_toep(cfg, dev(phi2), dev(traj))
    again = mr.calc_toep(cfg, dev(phi2), dev(traj))
    assert torch.equal(torch.view_as_real(K), torch.view_as_real(again))   # no atomics: bit-reproducible
    ref = toeplitz.calc_kernel(g, phi2, traj)
    assert rel(K.cpu().numpy(), ref) < 10 * eps + 2e-7


@pytest.mark.parametrize("tt,n,L,spokes,nkx", [("2D", (18, 14), 3, 300, 28), ("2D", (16, 16), 9, 40, 32),
                                               ("stack", (12, 10, 3), 2, 200, 20),
                                               ("3D", (8, 6, 10), 5, 250, 16)])
def test_nufft_tiles(mr, tt, n, L, spokes, nkx):
    from oracle import nudft
    print(f"[gridding] nufft {tt} {n} L={L} {spokes}x{nkx}", flush=True)
    g, traj, phi2 = _problem(tt, n, L, spokes, nkx, 5 + L)
    rng = np.random.default_rng(L)
    shape = g.img_shape()
    x = (rng.standard_normal((L,) + shape) + 1j * rng.standard_normal((L,) + shape)).astype(np.complex64)
    S = (rng.standard_normal((2,) + shape) + 1j * rng.standard_normal((2,) + shape)).astype(np.complex64)
    cfg = mr.make_config(tt, n, L, n_coils=2)
    with mr.create_op(cfg, dev(S), dev(phi2), dev(traj), method="nufft") as op:
        y = op(dev(x)).cpu().numpy()
    assert rel(y, nudft.aha_nudft(g, x, S, phi2, traj)) < 1e-5 + 2e-7
