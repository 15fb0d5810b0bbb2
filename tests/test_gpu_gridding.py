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


# mode counts that start with every radix (14 = 2 7, 9 = 3 3, 12 = 6 2, ...), a
# single mode, pencils of several workgroups and a partial last one, and
# counts without an unrolled butterfly (22, 13: the separate passes)
AXES = [("2D", (8, 7), (16, 14)), ("2D", (5, 6), (9, 12)), ("2D", (9, 9), (25, 35)),
        ("2D", (1, 20), (1, 40)), ("2D", (130, 4), (260, 8)), ("2D", (11, 6), (22, 13)),
        ("2D", (4, 96), (8, 192)), ("stack", (18, 12, 3), (36, 24, 3)),
        ("3D", (5, 4, 7), (10, 8, 14)), ("3D", (6, 3, 9), (12, 7, 18)), ("3D", (4, 5, 3), (8, 11, 6))]


@pytest.mark.parametrize("tt,n,M", AXES)
@pytest.mark.parametrize("chunk", [0, 2])
def test_kernel_build_axes(mr, tt, n, M, chunk, monkeypatch):
    from oracle import conventions as cv
    from oracle import toeplitz
    print(f"[gridding] axes {tt} {n} grid {M} chunk={chunk}", flush=True)
    if chunk:
        monkeypatch.setenv("MR_AHA_TOEP_MAX_CHUNK", str(chunk))
        monkeypatch.setenv("MR_AHA_HIP_MAX_BLOCKS", "7")
    L = 2
    _, traj, phi2 = _problem(tt, n, L, 20, 16, 3)
    g = cv.make_geometry(tt, n, L, 1, M)
    cfg = mr.make_config(tt, n, L, phi2_dim=M)
    K = mr.calc_toep(cfg, dev(phi2), dev(traj))
    assert rel(K.cpu().numpy(), toeplitz.calc_kernel(g, phi2, traj)) < 1e-5
    mask = torch.arange(0, int(np.prod(M)), 3, device="cuda")
    cfgm = mr.make_config(tt, n, L, phi2_dim=M, is_masked=True, num_masked=mask.numel())
    Km = mr.calc_toep(cfgm, dev(phi2), dev(traj), mask)
    assert torch.equal(torch.view_as_real(Km), torch.view_as_real(K.reshape(K.shape[0], -1)[:, mask]))


def test_kept_scratch(mr):
    """Builds of several sizes from several threads, each on its own stream,
    equal the same builds one after another (a scratch block has one owner at a
    time), and the memory kept between builds stays within the bound."""
    from concurrent.futures import ThreadPoolExecutor
    shapes = [("2D", (40, 36), 3), ("2D", (96, 80), 4), ("stack", (24, 20, 6), 3), ("3D", (16, 18, 14), 3)]
    probs = [_problem(tt, n, L, 120, 40, 30 + i) for i, (tt, n, L) in enumerate(shapes)]
    ins = [(dev(p[2]), dev(p[1])) for p in probs]
    torch.cuda.synchronize()

    def build(i, stream=None):
        tt, n, L = shapes[i]
        with torch.cuda.stream(stream):
            return mr.calc_toep(mr.make_config(tt, n, L, stream=stream), *ins[i])

    alone = [build(i) for i in range(4)]
    free0 = torch.cuda.mem_get_info()[0]
    streams = [torch.cuda.Stream() for _ in range(4)]
    with ThreadPoolExecutor(4) as ex:
        for _ in range(5):
            got = list(ex.map(build, range(4), streams))
            for a, b in zip(alone, got):
                assert torch.equal(torch.view_as_real(a), torch.view_as_real(b))
    torch.cuda.synchronize()
    del got
    assert free0 - torch.cuda.mem_get_info()[0] <= (4 << 30) + (64 << 20)


@pytest.mark.parametrize("tt,n,L,C", [("2D", (33, 27), 3, 5), ("2D", (17, 40), 1, 7),
                                      ("stack", (19, 24, 5), 2, 3), ("3D", (14, 11, 9), 2, 3)])
def test_nufft_coil_batches(mr, monkeypatch, tt, n, L, C):
    """Coils through the comparator one at a time, a few at a time (a last batch
    that is smaller) and all at once: the same sums in the same order, against
    the exact NUDFT at the gridding's accuracy (1e-5) and each other (1e-6)."""
    from oracle import nudft
    print(f"[gridding] nufft coil batches {tt} {n} L={L} C={C}", flush=True)
    g, traj, phi2 = _problem(tt, n, L, 23, 2 * max(n[:2]), L + C)
    rng = np.random.default_rng(L)
    cplx = lambda s: (rng.standard_normal(s) + 1j * rng.standard_normal(s)).astype(np.complex64)  # noqa: E731
    x, S = cplx((L,) + g.img_shape()), cplx((C,) + g.img_shape())
    ref = nudft.aha_nudft(g, x, S, phi2, traj)
    cfg = mr.make_config(tt, n, L, n_coils=C)
    outs = []
    for mb in ("0", "1", "1024"):
        monkeypatch.setenv("MR_AHA_HIP_NU_MB", mb)
        with mr.create_op(cfg, dev(S), dev(phi2), dev(traj), method="nufft") as op:
            for _ in range(2):   # the second pass finds the first one's buffers
                outs.append(op(dev(x)).cpu().numpy())
    assert rel(outs[0], ref) < 1e-5
    for y in outs[1:]:
        assert rel(y, outs[0]) < 1e-6
