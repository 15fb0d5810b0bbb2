"""Run-time-length axis passes (outer and y transforms) against the FP64 apply
and the one-tile passes (MR_AHA_HIP_AXRT=0), at the edges of their forms: one
element to 512, radices 11 and 13, planes that are not whole lines or narrower
than a tile, the last tile partly outside, pencils that wrap into the next
plane, coils that do not divide the coils of a tile, several coil groups.

Tolerance 1e-5 against the FP64 apply, as for every other form; 1e-6 between
the two forms, which take the same sums in another order.
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


SHAPES = [
    # 2D: y length 1 .. 512 (outer passes only)
    ("2D", (16, 1), (16, 1), 2, 3), ("2D", (9, 11), (18, 22), 3, 5), ("2D", (225, 26), (450, 52), 5, 7),
    ("2D", (33, 64), (48, 128), 2, 4), ("2D", (16, 130), (32, 260), 4, 3), ("2D", (5, 192), (10, 384), 2, 13),
    ("2D", (20, 198), (40, 396), 1, 2), ("2D", (6, 250), (12, 500), 3, 1), ("2D", (7, 256), (14, 512), 2, 9),
    ("2D", (300, 13), (600, 26), 2, 2), ("2D", (8, 300), (16, 600), 2, 2),
    # stacks: kz unpadded, y of every form
    ("stack", (18, 17, 40), (36, 34, 40), 2, 3), ("stack", (15, 65, 11), (30, 130, 11), 3, 2),
    ("stack", (10, 120, 48), (20, 240, 48), 2, 5), ("stack", (7, 150, 5), (14, 300, 5), 2, 2),
    ("stack", (12, 216, 3), (24, 432, 3), 1, 3), ("stack", (21, 8, 104), (42, 16, 104), 2, 2),
    # 3D: outer axis padded; whole lines and not, many tiles (n <= 384 form)
    ("3D", (16, 32, 72), (32, 64, 144), 2, 3), ("3D", (13, 9, 144), (26, 18, 288), 2, 2),
    ("3D", (128, 130, 140), (128, 130, 286), 1, 1),
]


@pytest.mark.parametrize("tt,n,M,L,C", SHAPES)
def test_axis_passes(mr, monkeypatch, tt, n, M, L, C):
    from oracle import conventions as cv
    from oracle import toeplitz
    print(f"[axis rt] {tt} n={n} M={M} L={L} C={C}", flush=True)
    rng = np.random.default_rng(sum(M) + L + C)
    g = cv.make_geometry(tt, n, L, C, M)
    cg = lambda s: (rng.standard_normal(s, dtype=np.float32)  # noqa: E731
                    + 1j * rng.standard_normal(s, dtype=np.float32)).astype(np.complex64)
    K, x, S = cg((g.T,) + g.grid_shape()), cg((L,) + g.img_shape()), cg((C,) + g.img_shape())
    cfg = mr.make_config(tt, n, L, phi2_dim=M, n_coils=C)
    ref = toeplitz.apply(g, x, S, K.astype(np.complex128))
    dx, dS, dK = dev(x), dev(S), dev(K)
    outs = {}
    for rt, group in (("1", None), ("1", "2"), ("0", None)):
        monkeypatch.setenv("MR_AHA_HIP_AXRT", rt)
        if group:
            monkeypatch.setenv("MR_AHA_HIP_COIL_GROUP", group)
        else:
            monkeypatch.delenv("MR_AHA_HIP_COIL_GROUP", raising=False)
        y = mr.aha_toeplitz(cfg, dx, dS, dK).cpu().numpy()
        assert rel(y, ref) < 1e-5, (rt, group, rel(y, ref))
        outs[(rt, group)] = y
    assert rel(outs[("1", None)], outs[("0", None)]) < 1e-6
    assert rel(outs[("1", "2")], outs[("1", None)]) < 1e-6
