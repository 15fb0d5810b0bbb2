"""The double-buffered outer passes of a stack at every compiled number of
partitions (16 .. 64 in steps of 8): fewer tiles than workgroups and more (the
persistent loop), one rank block and two, odd coil counts, one coil group and
several, against the run-time-length passes and the FP64 apply.

Tolerances: the passes differ from each other by rounding only (1e-6, relative
2-norm); an apply's FP32 sums and transforms stay below 1e-5 of FP64.
"""

import numpy as np
import pytest

from conftest import rel

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

CASES = [(nz, n, L, C, group) for nz in (16, 24, 32, 40, 48, 56, 64)
         for n, L, C, group in (((16, 10), 8, 3, "0"), ((32, 12), 16, 4, "3"))]
# more tiles than two workgroups per CU
CASES += [(16, (128, 136), 8, 2, "0"), (24, (96, 112), 8, 1, "0"), (40, (96, 112), 8, 1, "0")]


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


@pytest.mark.parametrize("nz,n,L,C,group", CASES)
def test_outer_passes(monkeypatch, nz, n, L, C, group):
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    import mr_aha_amd as mr
    from oracle import conventions as cv
    from oracle import toeplitz

    print(f"[zdma] {n}x{nz} L={L} C={C} coil group {group}", flush=True)
    if group != "0":
        monkeypatch.setenv("MR_AHA_HIP_COIL_GROUP", group)
    rng = np.random.default_rng(nz + L)
    g = cv.make_geometry("stack", n + (nz,), L, C)
    cplx = lambda s: (rng.standard_normal(s, dtype=np.float32)  # noqa: E731
                      + 1j * rng.standard_normal(s, dtype=np.float32)).astype(np.complex64)
    K, x, S = cplx((g.T,) + g.grid_shape()), cplx((L,) + g.img_shape()), cplx((C,) + g.img_shape())
    cfg = mr.make_config("stack", n + (nz,), L, n_coils=C)
    dx, dS, dK = dev(x), dev(S), dev(K)
    outs = {}
    for zdma in ("1", "0"):
        monkeypatch.setenv("MR_AHA_HIP_ZDMA", zdma)
        outs[zdma] = mr.aha_toeplitz(cfg, dx, dS, dK).cpu().numpy()
    assert rel(outs["1"], outs["0"]) < 1e-6
    if max(n) <= 32:
        assert rel(outs["1"], toeplitz.apply(g, x, S, K.astype(np.complex128))) < 1e-5
