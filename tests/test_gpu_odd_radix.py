"""Grid lengths with prime factors that have no unrolled butterfly: one large
prime, two of them (the second stage has twiddles), a prime alone, squares, few
pencils and many, every axis, against the FP64 five-stage apply.

Tolerance: a stage sums up to (R - 1) / 2 <= 130 products per output in FP32,
sqrt(130) roundings of 6e-8 (7e-7) per axis in the worst of these, twice along
each axis: 3e-6.
"""

import numpy as np
import pytest

from conftest import rel

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

CASES = [("2D", (143, 8), 3, 2), ("2D", (6, 143), 3, 2), ("2D", (131, 20), 2, 3), ("2D", (20, 131), 5, 1),
         ("2D", (58, 57), 7, 2), ("2D", (17, 17), 17, 2), ("2D", (12, 261), 1, 1), ("2D", (187, 121), 2, 1),
         ("stack", (16, 46, 31), 4, 2), ("stack", (19, 16, 37), 8, 3), ("3D", (29, 19, 23), 3, 2),
         ("3D", (16, 17, 34), 2, 1)]


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


@pytest.mark.parametrize("tt,n,L,C", CASES)
def test_odd_radices(tt, n, L, C):
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    import mr_aha_amd as mr
    from oracle import conventions as cv
    from oracle import toeplitz

    print(f"[odd] {tt} {n} L={L} C={C}", flush=True)
    rng = np.random.default_rng(sum(n) + L)
    g = cv.make_geometry(tt, n, L, C)
    cplx = lambda s: (rng.standard_normal(s) + 1j * rng.standard_normal(s)).astype(np.complex64)  # noqa: E731
    K, x, S = cplx((g.T,) + g.grid_shape()), cplx((L,) + g.img_shape()), cplx((C,) + g.img_shape())
    cfg = mr.make_config(tt, n, L, n_coils=C)
    y = mr.aha_toeplitz(cfg, dev(x), dev(S), dev(K)).cpu().numpy()
    e = rel(y, toeplitz.apply(g, x, S, K.astype(np.complex128)))
    print(f"[odd]   vs FP64 {e:.2e}", flush=True)
    assert e < 3e-6
