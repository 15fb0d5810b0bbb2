"""Run-time-length fused x pass against the FP64 apply, at the edges of its
forms: odd and even x lengths, every first radix, a last block of locations
shorter than a wavefront, images that fill the centred half of the pencil and
others, rows that do and do not allow 16-byte loads, an odd last coil, kernels
on an odd 8-byte address, workgroups of 512 and 1024, ranks 1 to 16.

Tolerance 1e-5 (relative 2-norm), as for every other form of the apply.
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


# (n, M, L, C): x lengths 480 = 8 10 6, 90 = 10 3 3, 98 = 2 7 7, 45 = 3 3 5,
# 64 = 8 8, 24 = 8 3, 12 = 6 2, 16 = 8 2, 400 = 8 10 5, 768, 900, 1, 2, 7
SHAPES = [((240, 4), (480, 8), 6, 3), ((45, 6), (90, 12), 5, 2), ((49, 4), (98, 8), 3, 5),
          ((22, 5), (45, 10), 7, 2), ((32, 6), (64, 12), 1, 3), ((12, 4), (24, 8), 2, 1),
          ((6, 3), (12, 6), 9, 4), ((8, 3), (16, 6), 11, 2), ((200, 4), (400, 8), 12, 3),
          ((180, 4), (400, 8), 13, 1), ((384, 2), (768, 4), 16, 2), ((384, 2), (768, 4), 10, 3),
          ((450, 2), (900, 4), 14, 1), ((100, 3), (200, 6), 15, 3), ((1, 4), (1, 8), 4, 2),
          ((1, 4), (2, 8), 3, 2), ((4, 3), (7, 6), 2, 2)]


@pytest.mark.parametrize("n,M,L,C", SHAPES)
@pytest.mark.parametrize("masked", [False, True])
def test_fused_any_length(mr, n, M, L, C, masked):
    from oracle import conventions as cv
    from oracle import toeplitz
    print(f"[fused rt] n={n} M={M} L={L} C={C} masked={masked}", flush=True)
    rng = np.random.default_rng(sum(M) + 31 * L + C)
    g = cv.make_geometry("2D", n, L, C, M)
    mask = np.flatnonzero(rng.random(g.P) < 0.6).astype(np.int64) if masked else None
    kshape = (g.T, mask.size) if masked else (g.T,) + g.grid_shape()
    cg = lambda s: (rng.standard_normal(s) + 1j * rng.standard_normal(s)).astype(np.complex64)  # noqa: E731
    K, x, S = cg(kshape), cg((L,) + g.img_shape()), cg((C,) + g.img_shape())
    for tri, shift in (("lower", 0), ("upper", 0), ("lower", 1)):
        buf = torch.empty(K.size + 1, dtype=torch.complex64, device="cuda")
        dK = buf[shift:shift + K.size].view(kshape)
        dK.copy_(dev(K))
        cfg = mr.make_config("2D", n, L, phi2_dim=M, n_coils=C, triangulation=tri, is_masked=masked,
                             num_masked=mask.size if masked else 0)
        ref = toeplitz.apply(g, x, S, K.astype(np.complex128), upper=(tri == "upper"), mask=mask)
        with mr.create_op(cfg, dev(S), None, None, mask=dev(mask) if masked else None,
                          _phi2_toep=dK) as op:
            assert op.xbd_group > 0
            y = op(dev(x)).cpu().numpy()
        assert rel(y, ref) < 1e-5, (tri, shift, rel(y, ref))
