"""More than 65535 strength sets in one spreading launch (a small grid of many
planes at a large rank), with tiles that have several segments of samples, so
that the sum of the segments runs over all sets."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def mr():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    import mr_aha_amd
    return mr_aha_amd


def test_build_beyond_65535_sets(mr, monkeypatch):
    """4x4x32 stack, L=64: 2080 x 32 components in one chunk. The same sums in
    chunks of 4096, bit for bit (every set is summed in the same order), and the
    first ranks against a build of those alone."""
    L, nz, spokes, nkx = 64, 32, 4, 160
    print(f"[sets] stack 4x4x{nz} L={L}, {spokes} x {nkx} samples", flush=True)
    rng = np.random.default_rng(4)
    d = rng.standard_normal((2, spokes))
    d /= np.sqrt((d ** 2).sum(0))
    r = np.pi * (2.0 * np.arange(nkx) / nkx - 1.0)
    a = rng.standard_normal((L, nz, spokes)) + 1j * rng.standard_normal((L, nz, spokes))
    phi2 = torch.from_numpy((a[None] * np.conj(a[:, None])).astype(np.complex64)).cuda()
    traj = torch.from_numpy((r[None, :, None] * d[:, None, :]).astype(np.float32)).cuda()
    n = (4, 4, nz)
    K = mr.calc_toep(mr.make_config("stack", n, L, mem_fraction=0.9), phi2, traj)
    assert K.shape[0] * nz > 65535
    few = mr.calc_toep(mr.make_config("stack", n, 2), phi2[:2, :2].contiguous(), traj)
    monkeypatch.setenv("MR_AHA_TOEP_MAX_CHUNK", "4096")
    parts = mr.calc_toep(mr.make_config("stack", n, L, mem_fraction=0.9), phi2, traj)
    bits = torch.view_as_real
    assert torch.equal(bits(K), bits(parts))
    assert torch.isfinite(bits(K)).all()
    # lower triangle, columns first: (0,0), (1,0), then (1,1) after column 0
    assert torch.equal(bits(K[[0, 1, L]]), bits(few))
