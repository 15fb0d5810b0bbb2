"""Device memory that the library keeps or takes beside its arrays: the scratch
of the kernel builds stays idle between them and goes back on request."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
MB = 1 << 20


@pytest.fixture(scope="module")
def mr():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    import mr_aha_amd
    return mr_aha_amd


def _radial(tt, n, L, spokes, nkx, seed):
    """Gram blocks and a radial trajectory on the device."""
    rng = np.random.default_rng(seed)
    nd = 3 if tt == "3D" else 2
    d = rng.standard_normal((nd, spokes))
    d /= np.sqrt((d ** 2).sum(0))
    r = np.pi * (2.0 * np.arange(nkx) / nkx - 1.0)
    planes = (n[2],) if tt == "stack" else ()
    a = rng.standard_normal((L,) + planes + (spokes,)) + 1j * rng.standard_normal((L,) + planes + (spokes,))
    up = lambda v: torch.from_numpy(np.ascontiguousarray(v)).cuda()  # noqa: E731
    return (up((a[None] * np.conj(a[:, None])).astype(np.complex64)),
            up((r[None, :, None] * d[:, None, :]).astype(np.float32)))


def _free():
    torch.cuda.synchronize()
    return torch.cuda.mem_get_info()[0]


def test_idle_scratch_goes_back(mr):
    """Builds of two sizes leave at most 4 GiB idle; releasing returns it to the
    device, and the next builds equal the first.

    The device counts free memory in pages: blocks of whole megabytes have theirs
    to themselves, smaller ones share theirs with other allocations and may not
    show. All of a build's 15 blocks but the fine grids and the weights can be
    that small, so two builds have fewer than 26 MB of those."""
    mr.release_scratch()
    assert mr.idle_scratch() == 0
    cases = [("2D", (160, 144), 6), ("stack", (64, 48, 12), 4)]
    ins = [_radial(tt, n, L, 120, 200, 7 + i) for i, (tt, n, L) in enumerate(cases)]

    def build():
        return [mr.calc_toep(mr.make_config(tt, n, L), *ins[i]) for i, (tt, n, L) in enumerate(cases)]

    first = build()
    torch.cuda.empty_cache()
    idle, free = mr.idle_scratch(), _free()
    assert 0 < idle <= 4 << 30
    assert mr.release_scratch() == idle
    assert mr.idle_scratch() == 0 and mr.release_scratch() == 0
    assert _free() - free > idle - 26 * MB > 26 * MB
    for a, b in zip(first, build()):
        assert torch.equal(torch.view_as_real(a), torch.view_as_real(b))
    assert mr.idle_scratch() == idle   # the same requests, so the same blocks


def test_nufft_batches_within_the_budget(mr):
    """The comparator's coils per launch follow mem_fraction: with a budget of a
    few MB it takes one coil at a time (192x176, L=4: 15 MB a coil), in the
    default one several, and both give the same result (the coils are summed in
    the same order; 1e-6 for the interpolation's sums)."""
    n, L, C = (192, 176), 4, 12
    phi2, traj = _radial("2D", n, L, 40, 256, 3)
    g = torch.Generator(device="cuda").manual_seed(9)
    S = torch.randn((C,) + n[::-1], dtype=torch.complex64, device="cuda", generator=g)
    x = torch.randn((L,) + n[::-1], dtype=torch.complex64, device="cuda", generator=g)
    mr.release_scratch()
    torch.cuda.empty_cache()

    def create(fraction):
        mr.release_scratch()
        before = _free()
        op = mr.create_op(mr.make_config("2D", n, L, n_coils=C, mem_fraction=fraction), S, phi2, traj,
                          method="nufft")
        mr.release_scratch()
        return op, before - _free()

    total = torch.cuda.mem_get_info()[1]
    wide, wide_bytes = create(0.5)
    with wide:
        ref = wide(x)
        torch.cuda.synchronize()
    narrow, narrow_bytes = create(8e6 / total)
    with narrow:
        y = narrow(x)
        assert float(torch.linalg.vector_norm(y - ref) / torch.linalg.vector_norm(ref)) < 1e-6
    print(f"[nufft] {wide_bytes >> 20} MB in batches, {narrow_bytes >> 20} MB one at a time", flush=True)
    assert wide_bytes > 6 * narrow_bytes
