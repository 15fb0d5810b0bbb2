"""Tile widths of the axis passes and which kernels they belong to: the
autotuner sweeps the passes on the one-tile kernels, and reports the tile of a
pass on a persistent kernel, which no width changes; the one-tile kernels split
grids of more than 2^32 work-items (with the persistent ones off, which do not
launch such grids)."""

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


def _op(mr, tt, n, L, C, **kw):
    nn = list(n) + [1] * (3 - len(n))
    g = torch.Generator(device="cuda").manual_seed(3)
    cfg = mr.make_config(tt, n, L, n_coils=C, **kw)
    rnd = lambda s: torch.randn(s, dtype=torch.complex64, device="cuda", generator=g)  # noqa: E731
    img = tuple(reversed(nn[: len(n)]))
    K, S, x = rnd(mr.phi2_toep_shape(cfg)), rnd((C,) + img), rnd((L,) + img)
    return mr.create_op(cfg, S, None, None, _phi2_toep=K), x


# outer, y, inverse y and inverse outer pass: pencils of a persistent kernel's
# tile (16, 8 in the narrow outer form, 16 positions x 8 ranks in the
# double-buffered outer passes), or None where the one-tile kernels run
CASES = [("stack", (48, 40, 10), 4, 3, (16, 16, 16, 16)),
         ("2D", (60, 44), 8, 3, (16, 0, 0, 16)),
         ("2D", (24, 198), 4, 2, (8, 0, 0, 8)),          # 396: narrow tiles
         ("stack", (32, 24, 16), 8, 2, (128, 16, 16, 128)),
         ("stack", (24, 160, 10), 4, 2, (16, None, None, 16)),   # 320 along y
         ("2D", (64, 128), 4, 2, (None, 0, 0, 16))]      # 256: whole-line one-tile forward pass


@pytest.mark.parametrize("tt,n,L,C,want", CASES)
def test_tuned_tiles(mr, tt, n, L, C, want):
    print(f"[tiles] {tt} {n} L={L} C={C}", flush=True)
    op, x = _op(mr, tt, n, L, C)
    with op:
        y0 = op(x)
        t = op.tiles
        assert (t["fo"], t["fy"], t["iy"], t["io"]) == (0, 0, 0, 0)
        for _ in range(2):
            t = op.autotune(x, reps=1)
            for got, w in zip((t["fo"], t["fy"], t["iy"], t["io"]), want):
                assert got == w if w is not None else got in (1, 2, 4, 8, 16, 32, 64), (t, want)
        y1 = op(x)
        assert float(torch.linalg.vector_norm(y1 - y0) / torch.linalg.vector_norm(y0)) < 1e-6


@pytest.mark.parametrize("tt,n,L,C", [("stack", (48, 40, 10), 4, 3), ("2D", (60, 44), 8, 3)])
def test_one_tile_kernels_in_chunks(mr, monkeypatch, tt, n, L, C):
    """Dispatches of 7 workgroups give the bits of single ones."""
    monkeypatch.setenv("MR_AHA_HIP_AXRT", "0")
    op, x = _op(mr, tt, n, L, C)
    with op:
        y0 = op(x).cpu().numpy()
        monkeypatch.setenv("MR_AHA_HIP_MAX_BLOCKS", "7")
        y1 = op(x).cpu().numpy()
    assert np.array_equal(y0, y1), rel(y1, y0)


def test_one_tile_outer_pass_beyond_32bit_grid(mr, monkeypatch):
    """160x160x8 stack, L=16, 21 coils: the one-tile outer pass at one pencil per
    workgroup has 8.6M workgroups of 512 work-items (more than 2^32) and equals
    the same pass at 64."""
    print("[tiles] stack 160x160x8 L16 C21, one pencil per workgroup", flush=True)
    monkeypatch.setenv("MR_AHA_HIP_AXRT", "0")
    n, nz, L, C = 160, 8, 16, 21
    op, x = _op(mr, "stack", (n, n, nz), L, C, mem_fraction=0.9)
    with op:
        group = op.info["group"][0]
        if n * n * L * group <= 0xFFFFFFFF // 512:
            pytest.skip(f"coil group {group}: the outer pass stays within one dispatch")
        monkeypatch.setenv("MR_AHA_HIP_FO_TX", "64")
        y64 = op(x)
        monkeypatch.setenv("MR_AHA_HIP_FO_TX", "1")
        y1 = op(x)
        torch.cuda.synchronize()
        assert torch.equal(y1, y64), float((y1 - y64).abs().max())
