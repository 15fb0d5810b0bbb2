"""Coils per workgroup of the run-time-length fused x pass at the edges of its
rule: two workgroups per CU up to 80 KB (10240 values), a coil pair in one
workgroup up to 128 KB, one coil beyond; ranks times x lengths around them."""

import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("mx,L,group", [(320, 15, 2),    # 4800: two pairs of coils per CU
                                        (640, 10, 2),    # 6400: a pair, 100 KB
                                        (512, 15, 2),    # 7680: 120 KB
                                        (630, 13, 2),    # 8190
                                        (600, 14, 1),    # 8400: a pair would take 131 KB
                                        (600, 16, 1), (640, 15, 1), (800, 16, 1), (1000, 16, 1)])
def test_group(mx, L, group, monkeypatch):
    import mr_aha_amd as mr
    print(f"[group] Mx={mx} L={L}", flush=True)
    C = 4
    g = torch.Generator(device="cuda").manual_seed(mx + L)
    cfg = mr.make_config("2D", (mx // 2, 6), L, n_coils=C)
    rnd = lambda s: torch.randn(s, dtype=torch.complex64, device="cuda", generator=g)  # noqa: E731
    K, S, x = rnd(mr.phi2_toep_shape(cfg)), rnd((C, 6, mx // 2)), rnd((L, 6, mx // 2))
    with mr.create_op(cfg, S, None, None, _phi2_toep=K) as op:
        assert op.xbd_group == group
        y = op(x)
    monkeypatch.setenv("MR_AHA_HIP_XBD", "0")
    with mr.create_op(cfg, S, None, None, _phi2_toep=K) as op:
        assert op.xbd_group == 0
        ref = op(x)
    assert float(torch.linalg.vector_norm(y - ref) / torch.linalg.vector_norm(ref)) < 1e-6
