"""Launch shapes of the run-time-length axis passes, on the CPU: the rules of
mr_axis_form.hpp, which the launches use, against the registers that the
compiler reports for every kernel of mr_axis_rt.hip.

The workgroups are persistent and the tiles are dealt out to them up front, so
no more of them may be launched than a CU holds at once.
"""

import ctypes
import importlib.util
import re
import subprocess
from pathlib import Path

import pytest

PKG = Path(__file__).resolve().parents[1] / "mr_aha_amd"
CSRC = PKG / "csrc"
Y, FO, IO = 0, 1, 2
NMAX = 512

HARNESS = r"""
#include "mr_axis_form.hpp"
extern "C" void t_form(int n, int outer, int few, int *out)
{
    const ax_form f = ax_pick(n, outer != 0, few != 0);
    out[0] = f.nt; out[1] = f.ke; out[2] = f.pt;
}
extern "C" int t_per_cu(int kind, int n, int outer, int few, int big)
{
    return ax_per_cu((ax_kind)kind, ax_pick(n, outer != 0, few != 0), big != 0, n);
}
"""


@pytest.fixture(scope="module")
def forms(tmp_path_factory):
    d = tmp_path_factory.mktemp("forms")
    (d / "t.cpp").write_text(HARNESS)
    so = d / "t.so"
    r = subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-Werror", "-shared", "-fPIC", f"-I{CSRC}",
                        str(d / "t.cpp"), "-o", str(so)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    return ctypes.CDLL(str(so))


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """{(kind, nt, ke, pt, big, compiled length): wavefronts per SIMD}"""
    spec = importlib.util.spec_from_file_location("_b", PKG / "build.py")
    b = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(b)
    out = tmp_path_factory.mktemp("obj") / "a.o"
    r = subprocess.run([b.HIPCC, *b.HIP_FLAGS, *b.COMMON, "--cuda-device-only", "-c",
                        str(CSRC / "mr_axis_rt.hip"), "-o", str(out),
                        "-Rpass-analysis=kernel-resource-usage"], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    found, key = {}, None
    for line in r.stderr.splitlines():
        m = re.search(r"Function Name: (\S+)", line)
        if m:
            k = re.search(r"mr_k_axis_(y|fo|io)I(.*?)EEv", m.group(1) + "EEv")
            args = [int(v) for v in re.findall(r"L[bi](\d+)E", k.group(2) + "E")]
            if k.group(1) == "y":
                key = (Y, *args[1:5], 0)
            else:
                key = (FO if k.group(1) == "fo" else IO, *args[:4], args[4] if len(args) > 4 else 0)
        m = re.search(r"Occupancy \[waves/SIMD\]: (\d+)", line)
        if m:
            found[key] = min(int(m.group(1)), found.get(key, 99))
    assert len(found) > 20
    return found


def _cases(forms):
    """(kind, n, outer, few, big, form) of every launch."""
    buf = (ctypes.c_int * 3)()
    for n in range(1, NMAX + 1):
        for kind, few in ((Y, 0), (FO, 0), (FO, 1), (IO, 0), (IO, 1)):
            for big in (0, 1):
                forms.t_form(n, int(kind != Y), few, buf)
                yield kind, n, int(kind != Y), few, big, tuple(buf)


def test_a_tile_fits_its_workgroup(forms):
    for kind, n, outer, few, big, (nt, ke, pt) in _cases(forms):
        assert n * pt <= nt * ke, (kind, n)


def test_no_more_workgroups_than_a_cu_holds(forms, kernels):
    for kind, n, outer, few, big, (nt, ke, pt) in _cases(forms):
        per = forms.t_per_cu(kind, n, outer, few, big)
        assert per >= 1
        # the kernel at a compiled length, where there is one, and the general one
        for length in (0, n):
            occ = kernels.get((kind, nt, ke, pt, big, length))
            assert occ is not None or length > 0, (kind, n, nt, ke, pt, big)
            if occ is not None:
                held = 4 * occ * 64 // nt if nt < 256 else occ // (nt // 256)
                assert per <= held, (kind, n, (nt, ke, pt), big, length, per, held)
        assert per == 1 or per * n * (pt + 1) * 8 <= 160 * 1024, (kind, n)


def test_every_kernel_is_launched_by_some_length(forms, kernels):
    used = {(kind, *form, big) for kind, _, _, _, big, form in _cases(forms)}
    for kind, nt, ke, pt, big, length in kernels:
        assert (kind, nt, ke, pt, big) in used, (kind, nt, ke, pt, big)
        assert length <= NMAX
