"""Lists behind the scratch blocks that the library keeps between calls
(mr_scratch.hpp), on the CPU: the header knows the device through three calls
only, here a host allocator that counts live blocks and records every block
given back (and, after a reset, that a dead one was touched)."""

import ctypes
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parents[1] / "mr_aha_amd" / "csrc"
MB = 1 << 20

HARNESS = r"""
#include "mr_scratch.hpp"
#include <set>
namespace {
int cur = 0;
unsigned long long next = 0x1000;
std::set<void *> live;
std::set<void *> given_back;
long long bad = 0;          // releases of memory that does not exist
size_t room = ~(size_t)0;   // bytes the device has left
std::map<void *, size_t> size_of;
struct fake {
    static int device() { return cur; }
    static void *alloc(size_t bytes)
    {
        if (bytes > room) return nullptr;
        room -= bytes;
        void *p = (void *)next;
        next += 0x1000;
        live.insert(p);
        size_of[p] = bytes;
        return p;
    }
    static void release(int, void *p)
    {
        if (!live.erase(p)) { ++bad; return; }
        room += size_of[p];
        given_back.insert(p);
    }
};
mr_scratch<fake> *ws = nullptr;
}
extern "C" {
void t_open(size_t max_idle, unsigned long long age)
{
    delete ws;
    ws = new mr_scratch<fake>(max_idle, age);
    cur = 0; next = 0x1000; bad = 0; room = ~(size_t)0;
    live.clear(); given_back.clear(); size_of.clear();
}
void *t_get(size_t b) { return ws->get(b); }
void t_put(void *p) { ws->put(p); }
size_t t_idle(int dev) { return ws->idle_bytes(dev); }
size_t t_release(int dev) { return ws->release_idle(dev); }
unsigned t_epoch(int dev) { return ws->epoch(dev); }
int t_forget(int dev, unsigned since) { return ws->forget(dev, since) ? 1 : 0; }
void t_device(int dev) { cur = dev; }
void t_room(size_t b) { room = b; }
// the device loses everything; its addresses are handed out again
void t_reset(void) { live.clear(); size_of.clear(); next = 0x1000; }
int t_live(void *p) { return live.count(p) ? 1 : 0; }
long long t_bad(void) { return bad; }
long long t_nlive(void) { return (long long)live.size(); }
}
"""


@pytest.fixture(scope="module")
def built(tmp_path_factory):
    d = tmp_path_factory.mktemp("scratch")
    src = d / "t.cpp"
    src.write_text("#include <map>\n" + HARNESS)
    so = d / "t.so"
    r = subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-Werror", "-shared", "-fPIC",
                        f"-I{CSRC}", str(src), "-o", str(so)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    t = ctypes.CDLL(str(so))
    for name, res, args in [("t_open", None, [ctypes.c_size_t, ctypes.c_ulonglong]),
                            ("t_get", ctypes.c_void_p, [ctypes.c_size_t]),
                            ("t_put", None, [ctypes.c_void_p]), ("t_idle", ctypes.c_size_t, [ctypes.c_int]),
                            ("t_release", ctypes.c_size_t, [ctypes.c_int]),
                            ("t_epoch", ctypes.c_uint, [ctypes.c_int]),
                            ("t_forget", ctypes.c_int, [ctypes.c_int, ctypes.c_uint]),
                            ("t_device", None, [ctypes.c_int]), ("t_room", None, [ctypes.c_size_t]),
                            ("t_reset", None, []), ("t_live", ctypes.c_int, [ctypes.c_void_p]),
                            ("t_bad", ctypes.c_longlong, []), ("t_nlive", ctypes.c_longlong, [])]:
        f = getattr(t, name)
        f.restype, f.argtypes = res, args
    return t


@pytest.fixture
def ws(built):
    built.t_open(64 * MB, 64)
    return built


def test_one_owner_and_reuse(ws):
    a = ws.t_get(8 * MB)
    b = ws.t_get(8 * MB)
    assert a != b
    ws.t_put(a)
    assert ws.t_get(8 * MB) == a      # kept
    c = ws.t_get(8 * MB)
    assert c not in (a, b)            # both in use
    for p in (a, b, c):
        ws.t_put(p)
    assert ws.t_idle(0) == 24 * MB and ws.t_nlive() == 3


def test_nothing_from_before_a_reset_is_used_again(ws):
    """An idle block, a block in use and one of another device; the operator
    that held the block in use is abandoned."""
    since = ws.t_epoch(0)
    idle, held = ws.t_get(8 * MB), ws.t_get(8 * MB)
    ws.t_put(idle)
    ws.t_device(1)
    other = ws.t_get(8 * MB)
    ws.t_put(other)
    ws.t_device(0)
    ws.t_reset()
    assert ws.t_forget(0, since) == 1
    assert ws.t_idle(0) == 0 and ws.t_idle(1) == 8 * MB
    fresh = ws.t_get(8 * MB)
    assert ws.t_live(fresh) == 1      # allocated after the reset, not kept from before it
    assert fresh == idle              # (at an address that was handed out before)
    # operators from before the reset that are abandoned later change nothing
    assert ws.t_forget(0, since) == 0
    ws.t_put(fresh)
    assert ws.t_get(8 * MB) == fresh
    ws.t_put(held if held != fresh else None)   # a stale owner: not on the lists
    ws.t_put(fresh)
    assert ws.t_idle(0) == 8 * MB
    assert ws.t_release(0) == 8 * MB
    assert ws.t_bad() == 0            # no dead block was ever given back


def test_a_second_reset(ws):
    since = ws.t_epoch(0)
    ws.t_put(ws.t_get(4 * MB))
    ws.t_reset()
    assert ws.t_forget(0, since) == 1
    again = ws.t_epoch(0)
    assert again != since
    ws.t_put(ws.t_get(4 * MB))
    ws.t_reset()
    assert ws.t_forget(0, again) == 1
    assert ws.t_live(ws.t_get(4 * MB)) == 1 and ws.t_bad() == 0


def test_a_block_serves_requests_of_its_size(ws):
    """Up to an eighth smaller, never less: what a caller is given stays near
    what it asked for."""
    a = ws.t_get(9 * MB)
    ws.t_put(a)
    assert ws.t_get(8 * MB) == a
    ws.t_put(a)
    small = ws.t_get(6 * MB)
    assert small != a
    assert ws.t_get(10 * MB) not in (a, small)
    assert ws.t_idle(0) == 9 * MB


def test_idle_bytes_stay_within_the_limit(ws):
    held = [ws.t_get(24 * MB) for _ in range(4)]
    for p in held:
        ws.t_put(p)
        assert ws.t_idle(0) <= 64 * MB
    assert ws.t_idle(0) == 48 * MB and ws.t_nlive() == 2
    assert [ws.t_live(p) for p in held] == [0, 0, 1, 1]   # the longest idle went first
    big = ws.t_get(65 * MB)
    ws.t_put(big)
    assert ws.t_idle(0) <= 64 * MB and ws.t_live(big) == 0


def test_unused_blocks_go_back(built):
    built.t_open(64 * MB, 8)
    a = built.t_get(8 * MB)
    built.t_put(a)
    for _ in range(8):
        built.t_put(built.t_get(2 * MB))
        assert built.t_live(a) == 1
    built.t_put(built.t_get(2 * MB))
    assert built.t_live(a) == 0 and built.t_idle(0) == 2 * MB


def test_a_full_device_takes_idle_blocks_back(ws):
    ws.t_put(ws.t_get(8 * MB))
    ws.t_device(1)
    other = ws.t_get(4 * MB)
    ws.t_put(other)
    ws.t_device(0)
    ws.t_room(1 * MB)
    p = ws.t_get(9 * MB)          # more than the idle block, less than both
    assert p and ws.t_idle(0) == 0
    assert ws.t_idle(1) == 4 * MB and ws.t_live(other) == 1
    assert ws.t_get(1 * MB) is None
    assert ws.t_bad() == 0


def test_an_array_that_does_not_fit_takes_idle_scratch(monkeypatch):
    """Arrays of the Python interface are torch's; when torch has no memory left
    the idle scratch is given back and the allocation tried once more."""
    torch = pytest.importorskip("torch")
    from mr_aha_amd import api
    real, calls = torch.empty, []

    def empty(shape, **kw):
        calls.append(tuple(shape))
        if len(calls) == 1:
            raise torch.OutOfMemoryError("out of memory")
        return real(shape, **kw)

    monkeypatch.setattr(torch, "empty", empty)
    monkeypatch.setattr(api, "release_scratch", lambda device=-1: 8 * MB)
    assert api._empty((2, 3), "cpu").shape == (2, 3) and len(calls) == 2
    calls.clear()
    monkeypatch.setattr(api, "release_scratch", lambda device=-1: 0)
    with pytest.raises(torch.OutOfMemoryError):
        api._empty((2, 3), "cpu")
    assert len(calls) == 1


def test_admission_counts_idle_scratch(monkeypatch):
    """A request is admitted only when it, those running and the idle scratch
    fit the budget together; the scratch makes room, the running ones do not."""
    from mr_aha_amd import api, serve
    idle = [6 * MB]
    given = []

    def release(device=-1):
        given.append(idle[0])
        idle[0] = 0
        return given[-1]

    monkeypatch.setattr(api, "idle_scratch", lambda device=-1: idle[0])
    monkeypatch.setattr(api, "release_scratch", release)
    srv = serve.Server(budget_bytes=16 * MB, slots=2)
    assert srv._fits(10 * MB) and not given
    assert srv._fits(11 * MB) and given == [6 * MB]
    idle[0], srv._used, srv._running = 3 * MB, 8 * MB, 1
    assert not srv._fits(9 * MB) and given == [6 * MB]
    assert srv._fits(8 * MB) and given == [6 * MB, 3 * MB]
    srv._running = 2
    assert not srv._fits(1)


def test_build_footprint_bounds_the_scratch():
    """Every block that a build takes, by its formula: chunk, strengths, sample
    tables (an eighth more each) and a megabyte for each of the dozen blocks."""
    from types import SimpleNamespace
    from mr_aha_amd import serve
    for tt, n, L, ntr, nkx in [("2D", (320, 320), 16, 512, 640), ("stack", (256, 256, 48), 16, 400, 512),
                               ("3D", (96, 96, 96), 4, 4000, 192), ("2D", (16, 16), 1, 1, 8)]:
        req = SimpleNamespace(traj_type=tt, n_dim=n, L=L, precision="fp32", n_coils=4,
                              traj=SimpleNamespace(shape=(3 if tt == "3D" else 2, nkx, ntr)))
        m, d = ntr * nkx, 3 if tt == "3D" else 2
        planes = n[2] if tt == "stack" else 1
        blocks = [serve.BUILD_BYTES, L * (L + 1) // 2 * planes * ntr * 16, m * d * 16 * 8, 3 * m * 4]
        blocks += [m * 4] * 5
        assert serve.build_bytes(req) >= sum(b * 9 // 8 + MB for b in blocks)
        assert serve.footprint_bytes(req) > serve.build_bytes(req)
