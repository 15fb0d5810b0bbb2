"""Performance cases of the Toeplitz A^H A library, through its public entry points.

What a reconstruction program does with this package:

* ``apply``  ``op(x)``: one normal-operator apply with a kernel built once and
  kept in the operator, the inner loop of every iterative reconstruction. 2D,
  stack-of-stars and 3D grids, ranks from a few to several tens, unmasked and
  masked kernels, the FP32 and the 16-bit kernel storage.
* ``cg``     ``op.cg(b)``: the regularised solve, its iterations replayed as
  graphs, as the server runs it.
* ``build``  ``calc_toep`` (after ``calc_mask`` where the kernel is masked):
  once per trajectory, and the first part of every served request.
* ``nufft``  ``op(x)`` of a ``method="nufft"`` operator, the comparator that
  needs no kernel.

Inputs come from the seed alone: golden-angle radial or Fibonacci-sphere
spokes, rank-1 Gram blocks of a random rank x time basis, smooth coil maps of
unit root-sum-of-squares, a phantom of ellipses with decaying rank
coefficients. The kernels of the apply and CG cases have the density of radial
sampling (1/|k| inside the sampled disc or ball, almost nothing in the corners)
times a few Gram matrices, so every location's block is Hermitian positive
semidefinite as a built kernel's is.
"""

from __future__ import annotations

import math

import numpy as np
import torch

import mr_aha_amd as mr

GOLDEN = (math.sqrt(5.0) - 1.0) / 2.0
DEV = "cuda"
CG_REFRESH = 10
CG_LAMBDA = 0.1    # the operators' largest eigenvalue is a few units


# ---------------------------------------------------------------------------
# Cases
# ---------------------------------------------------------------------------

def _case(kind, traj, n, L, C, masked=False, fmt="fp32", tri="lower", spokes=0, nkx=0, iters=0):
    n = list(n) + [1] * (3 - len(n))
    return dict(kind=kind, traj=traj, nx=n[0], ny=n[1], nz=n[2], L=L, C=C, masked=masked, fmt=fmt,
                tri=tri, spokes=spokes, nkx=nkx, iters=iters)


def listed():
    def named(name, *a, **k):
        return dict(_case(*a, **k), name=name)

    return [
        # the smallest reconstruction: one 2D slice, launches and latency
        named("apply_2d_128_L4", "apply", "2D", (128, 128), 4, 4),
        # a non-square odd matrix and rank (cropped field of view), upper storage
        named("apply_2d_225x198_L5", "apply", "2D", (225, 198), 5, 7, tri="upper"),
        # a large rank: many-contrast 2D, the L > 16 kernels
        named("apply_2d_320_L72", "apply", "2D", (320, 320), 72, 12),
        # a stack of an everyday size, non-square, with the mask of its radial trajectory
        named("apply_stack_240x216x40_L6_masked", "apply", "stack", (240, 216, 40), 6, 10,
              masked=True),
        # a served stack with its kernel held in 16 bits
        named("apply_stack_256x48_L16_bf16", "apply", "stack", (256, 256, 48), 16, 16, fmt="bf16"),
        # the benchmark's stack of stars, the largest
        named("apply_stack_320x56_L16", "apply", "stack", (320, 320, 56), 16, 12),
        # the kooshball: all three axes padded
        named("apply_3d_160_L8", "apply", "3D", (160, 160, 160), 8, 8),
        # a served 2D solve
        named("cg_2d_192_L8", "cg", "2D", (192, 192), 8, 12, iters=30),
        # kernel builds: a served 2D slice, a served stack, a masked 3D volume
        named("build_2d_256_L8", "build", "2D", (256, 256), 8, 8, spokes=512, nkx=512),
        named("build_stack_192x32_L8", "build", "stack", (192, 192, 32), 8, 8, spokes=384,
              nkx=384),
        named("build_3d_96_L4_masked", "build", "3D", (96, 96, 96), 4, 4, masked=True, spokes=4000,
              nkx=192),
        # the comparator on the smallest slice's larger sibling
        named("nufft_2d_192_L4", "nufft", "2D", (192, 192), 4, 4, spokes=128, nkx=384),
    ]


def _smooth(m):
    for p in (2, 3, 5, 7):
        while m % p == 0:
            m //= p
    return m == 1


def _size(rng, lo, hi):
    """Log-uniform; mostly the multiples of 16 and 8 that scanners use, some
    even and some odd."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    step = rng.choice([16, 16, 8, 2, 1])
    return int(min(hi, max(lo, step * round(v / step))))


def _matrix(rng, traj, lo, hi, zlo, zhi):
    nx = _size(rng, lo, hi)
    ny = nx if rng.random() < 0.6 else int(min(hi, max(lo, round(nx * rng.uniform(0.75, 1.2)))))
    if traj == "2D":
        return nx, ny
    if traj == "stack":
        return nx, ny, rng.randint(zlo, zhi)
    return nx, ny, nx if rng.random() < 0.5 else int(min(hi, max(lo, round(nx * rng.uniform(0.6, 1.0)))))


def _rank(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the same ranges, no costlier than the largest listed."""
    kind = rng.choices(["apply", "cg", "build", "nufft"], [6, 1, 2, 1])[0]
    while True:
        tri = rng.choice(["lower", "lower", "upper"])
        if kind == "apply":
            traj = rng.choice(["2D", "stack", "stack", "3D"])
            masked, fmt = rng.random() < 0.25, "fp32"
            if not masked and traj != "3D" and rng.random() < 0.2:
                # 16-bit storage exists for these x sizes and ranks
                fmt, L = rng.choice(["bf16", "fp16"]), rng.choice([4, 8, 16])
                nx = rng.choice([128, 160, 192, 256, 320])
                n = (nx, nx) if traj == "2D" else (nx, nx, rng.randint(12, 56))
            else:
                n = _matrix(rng, traj, *((96, 384, 1, 1) if traj == "2D" else
                                         (96, 320, 12, 64) if traj == "stack" else (48, 160, 1, 1)))
                L = _rank(rng, 2, 72 if traj == "2D" else 16 if traj == "stack" else 8)
            c = _case(kind, traj, n, L, rng.randint(2, 16), masked=masked, fmt=fmt, tri=tri)
            M = _grid(c)
            P = M[0] * M[1] * M[2]
            # other lengths than products of 2, 3, 5 and 7 cost many times as much
            cap = 4e9 if all(_smooth(m) for m in M) else 2e8
            if P * L * c["C"] > cap or P * L * (L + 1) / 2 > 3e9:
                continue
        elif kind == "cg":
            n = _matrix(rng, "2D", 96, 320, 1, 1)
            c = _case(kind, "2D", n, _rank(rng, 3, 16), rng.randint(4, 16), tri=tri,
                      iters=rng.randint(20, 50))
            if not all(_smooth(m) for m in _grid(c)):
                continue
        elif kind == "build":
            traj = rng.choice(["2D", "2D", "stack", "3D"])
            n = _matrix(rng, traj, *((96, 320, 1, 1) if traj == "2D" else
                                     (96, 224, 8, 32) if traj == "stack" else (40, 96, 1, 1)))
            L = _rank(rng, 2, 16 if traj == "2D" else 8 if traj == "stack" else 4)
            spokes = int(round(max(n[:2]) * rng.uniform(0.5, 2.0))) if traj != "3D" else \
                int(round(n[0] ** 2 * rng.uniform(0.2, 0.43)))
            c = _case(kind, traj, n, L, 4, masked=rng.random() < 0.25, tri=tri, spokes=spokes,
                      nkx=2 * max(n[:2]))
            M = _grid(c)
            cap = 1.7e8 if all(_smooth(m) for m in M) else 2e7
            if M[0] * M[1] * M[2] * L * (L + 1) / 2 > cap:
                continue
        else:
            n = _matrix(rng, "2D", 64, 192, 1, 1)
            c = _case(kind, "2D", n, _rank(rng, 2, 8), rng.randint(2, 8), tri=tri,
                      spokes=rng.randint(32, 160), nkx=2 * max(n))
        return c


def _image(c):
    """Row-major image shape."""
    return (c["ny"], c["nx"]) if c["traj"] == "2D" else (c["nz"], c["ny"], c["nx"])


def _grid(c):
    """(Mx, My, Mz) of the upsampled grid; a stack's kz and a 2D z are not padded."""
    return (2 * c["nx"], 2 * c["ny"], 2 * c["nz"] if c["traj"] == "3D" else c["nz"])


def _grid_rm(c):
    M = _grid(c)
    return (M[1], M[0]) if c["traj"] == "2D" else (M[2], M[1], M[0])


def _pairs(L, upper):
    """(row, column) of every packed entry."""
    if upper:
        return [(i, j) for j in range(L) for i in range(j + 1)]
    return [(i, j) for j in range(L) for i in range(j, L)]


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------

def _gen(seed, what):
    return torch.Generator(device=DEV).manual_seed(int(seed) * 16 + what)


def _cgauss(shape, g):
    return torch.complex(torch.randn(shape, generator=g, device=DEV),
                         torch.randn(shape, generator=g, device=DEV))


def _axes(shape):
    """Centered coordinates in [-1, 1) of every axis, broadcastable."""
    out = []
    for a, s in enumerate(shape):
        v = (torch.arange(s, device=DEV, dtype=torch.float32) - s // 2) / max(s / 2, 1.0)
        out.append(v.reshape([-1 if b == a else 1 for b in range(len(shape))]))
    return out


def _maps(c, seed):
    """Smooth complex coil maps of unit root-sum-of-squares, (C, [z,] y, x)."""
    shape, C = _image(c), c["C"]
    ax = _axes(shape)
    r = torch.rand((C, 8), generator=_gen(seed, 1), device=DEV).cpu().numpy()
    S = torch.empty((C,) + shape, dtype=torch.complex64, device=DEV)
    for k in range(C):
        ang = 2 * math.pi * (k + 0.3 * r[k, 0]) / C
        cen = [0.9 * math.sin(ang), 0.9 * math.cos(ang)]
        if len(shape) == 3:
            cen = [1.2 * (float(r[k, 1]) - 0.5)] + cen
        mag = torch.exp(-0.5 * sum(((a - p) / 0.9) ** 2 for a, p in zip(ax, cen)))
        ph = sum(1.5 * (float(q) - 0.5) * a for q, a in zip(r[k, 2:], ax)) + 6.0 * float(r[k, 7])
        S[k] = torch.polar(mag.expand(shape).contiguous(), ph.expand(shape).contiguous())
    S /= torch.sqrt((S.real ** 2 + S.imag ** 2).sum(0))
    return S


def _phantom(c, seed):
    """Ellipses with rank coefficients that fall off, and noise, (L, [z,] y, x)."""
    shape, L = _image(c), c["L"]
    ax = _axes(shape)
    g = _gen(seed, 2)
    r = torch.rand((8, 6), generator=g, device=DEV).cpu().numpy()
    amp = _cgauss((8, L), g) / (1.0 + torch.arange(L, device=DEV)) ** 0.7
    x = 0.05 * _cgauss((L,) + shape, g)
    for e in range(8):
        inside = sum(((a - 1.2 * (float(p) - 0.5)) / (0.1 + 0.5 * float(w))) ** 2
                     for a, p, w in zip(ax, r[e, :3], r[e, 3:])) < 1.0
        x += amp[e].reshape([L] + [1] * len(shape)) * inside.to(torch.float32)
    return x.contiguous()


def _basis(L, frames, g):
    q, _ = np.linalg.qr(_cgauss((frames, L), g).cpu().numpy())
    return torch.from_numpy(np.ascontiguousarray(q.T)).to(DEV)


def _mask(c):
    """Centered indices of the sampled disc (every kz plane) or ball."""
    M, d3 = _grid(c), c["traj"] == "3D"
    ax = [torch.arange(m, device=DEV) - m // 2 for m in M]
    x2 = (2.0 * ax[0] / M[0]).double() ** 2
    y2 = (2.0 * ax[1] / M[1]).double() ** 2
    z2 = (2.0 * ax[2] / M[2]).double() ** 2 * (1.0 if d3 else 0.0)
    inside = (z2[:, None, None] + y2[None, :, None] + x2[None, None, :]) <= 1.0
    return torch.nonzero(inside.reshape(-1)).reshape(-1).contiguous()


def _kernel(c, seed, mask):
    """Packed kernel (T, grid) or (T, len(mask)) of positive semidefinite blocks."""
    L, J, M = c["L"], 6, _grid(c)
    g = _gen(seed, 3)
    frames = 4 * L
    Phi = _basis(L, frames, g)
    B = torch.stack([(Phi * torch.rand(frames, generator=g, device=DEV)) @ Phi.mH.contiguous()
                     for _ in range(J)])
    rows, cols = map(list, zip(*_pairs(L, c["tri"] == "upper")))
    comp = B[:, rows, cols].T.contiguous()          # (T, J)
    kx, ky, kz = (torch.arange(m, device=DEV, dtype=torch.float32) - m // 2 for m in M)
    d3 = c["traj"] == "3D"
    fx, fy, fz = kx * (2.0 / M[0]), ky * (2.0 / M[1]), kz * (2.0 / M[2])
    rad2 = (fy ** 2)[None, :, None] + (fx ** 2)[None, None, :] + (fz ** 2 if d3 else 0 * fz)[:, None, None]
    dens = torch.where(rad2 <= 1.0, 1.0 / (1.0 + rad2 * 0.25 * M[0] ** 2).sqrt() ** (2 if d3 else 1),
                       torch.full((), 1e-6, device=DEV))
    dens /= float(M[0] * M[1] * (M[2] if d3 else 1))
    th = torch.atan2(fy[None, :, None], fx[None, None, :])
    w = torch.empty((J,) + tuple(reversed(M)), dtype=torch.float32, device=DEV)
    for j in range(J):
        w[j] = dens * (1.0 + 0.7 * torch.cos((j + 1) * th + 0.4 * j * kz[:, None, None] + j))
    w = w.reshape(J, -1)
    if mask is not None:
        w = w[:, mask].contiguous()
    K = torch.empty((len(rows), w.shape[1]), dtype=torch.complex64, device=DEV)
    parts = torch.view_as_real(K)
    step = max(1, (1 << 28) // w.shape[1])          # real products, a few rows at a time
    for t in range(0, len(rows), step):
        parts[t:t + step, :, 0] = comp[t:t + step].real.contiguous() @ w
        parts[t:t + step, :, 1] = comp[t:t + step].imag.contiguous() @ w
    return K if mask is not None else K.reshape((len(rows),) + _grid_rm(c))


def _trajectory(c):
    """(ndim, Nkx, spokes) float32 radians in [-pi, pi)."""
    s = torch.arange(c["spokes"], device=DEV, dtype=torch.float64)[None, :]
    r = math.pi * (2.0 * torch.arange(c["nkx"], device=DEV, dtype=torch.float64) / c["nkx"] - 1.0)
    r = r[:, None]
    if c["traj"] != "3D":
        th = math.pi * GOLDEN * s
        return torch.stack([r * torch.cos(th), r * torch.sin(th)]).float().contiguous()
    z = 1.0 - (2.0 * s + 1.0) / (2.0 * c["spokes"])
    rho = torch.sqrt(torch.clamp(1.0 - z ** 2, min=0.0))
    az = math.pi * (3.0 - math.sqrt(5.0)) * s
    return torch.stack([r * rho * torch.cos(az), r * rho * torch.sin(az), r * z.expand_as(r * z)]) \
        .float().contiguous()


def _gram(c, seed):
    """Rank-1 Gram blocks, phi2[j, i, [kz,] spoke] = Phi(i, t) conj(Phi(j, t))."""
    S, planes = c["spokes"], c["nz"] if c["traj"] == "stack" else 1
    Phi = _basis(c["L"], 100, _gen(seed, 4))
    t = (torch.arange(S, device=DEV)[None, :] + S * torch.arange(planes, device=DEV)[:, None]) % 100
    p = Phi[:, t if c["traj"] == "stack" else t[0]]
    return (p[None, :] * p[:, None].conj()).contiguous()


def _inputs(c, seed):
    d = dict(mask=None)
    if c["kind"] in ("apply", "cg"):
        d["mask"] = _mask(c) if c["masked"] else None
        d["K"] = _kernel(c, seed, d["mask"])
    else:
        d["traj"], d["phi2"] = _trajectory(c), _gram(c, seed)
    if c["kind"] != "build":
        d["S"], d["x"] = _maps(c, seed), _phantom(c, seed)
    return d


# ---------------------------------------------------------------------------
# The passes
# ---------------------------------------------------------------------------

def prepare(case, seed):
    c = case
    d = _inputs(c, seed)
    n = (c["nx"], c["ny"]) if c["traj"] == "2D" else (c["nx"], c["ny"], c["nz"])
    stream = None
    if c["kind"] == "cg":
        stream = torch.cuda.Stream()   # graph replay needs a stream of its own
        torch.cuda.synchronize()
    cfg = mr.make_config(c["traj"], n, c["L"], n_coils=c["C"], triangulation=c["tri"],
                         is_masked=c["masked"],
                         num_masked=0 if d["mask"] is None else d["mask"].numel(), stream=stream)
    st = dict(case=c, cfg=cfg, d=d, stream=stream)
    if c["kind"] in ("apply", "cg"):
        st["op"] = mr.create_op(cfg, d["S"], None, None, d["mask"], _phi2_toep=d["K"])
        if c["fmt"] != "fp32":
            st["op"].set_kernel_format(c["fmt"])
    elif c["kind"] == "nufft":
        st["op"] = mr.create_op(cfg, d["S"], d["phi2"], d["traj"], method="nufft")
    return st


def run(state):
    c, d = state["case"], state["d"]
    if c["kind"] == "build":
        if not c["masked"]:
            return mr.calc_toep(state["cfg"], d["phi2"], d["traj"])
        mask = mr.calc_mask(state["cfg"], d["traj"])
        return mask, mr.calc_toep(state["cfg"], d["phi2"], d["traj"], mask)
    if c["kind"] == "cg":
        now = torch.cuda.current_stream()
        state["stream"].wait_stream(now)
        x, hist = state["op"].cg(d["x"], lam=CG_LAMBDA, iters=c["iters"], refresh=CG_REFRESH,
                                 graph=True)   # returns when the solve is done
        return x, np.asarray(hist, dtype=np.float32)
    return state["op"](d["x"])


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------

def work(case):
    c = case
    L, C, M = c["L"], c["C"], _grid(c)
    N = c["nx"] * c["ny"] * c["nz"]
    P = M[0] * M[1] * M[2]
    T = L * (L + 1) // 2
    lg = [5.0 * m * math.log2(m) if m > 1 else 0.0 for m in M]
    if c["kind"] in ("apply", "cg"):
        kept = P
        if c["masked"]:
            kept = int(P * (math.pi / 6 if c["traj"] == "3D" else math.pi / 4))
        entry = 8.0
        if c["fmt"] != "fp32":
            nb = ((L + 3) // 4) * ((L + 3) // 4 + 1) // 2
            entry = 4.0 + 4.0 * nb / T
        nbytes = T * kept * entry + 8.0 * N * (2 * L + C)
        # one direction of one volume, only the lines that hold or keep something
        fft = lg[2] * c["nx"] * c["ny"] + lg[1] * c["nx"] * M[2] + lg[0] * M[1] * M[2]
        flops = 2.0 * fft * L * C + 8.0 * L * L * kept * C + 14.0 * N * L * C
        k = c["iters"] + c["iters"] // CG_REFRESH if c["kind"] == "cg" else 1
        return {"bytes": nbytes, "flops": flops * k}
    planes = c["nz"] if c["traj"] == "stack" else 1
    nd = 3 if c["traj"] == "3D" else 2
    samples = c["spokes"] * c["nkx"]
    gram = 8.0 * L * L * planes * c["spokes"]
    if c["kind"] == "build":
        kept = P * (math.pi / (6 if nd == 3 else 4) if c["masked"] else 1.0)
        fft = lg[0] * M[1] * M[2] + lg[1] * M[0] * M[2] + (lg[2] * M[0] * M[1] if nd == 3 else 0.0)
        # gridding: the weights of 7 points an axis, summed
        return {"bytes": gram + 4.0 * nd * samples + 8.0 * T * kept,
                "flops": 2.0 * fft * T + 2.0 * samples * 7 ** nd}
    fft = (lg[0] * M[1] + lg[1] * M[0]) * planes
    return {"bytes": gram + 4.0 * nd * samples + 8.0 * N * (2 * L + C),
            "flops": C * L * (2.0 * fft + 8.0 * samples * planes * 49 + 8.0 * L * samples * planes)}


# ---------------------------------------------------------------------------
# The same in 64 bits
# ---------------------------------------------------------------------------

def _quantised(K, c):
    """The packed FP32 kernel as the 16-bit format holds it: per location and
    4x4 block of the matrix a scale (the largest stored component), the entries
    over it rounded to nearest."""
    pairs = _pairs(c["L"], c["tri"] == "upper")
    kind = torch.bfloat16 if c["fmt"] == "bf16" else torch.float16
    blocks = {}
    for t, (i, j) in enumerate(pairs):
        blocks.setdefault((max(i // 4, j // 4), min(i // 4, j // 4)), []).append(t)
    for ts in blocks.values():
        s = torch.zeros_like(K[0].real)
        for t in ts:
            s = torch.maximum(s, torch.maximum(K[t].real.abs(), K[t].imag.abs()))
        s = torch.where(s > 0, s, torch.ones_like(s))
        inv = 1.0 / s
        for t in ts:
            K[t] = torch.complex((K[t].real * inv).to(kind).float() * s,
                                 (K[t].imag * inv).to(kind).float() * s)
    return K


class _Exact:
    """A^H A of an apply case in complex128, coil by coil."""

    def __init__(self, c, d):
        self.c, self.S = c, d["S"]
        self.full = None if d["mask"] is None else d["mask"]
        self.K = _quantised(d["K"], c) if c["fmt"] != "fp32" else d["K"]
        self.shape, self.grid = _image(c), _grid_rm(c)
        self.dims = tuple(range(1, 1 + len(self.shape)))
        # centered image sample i sits at natural position (i - n//2) mod M
        self.at = [(torch.arange(n, device=DEV) - n // 2) % m for n, m in zip(self.shape, self.grid)]

    def entry(self, t):
        if self.full is None:
            k = self.K[t].to(torch.complex128)
        else:
            k = torch.zeros(math.prod(self.grid), dtype=torch.complex128, device=DEV)
            k[self.full] = self.K[t].to(torch.complex128)
            k = k.reshape(self.grid)
        return torch.fft.ifftshift(k)

    def index(self):
        nd = len(self.shape)
        return (slice(None),) + tuple(a.reshape([-1 if b == i else 1 for b in range(nd)])
                                      for i, a in enumerate(self.at))

    def __call__(self, x):
        c, L = self.c, self.c["L"]
        P = math.prod(self.grid)
        out = torch.zeros((L,) + self.shape, dtype=torch.complex128, device=DEV)
        per = max(1, min(c["C"], int(1.5e9 // (P * L))))   # coils at a time
        ix = (slice(None),) + self.index()
        for c0 in range(0, c["C"], per):
            S = self.S[c0:c0 + per].to(torch.complex128)
            nc = S.shape[0]
            v = torch.zeros((nc, L) + self.grid, dtype=torch.complex128, device=DEV)
            v[ix] = S[:, None] * x[None]
            for k in range(nc):
                v[k] = torch.fft.fftn(v[k], dim=self.dims)
            y = torch.zeros_like(v)
            for t, (i, j) in enumerate(_pairs(L, c["tri"] == "upper")):
                a = self.entry(t)
                y[:, j].addcmul_(v[:, i], a)
                if i != j:
                    y[:, i].addcmul_(v[:, j], a.conj().resolve_conj())
            del v
            for k in range(nc):
                out += S[k].conj() * torch.fft.ifftn(y[k], dim=self.dims, norm="forward")[self.index()]
        return out


def _exact_cg(c, d):
    """Conjugate gradients in 64 bits; the residual is the true one throughout."""
    A, lam = _Exact(c, d), CG_LAMBDA
    b = d["x"].to(torch.complex128)
    x, r, p = torch.zeros_like(b), b.clone(), b.clone()
    dot = lambda u, v: float((u.conj() * v).real.sum())  # noqa: E731
    rr = bb = dot(b, b)
    hist = [1.0]
    for _ in range(c["iters"]):
        Ap = A(p) + lam * p
        alpha = rr / dot(p, Ap)
        x += alpha * p
        r -= alpha * Ap
        new = dot(r, r)
        hist.append(math.sqrt(new / bb))
        p = r + (new / rr) * p
        rr = new
    return x, np.asarray(hist)


def _phases(coord, m):
    """e^{-i d x} of every sample (rows) and centered mode or pixel d (columns)."""
    d = (torch.arange(m, device=DEV) - m // 2).double()
    a = coord.reshape(-1, 1).double() * d[None, :]
    return torch.polar(torch.ones_like(a), -a)


def _exact_mask(c, traj):
    M = _grid(c)
    nd = traj.shape[0]
    at = []
    for a in range(nd):
        sc = torch.tensor(M[a] / 6.283185307179586, dtype=torch.float32, device=DEV)
        at.append((torch.round(traj[a].reshape(-1) * sc).long() + M[a] // 2) % M[a])
    marks = torch.zeros(tuple(reversed(M[:nd])), dtype=torch.bool, device=DEV)
    marks[tuple(reversed(at))] = True
    for ax in range(nd):
        marks = torch.stack([torch.roll(marks, s, ax) for s in range(-2, 3)]).any(0)
    flat = torch.nonzero(marks.reshape(-1)).reshape(-1)
    if c["traj"] == "stack":
        flat = torch.cat([flat + M[0] * M[1] * k for k in range(M[2])])
    return flat


def _exact_build(c, d):
    """The inverse DFT of the exact point-spread functions, sums over all samples."""
    M, L, traj = _grid(c), c["L"], d["traj"]
    nd, S = traj.shape[0], c["spokes"]
    planes = c["nz"] if c["traj"] == "stack" else 1
    pairs = _pairs(L, c["tri"] == "upper")
    B = d["phi2"].reshape(L, L, planes, S)
    coef = torch.stack([B[j, i] for i, j in pairs]).reshape(-1, S).to(torch.complex128)
    shape = tuple(reversed(M[:nd]))
    psf = torch.zeros((coef.shape[0], math.prod(shape)), dtype=torch.complex128, device=DEV)
    step = max(1, min(S, int(2.5e8 // math.prod(shape))))
    for s0 in range(0, S, step):
        rows = []
        for s in range(s0, min(S, s0 + step)):
            E = [_phases(traj[a, :, s], M[a]) for a in range(nd)]
            left = E[1].T if nd == 2 else (E[2].T[:, None, :] * E[1].T[None]).reshape(-1, c["nkx"])
            rows.append((left.contiguous() @ E[0]).reshape(-1))
        psf.addmm_(coef[:, s0:s0 + len(rows)].contiguous(), torch.stack(rows))
    K = torch.empty((coef.shape[0],) + shape, dtype=torch.complex64, device=DEV)
    dims = tuple(range(nd))
    for q in range(coef.shape[0]):
        K[q] = torch.fft.fftshift(torch.fft.ifftn(torch.fft.ifftshift(psf[q].reshape(shape), dims)), dims)
    K = K.reshape((len(pairs),) + ((planes,) if c["traj"] == "stack" else ()) + shape)
    if not c["masked"]:
        return K
    mask = _exact_mask(c, traj)
    return mask, K.reshape(len(pairs), -1)[:, mask].contiguous()


def _exact_nufft(c, d):
    """Sums over all samples and pixels (2D)."""
    traj, L, S = d["traj"], c["L"], c["spokes"]
    Ex, Ey = (_phases(traj[a], m) for a, m in ((0, c["nx"]), (1, c["ny"])))   # (samples, pixels)
    B = d["phi2"].to(torch.complex128)                                       # [j, i, spoke]
    out = torch.zeros((L, c["ny"], c["nx"]), dtype=torch.complex128, device=DEV)
    for k in range(c["C"]):
        s = d["S"][k].to(torch.complex128)
        v = [((s * d["x"][l].to(torch.complex128)) @ Ex.T.contiguous() * Ey.T).sum(0).reshape(-1, S)
             for l in range(L)]
        for l in range(L):
            y = sum(v[j] * B[l, j][None] for j in range(L)).reshape(-1, 1)
            out[l] += s.conj() * ((y * Ey.conj()).T.contiguous() @ Ex.conj().resolve_conj())
    return out


def exact(case, seed):
    c = case
    if c["kind"] == "build" and c["traj"] == "3D" and \
            8.0 * c["spokes"] * c["nkx"] * math.prod(_grid(c)) > 1e14:
        return None
    d = _inputs(c, seed)
    if c["kind"] == "apply":
        return _Exact(c, d)(d["x"].to(torch.complex128))
    if c["kind"] == "cg":
        return _exact_cg(c, d)
    return _exact_build(c, d) if c["kind"] == "build" else _exact_nufft(c, d)
