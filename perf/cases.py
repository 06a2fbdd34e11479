"""Workloads of the reconstruction library, from the smallest operator call to
whole solves and the set-up of a protocol, through the package's public entry
points.  Each case is a dict of plain values:

  kind     apply | cg | backproject | forward | build | cartesian | calibrate
  size     image size, e.g. "256x256" (Julia order, x first)
  coils, K coil count and subspace size; real: a Float32 basis (real kernel)
  nt, spokes, nr   frames, spokes per frame, samples per spoke (golden angle in
                   2D, golden-means koosh-ball in 3D)
  precision, mode, iters, dcf, masked, lines   options of the kind

The plain 64-bit values (`exact`) are direct non-uniform sums (matrix products
of exponentials), dense FFTs and the textbook CG recurrence in torch.
"""
from __future__ import annotations

import importlib.util
import math
import os
import sys

import numpy as np
import torch

DEV = "cuda:0"


def _pkg():
    name = "mrisubspacerecon_amd"
    if name not in sys.modules:
        here = os.path.join(os.getcwd(), "mrfingerprintingrecon.jl_amd")
        spec = importlib.util.spec_from_file_location(name, os.path.join(here, "__init__.py"),
                                                      submodule_search_locations=[here])
        mod = importlib.util.module_from_spec(spec)
        sys.modules[name] = mod
        spec.loader.exec_module(mod)
    return sys.modules[name]


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # one operator call on the tests' smallest image: latency and launches
        dict(name="apply-64", kind="apply", size="64x64", coils=8, K=4, real=False, nt=100,
             spokes=1, nr=128, precision="f32"),
        # an image size off the powers of two, rectangular, ComplexF64 vectors
        dict(name="apply-240x300", kind="apply", size="240x300", coils=12, K=6, real=True, nt=600,
             spokes=1, nr=480, precision="f64"),
        # a small solve with the default options of cg_
        dict(name="cg-128x96", kind="cg", size="128x96", coils=6, K=4, real=False, nt=400,
             spokes=1, nr=256, precision="f64", mode="device", iters=20),
        # the headline solve's CG (captured graph, compact intermediates)
        dict(name="cg-256", kind="cg", size="256x256", coils=20, K=5, real=False, nt=1000,
             spokes=1, nr=512, precision="f64c", mode="graph", iters=25),
        # the 3D operator, which a 128^3 solve calls once per iteration
        dict(name="apply-128c", kind="apply", size="128x128x128", coils=16, K=4, real=False,
             nt=2000, spokes=4, nr=256, precision="f64c"),
        # CG's right-hand side for new data of a known 2D protocol
        dict(name="backproject-256", kind="backproject", size="256x256", coils=20, K=5, real=False,
             nt=1000, spokes=1, nr=512, dcf="none", masked=False),
        # the same in 3D with the koosh-ball density weights
        dict(name="backproject-96c", kind="backproject", size="96x96x96", coils=12, K=4,
             real=False, nt=1000, spokes=4, nr=192, dcf="radial_3D", masked=False),
        # the data of known coefficient images (simulation, data consistency)
        dict(name="forward-256", kind="forward", size="256x256", coils=20, K=5, real=False,
             nt=1000, spokes=1, nr=512),
        # a new protocol: trajectory planning and the Toeplitz kernel, 2D and 3D
        dict(name="build-256", kind="build", size="256x256", coils=1, K=5, real=False, nt=1000,
             spokes=1, nr=512),
        dict(name="build-80x72x64", kind="build", size="80x72x64", coils=1, K=4, real=True, nt=500,
             spokes=4, nr=160),
        # a Cartesian scan: backprojection and solve
        dict(name="cartesian-256", kind="cartesian", size="256x256", coils=20, K=5, real=False,
             nt=1000, lines=8, precision="f64", mode="graph", iters=25),
        # coil-map calibration of the 2D protocol (region, coil-wise solves, k-space)
        dict(name="calibrate-256", kind="calibrate", size="256x256", coils=20, nt=1000, spokes=1,
             nr=512, iters=100),
    ]


def _smooth_up(n):
    """Smallest 2^a 3^b 5^c >= n."""
    while True:
        m = n
        for p in (2, 3, 5):
            while m % p == 0:
                m //= p
        if m == 1:
            return n
        n += 1


_SMOOTH = sorted({_smooth_up(n) for n in range(16, 401)})


def _size(rng, d):
    lo, hi = ((48, 384) if d == 2 else (24, 128))
    first = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    out = []
    for i in range(d):
        want = first * (1.0 if i == 0 else rng.choice([1.0, 1.0, 0.75, 0.85, 1.2]))
        out.append(min((n for n in _SMOOTH if lo <= n <= hi), key=lambda n: abs(math.log(n / want))))
    return out


def _seconds(case):
    w = work(case)
    return w["bytes"] / 4e12 + w["flops"] / 5e13


def draw(rng):
    most = max(_seconds(c) for c in listed())
    while True:
        case = _draw(rng)
        if _seconds(case) <= most:
            return case


def _draw(rng):
    kind = rng.choice(["apply", "apply", "cg", "backproject", "backproject", "forward", "build",
                       "cartesian", "calibrate"])
    d = 3 if kind in ("apply", "cg", "backproject", "forward", "build") and rng.random() < 0.35 else 2
    n = _size(rng, d)
    coils = int(round(math.exp(rng.uniform(math.log(3.0), math.log(32.0 if d == 2 else 16.0)))))
    K = rng.randint(2, 8 if d == 2 else 5)
    nt = rng.randint(200, 1000)
    spokes = rng.randint(1, 3) if d == 2 else rng.randint(2, 4)
    nr = 2 * max(n)
    case = dict(kind=kind, size="x".join(str(v) for v in n), coils=coils, K=K,
                real=rng.random() < 0.4, nt=nt, spokes=spokes, nr=nr)
    if kind == "apply":
        case["precision"] = rng.choice(["f32", "f64", "f64c"])
    elif kind == "cg":
        case.update(precision=rng.choice(["f64", "f64c"]), mode=rng.choice(["device", "graph"]),
                    iters=rng.randint(8, 25 if d == 2 else 12))
    elif kind == "backproject":
        case.update(dcf=rng.choice(["none", "radial_%dD" % d]), masked=rng.random() < 0.4)
    elif kind == "build":
        case.update(coils=1, K=rng.randint(1, 6 if d == 2 else 4))
    elif kind == "cartesian":
        for k in ("spokes", "nr"):
            del case[k]
        case.update(lines=rng.randint(2, 10), precision=rng.choice(["f64", "f64c"]),
                    mode=rng.choice(["device", "graph"]), iters=rng.randint(8, 25))
    elif kind == "calibrate":
        n = max(96, n[0])
        n = min((v for v in _SMOOTH if v >= 96), key=lambda v: abs(v - n))
        for k in ("K", "real"):
            del case[k]
        case.update(size="%dx%d" % (n, n), nr=2 * n, iters=rng.randint(30, 100))
    return case


def _shape(case):
    return tuple(int(v) for v in case["size"].split("x"))


def work(case):
    """Bytes and operations of one pass that no implementation avoids: every
    input read once, every output written once; zero-padded FFTs counted on
    their non-zero lines, interpolation at 8 taps per dimension."""
    N = _shape(case)
    d = len(N)
    V = math.prod(N)
    G = (2 ** d) * V
    C, K = case["coils"], case.get("K", 1)
    P = K * (K + 1) // 2
    sl = 4 if case.get("real", True) else 8
    fill = math.pi / 4 if d == 2 else math.pi / 6      # share of the grid a radial scan reaches
    kernel = fill * G * P * sl

    def fft(channels, doubled):
        """5 n log2 n per line; a doubled axis transforms only what precedes it."""
        ops = 0.0
        for a in range(d):
            lines_cells = V * (2 ** (a + 1)) if doubled else V
            n = 2 * N[a] if doubled else N[a]
            ops += 5.0 * lines_cells * math.log2(n)
        return channels * ops

    M = case["nt"] * case.get("spokes", 1) * case.get("nr", 1)
    kind = case["kind"]
    if kind in ("apply", "cg"):
        sv = 8 if case["precision"] == "f32" or kind == "cg" else 16
        flops = 2 * fft(C * K, True) + C * fill * G * 8 * K * K + 2 * 8 * C * K * V
        one = 2 * sv * K * V + 8 * C * V + kernel
        it = case.get("iters", 1)
        return {"bytes": float(it * one), "flops": float(it * flops)}
    if kind == "backproject":
        flops = M * C * K * (8 + 4 * 8 ** d) + fft(C * K, True) + 8 * C * K * V
        return {"bytes": float(8 * M * C + 4 * d * M + 8 * C * V + 8 * K * V), "flops": float(flops)}
    if kind == "forward":
        flops = M * C * K * (8 + 4 * 8 ** d) + fft(C * K, True) + 8 * C * K * V
        return {"bytes": float(8 * M * C + 4 * d * M + 8 * C * V + 8 * K * V), "flops": float(flops)}
    if kind == "build":
        flops = M * P * (8 + 4 * 8 ** d) + 2 * P * 5 * (2 ** d) * G * math.log2(4 ** d * G) / 2
        return {"bytes": float(4 * d * M + kernel + 8 * fill * G), "flops": float(flops)}
    if kind == "cartesian":
        M = case["nt"] * case["lines"] * N[0]
        it = case["iters"]
        flops = M * C * K * 8 + fft(C * K, False) + \
            it * (2 * fft(C * K, False) + C * V * 8 * K * K + 16 * C * K * V)
        return {"bytes": float(8 * M * C + 4 * d * M + 8 * C * V + it * (16 * K * V + 8 * C * V + V * K * K * sl)),
                "flops": float(flops)}
    # calibrate: the central samples, K = 1 solves of every coil on the calibration size
    n = 32.0 * 32.0
    inside = M * 32.0 / max(N)
    flops = inside * C * (8 + 4 * 64) + case["iters"] * C * (2 * 5 * 4 * n * 12)
    return {"bytes": float(4 * d * M + 8 * inside * C + 8 * C * n + case["iters"] * (C * n * 16 + 4 * n * 4)),
            "flops": float(flops)}


# --------------------------------------------------------------------- inputs
def _gen(seed, salt):
    g = torch.Generator(device=DEV)
    g.manual_seed((seed * 7919 + salt) % (2 ** 62))
    return g


def _trajectory(case, seed):
    """(Nt, spokes*nr, d) float32: golden-angle radial or golden-means
    koosh-ball, starting at a spoke given by the seed (of a "build" case, whose
    mask has as many cells as the samples reach, by the case)."""
    d = len(_shape(case))
    nt, ns, nr = case["nt"], case["spokes"], case["nr"]
    kr = (torch.arange(nr, device=DEV, dtype=torch.float64) - (nr - 1) / 2.0) / nr
    s = (torch.arange(nt, device=DEV)[:, None] + nt * torch.arange(ns, device=DEV)[None]).double()
    s = s + (13 * nt if case["kind"] == "build" else seed % 9973)
    if d == 2:
        ang = s * (math.pi / ((1.0 + math.sqrt(5.0)) / 2.0))
        u = torch.stack([-torch.cos(ang), torch.sin(ang)], -1)
    else:
        th = torch.arccos(torch.remainder(s * 0.4655712318767680, 1.0))
        ph = s * (2.0 * math.pi * 0.6823278038280193)
        u = torch.stack([-torch.sin(th) * torch.cos(ph), torch.sin(th) * torch.sin(ph),
                         torch.cos(th)], -1)
    k = u[:, :, None, :] * kr[None, None, :, None]
    return k.clamp(-0.5, 0.5).to(torch.float32).reshape(nt, ns * nr, d).contiguous()


def _basis(case, seed):
    """(K, Nt): the leading left singular vectors of a T2-decay dictionary."""
    nt, K = case["nt"], case["K"]
    rng = np.random.default_rng(seed)
    t2 = rng.uniform(20.0, 300.0, size=100)
    t = (np.arange(1, nt + 1) * (1000.0 / nt))[:, None]
    ph = np.exp(1j * 0.3 * t / 1000.0) if not case["real"] else 1.0
    u, _, _ = np.linalg.svd(np.exp(-t / t2[None]), full_matrices=False)
    u = (u[:, :K] * ph).T
    return torch.from_numpy(np.ascontiguousarray(u.astype(np.float32 if case["real"] else np.complex64))).to(DEV)


def _coords(N):
    """Coordinates r - N/2 per axis, broadcast over (..., N2, N1)."""
    d = len(N)
    out = []
    for a in range(d):
        sh = [1] * d
        sh[d - 1 - a] = N[a]
        out.append((torch.arange(N[a], device=DEV, dtype=torch.float64) - N[a] / 2).reshape(sh))
    return out


def _coil_centres(case):
    N, C = _shape(case), case["coils"]
    fov = float(max(N))
    out = []
    for c in range(C):
        if len(N) == 2:
            a = 2 * math.pi * c / C
            out.append((0.3 * fov * math.cos(a), 0.3 * fov * math.sin(a)))
        else:
            z = 1 - 2 * (c + 0.5) / C
            r = math.sqrt(max(0.0, 1 - z * z))
            a = c * math.pi * (3 - math.sqrt(5))
            out.append((0.3 * fov * r * math.cos(a), 0.3 * fov * r * math.sin(a), 0.3 * fov * z))
    return out, fov / 3.0


def _maps(case, seed):
    """(C, ..., N2, N1) complex64 Gaussian coil profiles of unit root sum of squares."""
    N = _shape(case)
    rng = np.random.default_rng(seed + 17)
    x = _coords(N)
    centres, sig = _coil_centres(case)
    m = torch.empty((case["coils"],) + N[::-1], dtype=torch.complex64, device=DEV)
    rss = torch.zeros(N[::-1], dtype=torch.float64, device=DEV)
    for c, ctr in enumerate(centres):
        a = torch.exp(-sum((xi - ci) ** 2 for xi, ci in zip(x, ctr)) / (2 * sig * sig))
        ph = rng.uniform(0, 2 * math.pi)
        m[c] = torch.complex(a * math.cos(ph), a * math.sin(ph)).to(torch.complex64)
        rss += a * a
    m /= rss.sqrt().to(torch.float32)
    return m


def _blobs(case, seed):
    """Gaussian blobs (coefficient, centre, width, amplitude) of the phantom."""
    N = _shape(case)
    rng = np.random.default_rng(seed + 29)
    fov = float(min(N))
    out = []
    for k in range(case.get("K", 1)):
        for _ in range(3):
            out.append((k, rng.uniform(-0.25, 0.25, size=len(N)) * fov, rng.uniform(0.03, 0.12) * fov,
                        complex(rng.normal(), rng.normal())))
    return out


def _phantom(case, seed):
    """(K, ..., N2, N1) complex64 coefficient images: blobs and 2 % noise."""
    N, K = _shape(case), case["K"]
    x = _coords(N)
    img = torch.zeros((K,) + N[::-1], dtype=torch.complex128, device=DEV)
    for k, ctr, s, a in _blobs(case, seed):
        e = torch.exp(-sum((xi - float(ci)) ** 2 for xi, ci in zip(x, ctr)) / (2 * s * s))
        img[k] += a * e
    img += 0.02 * torch.randn(img.shape, dtype=torch.complex128, device=DEV, generator=_gen(seed, 3))
    return img.to(torch.complex64)


def _signal(case, seed, trj, U):
    """(C, Nt, Nsamp) complex64: the blobs' analytic k-space signal seen by
    Gaussian coils, with noise 30 dB below it."""
    centres, sc = _coil_centres(case)
    d = len(_shape(case))
    kx = trj.double().permute(2, 0, 1)
    k2 = (kx ** 2).sum(0)
    data = torch.empty((case["coils"],) + tuple(trj.shape[:2]), dtype=torch.complex64, device=DEV)
    Uc = U.to(torch.complex128)
    for c, cc in enumerate(centres):
        y = torch.zeros(tuple(trj.shape[:2]), dtype=torch.complex128, device=DEV)
        for k, ctr, s, a in _blobs(case, seed):
            var = 1.0 / (1.0 / s ** 2 + 1.0 / sc ** 2)
            mu = [var * (float(p) / s ** 2 + q / sc ** 2) for p, q in zip(ctr, cc)]
            amp = a * math.exp(-0.5 * sum((float(p) - q) ** 2 for p, q in zip(ctr, cc)) / (s ** 2 + sc ** 2))
            amp *= (2 * math.pi * var) ** (d / 2)
            mag = torch.exp(-2 * math.pi ** 2 * var * k2)
            arg = -2 * math.pi * sum(m * kx[i] for i, m in enumerate(mu))
            y += (amp * Uc[k])[:, None] * torch.polar(mag, arg)
        data[c] = y.to(torch.complex64)
    rms = float(data.abs().double().pow(2).mean().sqrt())
    data += (rms * 10 ** -1.5) * torch.randn(data.shape, dtype=torch.complex64, device=DEV, generator=_gen(seed, 5))
    return data


def _cells(trj, n):
    """Base cell of every sample on the grid n: floor(mod(-k, 1) n), (M, d)."""
    t = -trj.reshape(-1, trj.shape[-1]).double()
    t = t - torch.floor(t)
    nn = torch.tensor(n, device=DEV, dtype=torch.float64)
    return torch.minimum(torch.floor(t * nn), nn - 1).to(torch.int64)


def _mask_cells(trj, n):
    """Sorted 0-based linear indices (x fastest) of the cells within base-3 ..
    base+4 of a sample, periodic."""
    d = len(n)
    base = torch.zeros(n[::-1], dtype=torch.bool, device=DEV)
    q = _cells(trj, n)
    base[tuple(q[:, a] for a in range(d - 1, -1, -1))] = True
    for a in range(d):
        out = torch.zeros_like(base)
        for o in range(-3, 5):
            out |= torch.roll(base, o, dims=d - 1 - a)
        base = out
    return torch.nonzero(base.reshape(-1)).reshape(-1)


def _stored_kernel(case, trj, U):
    """A precomputed packed kernel (Nkm, P) and its 1-based mask, as a protocol's
    kernel file holds them: the samples' Gram matrices of the basis gridded over
    their eight nearest cells per dimension (positive semidefinite per cell)."""
    N = _shape(case)
    n = tuple(2 * v for v in N)
    d, K = len(n), case["K"]
    G = math.prod(n)
    q = _cells(trj, n)
    lin = torch.zeros(q.shape[0], dtype=torch.int64, device=DEV)
    for a in range(d - 1, -1, -1):
        lin = lin * n[a] + q[:, a]
    frame = torch.arange(case["nt"], device=DEV).repeat_interleave(trj.shape[1])
    km = _mask_cells(trj, n)
    taps = [math.comb(7, i) / 128.0 for i in range(8)]
    real = case["real"]
    lam = torch.empty((km.numel(), K * (K + 1) // 2), dtype=torch.float32 if real else torch.complex64, device=DEV)
    U64 = U.to(torch.float64 if real else torch.complex128)
    p = 0
    for k in range(K):
        for j in range(k + 1):
            gram = (U64[j].conj() * U64[k])
            parts = []
            for part in ([gram] if real else [gram.real, gram.imag]):
                fixed = torch.round(part * 2.0 ** 44).to(torch.int64)[frame]
                acc = torch.zeros(G, dtype=torch.int64, device=DEV)
                acc.index_add_(0, lin, fixed)
                g = acc.double().reshape(n[::-1]) * 2.0 ** -44
                for a in range(d):
                    g = sum(w * torch.roll(g, o, dims=d - 1 - a) for w, o in zip(taps, range(-3, 5)))
                parts.append(g.reshape(-1)[km])
            lam[:, p] = (parts[0] if real else torch.complex(parts[0], parts[1])).to(lam.dtype)
            p += 1
    return lam, km + 1


def _cartesian_trj(case, seed):
    """(Nt, lines*N1, 2) int32: `lines` random phase-encode lines per frame."""
    nx, ny = _shape(case)
    g = _gen(seed, 11)
    pe = torch.rand((case["nt"], ny), device=DEV, generator=g).argsort(1)[:, :case["lines"]] + 1
    t = torch.empty((case["nt"], case["lines"], nx, 2), dtype=torch.int32, device=DEV)
    t[..., 0] = torch.arange(1, nx + 1, device=DEV, dtype=torch.int32)
    t[..., 1] = pe.to(torch.int32)[:, :, None]
    return t.reshape(case["nt"], -1, 2).contiguous()


def _mask(case, seed, trj):
    if not case.get("masked"):
        return None
    return torch.rand(tuple(trj.shape[:2]), device=DEV, generator=_gen(seed, 7)) < 0.8


def _inputs(case, seed):
    """Everything made from the seed: what prepare hands over and exact reads."""
    kind = case["kind"]
    s = {}
    if kind == "calibrate":
        full = dict(case, K=1, real=True)
        s["trj"] = _trajectory(case, seed)
        one = torch.ones((1, case["nt"]), dtype=torch.float32, device=DEV)
        s["data"] = _signal(full, seed, s["trj"], one)
        return s
    s["U"] = _basis(case, seed)
    if kind == "cartesian":
        s["trj"] = _cartesian_trj(case, seed)
        s["maps"] = _maps(case, seed)
        nx, ny = _shape(case)
        # the phantom's k-space on the scanned cells
        x = _phantom(case, seed)
        q = _cart_cells(s["trj"], (nx, ny))
        data = torch.empty((case["coils"], case["nt"], s["trj"].shape[1]), dtype=torch.complex64, device=DEV)
        for c in range(case["coils"]):
            f = torch.fft.fftn(torch.fft.ifftshift(s["maps"][c] * x, dim=(-2, -1)), dim=(-2, -1)).reshape(case["K"], -1)
            data[c] = sum(s["U"][k][:, None] * f[k][q] for k in range(case["K"]))
        s["data"] = data + 0.5 * torch.randn(data.shape, dtype=torch.complex64, device=DEV, generator=_gen(seed, 5))
        return s
    s["trj"] = _trajectory(case, seed)
    if kind == "build":
        return s
    s["maps"] = _maps(case, seed)
    if kind in ("apply", "cg"):
        s["lam"], s["km"] = _stored_kernel(case, s["trj"], s["U"])
        x = _phantom(case, seed)
        if kind == "cg":
            x = _apply64(_shape(case), _dense(case, s), s["maps"], x).to(torch.complex64)
        s["b"] = x
    elif kind == "backproject":
        s["mask"] = _mask(case, seed, s["trj"])
        s["data"] = _signal(case, seed, s["trj"], s["U"])
    elif kind == "forward":
        s["x"] = _phantom(case, seed)
    return s


# ------------------------------------------------------------- prepare and run
def prepare(case, seed):
    msr = _pkg()
    N, kind = _shape(case), case["kind"]
    s = _inputs(case, seed)
    st = {"case": case, "N": N}
    if kind in ("apply", "cg"):
        A = msr.NFFTNormalOp(N, s["lam"], s["km"], cmaps=s["maps"])
        b = s["b"].reshape(-1)
        if kind == "apply" and case["precision"] != "f32":
            b = b.to(torch.complex128)
        st.update(A=A, b=b, x=torch.empty_like(b))
    elif kind == "backproject":
        st.update(traj=msr.plan_trajectory(s["trj"], s["mask"]), maps=list(s["maps"]), U=s["U"],
                  data=s["data"])
    elif kind == "forward":
        st.update(traj=msr.plan_trajectory(s["trj"]), maps=list(s["maps"]), U=s["U"], x=s["x"])
    elif kind == "build":
        st.update(trj=s["trj"], U=s["U"])
    elif kind == "cartesian":
        traj = msr.plan_trajectory(s["trj"])
        maps = list(s["maps"])
        st.update(traj=traj, maps=maps, U=s["U"], data=s["data"],
                  A=msr.FFTNormalOp(N, traj, s["U"], cmaps=maps),
                  b=torch.empty((case["K"],) + N[::-1], dtype=torch.complex64, device=DEV),
                  x=torch.empty(case["K"] * math.prod(N), dtype=torch.complex64, device=DEV))
    else:
        st.update(trj=s["trj"], data=s["data"])
    return st


def run(st):
    msr = _pkg()
    case, kind = st["case"], st["case"]["kind"]
    if kind == "apply":
        if case["precision"] == "f32":
            return msr.mul_(st["x"], st["A"], st["b"])
        return st["A"].A.mul_f64_(st["x"], st["b"], compact=case["precision"] == "f64c")
    if kind == "cg":
        return msr.cg_(st["x"], st["A"], st["b"], maxiter=case["iters"], reltol=0.0,
                       initially_zero=True, mode=case["mode"], precision=case["precision"])
    if kind == "backproject":
        return msr.calculate_backprojection(st["data"], st["traj"], st["maps"], U=st["U"],
                                            density_compensation=case["dcf"])
    if kind == "forward":
        return msr.forward(st["x"], st["traj"], cmaps=st["maps"], U=st["U"])
    if kind == "build":
        A = msr.NFFTNormalOp(st["N"], st["trj"], st["U"])
        return A.prod.A.Λ, A.prod.A.kmask_indcs
    if kind == "cartesian":
        b = msr.calculate_backprojection(st["data"], st["traj"], st["maps"], U=st["U"], out=st["b"])
        x = msr.cg_(st["x"], st["A"], b.reshape(-1), maxiter=case["iters"], reltol=0.0,
                    initially_zero=True, mode=case["mode"], precision=case["precision"])
        return b, x
    N = st["N"]
    calib = msr.default_calib_size(N)
    trj, mask = msr.calibration_region(st["trj"], N, calib)
    x = msr.reconstruct_coilwise(st["data"], trj, calib, sample_mask=mask, Niter_cg=case["iters"])
    return x, msr.calibration_kspace(x)


# ---------------------------------------------------- the same in plain 64 bits
def _dense(case, s):
    """Packed 64-bit kernel on the whole grid, (P, cells)."""
    G = math.prod(2 * v for v in _shape(case))
    lam = s["lam"]
    out = torch.zeros((lam.shape[1], G), dtype=torch.float64 if not lam.is_complex() else torch.complex128, device=DEV)
    out[:, s["km"] - 1] = lam.T.to(out.dtype)
    return out


def _multiply(dense, kl):
    """Per-cell Hermitian multiply of (K, cells) by a packed upper triangle."""
    K = kl.shape[0]
    out = torch.zeros_like(kl)
    for k in range(K):
        for j in range(k + 1):
            v = dense[j + k * (k + 1) // 2]
            out[j] += v * kl[k]
            if j != k:
                out[k] += v.conj() * kl[j]
    return out


def _apply64(N, dense, maps, b, double=True):
    d = len(N)
    n = tuple((2 if double else 1) * v for v in N)
    K = b.shape[0]
    b = b.to(torch.complex128)
    out = torch.zeros_like(b)
    axes = tuple(range(1, d + 1))
    crop = (slice(None),) + tuple(slice(0, v) for v in N[::-1])
    for c in range(1 if maps is None else maps.shape[0]):
        m = None if maps is None else maps[c].to(torch.complex128)
        f = torch.zeros((K,) + n[::-1], dtype=torch.complex128, device=DEV)
        f[crop] = b if m is None else m * b
        f = torch.fft.fftn(f, dim=axes)
        f = _multiply(dense, f.reshape(K, -1)).reshape(f.shape)
        f = torch.fft.ifftn(f, dim=axes)[crop]
        out += f if m is None else m.conj() * f
    return out


def _cg64(apply, b, iters):
    x, r, u = torch.zeros_like(b), b.clone(), torch.zeros_like(b)
    res, prev = float(torch.linalg.norm(b)), 1.0
    for _ in range(iters):
        if res <= 0.0:
            break
        u = r + (res * res / (prev * prev)) * u
        c = apply(u)
        a = res * res / complex((u.conj() * c).sum())
        x = x + a * u
        r = r - a * c
        prev, res = res, float(torch.linalg.norm(r))
    return x


def _waves(k, n, sign, centred):
    r = torch.arange(n, device=DEV, dtype=torch.float64)
    r = r - n // 2 if centred else torch.where(r < (n + 1) // 2, r, r - n)
    ph = sign * 2.0 * math.pi * k.double()[:, None] * r[None]
    return torch.polar(torch.ones_like(ph), ph)


def _sum_to_grid(trj, v, n, centred=True):
    """out[ch, r] = sum_m v[ch, m] exp(+2 pi i k_m r); trj (M, d), v(slice) -> (ch, m)."""
    d = len(n)
    M = trj.shape[0]
    nch = v(slice(0, 1)).shape[0]
    outer = math.prod(n[1:])
    out = torch.zeros((nch * n[-1] if d == 3 else nch, math.prod(n[:-1]) if d == 3 else outer * n[0]),
                      dtype=torch.complex128, device=DEV)
    chunk = 8192 if d == 3 else 65536
    for a in range(0, M, chunk):
        sl = slice(a, min(M, a + chunk))
        E = [_waves(trj[sl, i], n[i], 1.0, centred) for i in range(d)]
        vv = v(sl)
        if d == 2:
            for ch in range(nch):
                w = (vv[ch][:, None] * E[1]).T.contiguous()
                out[ch] += (w @ E[0]).reshape(-1)
        else:
            right = (E[1][:, :, None] * E[0][:, None, :]).reshape(E[0].shape[0], -1)
            left = (vv[:, None, :] * E[2].T[None]).reshape(nch * n[2], -1)
            out.addmm_(left, right)
    return out.reshape((nch,) + tuple(n[::-1]))


def _sum_at_samples(trj, x):
    """y[ch, m] = sum_r x[ch, r] exp(-2 pi i k_m r) of centred images."""
    d = trj.shape[1]
    n = x.shape[1:][::-1]
    out = torch.empty((x.shape[0], trj.shape[0]), dtype=torch.complex128, device=DEV)
    chunk = 4096 if d == 3 else 16384
    for a in range(0, trj.shape[0], chunk):
        sl = slice(a, min(trj.shape[0], a + chunk))
        E = [_waves(trj[sl, i], n[i], -1.0, True) for i in range(d)]
        if d == 2:
            t = (x.reshape(-1, n[0]) @ E[0].T.contiguous()).reshape(x.shape[0], n[1], -1)
            out[:, sl] = (t * E[1].T[None]).sum(1)
        else:
            xy = (E[1][:, :, None] * E[0][:, None, :]).reshape(E[0].shape[0], -1)
            t = (x.reshape(-1, n[0] * n[1]) @ xy.T.contiguous()).reshape(x.shape[0], n[2], -1)
            out[:, sl] = (t * E[2].T[None]).sum(1)
    return out


def _nudft_seconds(case, channels, n, M):
    return 8.0 * channels * math.prod(n) * M / 2.5e13


def _kernel64(N, trj, U, mask=None):
    """Packed 64-bit kernel (Nkm, P) on its mask, and the 0-based mask."""
    n = tuple(2 * v for v in N)
    K = U.shape[0]
    kc = trj.reshape(-1, trj.shape[-1])
    frame = torch.arange(trj.shape[0], device=DEV).repeat_interleave(trj.shape[1])
    if mask is not None:
        kc, frame = kc[mask.reshape(-1)], frame[mask.reshape(-1)]
    U64 = U.to(torch.complex128)
    pairs = [(j, k) for k in range(K) for j in range(k + 1)]
    gram = torch.stack([U64[j].conj() * U64[k] for j, k in pairs])
    p = _sum_to_grid(kc, lambda sl: gram[:, frame[sl]], n, centred=False)
    lam = torch.fft.fftn(p, dim=tuple(range(1, len(n) + 1))).reshape(len(pairs), -1)
    km = _mask_cells(kc, n)
    lam = lam[:, km].T.contiguous()
    return (lam if U.is_complex() else lam.real.contiguous()), km


def _backproject64(N, trj, data, U, maps, mask=None, dcf="none"):
    kc = trj.reshape(-1, trj.shape[-1])
    frame = torch.arange(trj.shape[0], device=DEV).repeat_interleave(trj.shape[1])
    y = data.reshape(data.shape[0], -1)
    if mask is not None:
        m = mask.reshape(-1)
        kc, frame, y = kc[m], frame[m], y[:, m]
    w = None
    if dcf != "none":
        w = (kc.double() ** 2).sum(1)
        w = w if dcf == "radial_3D" else w.sqrt()
    Uc = U.to(torch.complex128).conj()
    C, K = y.shape[0], U.shape[0]

    def v(sl):
        yy = y[:, sl].to(torch.complex128)
        if w is not None:
            yy = yy * w[sl]
        return (yy[:, None] * Uc[:, frame[sl]][None]).reshape(C * K, -1)

    img = _sum_to_grid(kc, v, N).reshape((C, K) + N[::-1])
    if maps is None:
        return img
    return (maps.to(torch.complex128).conj()[:, None] * img).sum(0)


def _cart_cells(trj, N):
    q = torch.zeros(trj.shape[:-1], dtype=torch.int64, device=DEV)
    stride = 1
    for a, n in enumerate(N):
        q += torch.remainder(trj[..., a].to(torch.int64) - n // 2 - 1, n) * stride
        stride *= n
    return q


def exact(case, seed):
    kind, N = case["kind"], _shape(case)
    d = len(N)
    M = case["nt"] * case.get("spokes", 1) * case.get("nr", 1)
    if kind in ("backproject", "forward") and _nudft_seconds(case, case["coils"] * case["K"], N, M) > 16.0:
        return None
    if kind == "build" and _nudft_seconds(case, case["K"] * (case["K"] + 1) // 2, [2 * v for v in N], M) > 16.0:
        return None
    s = _inputs(case, seed)
    if kind in ("apply", "cg"):
        dense = _dense(case, s)
        if kind == "apply":
            return _apply64(N, dense, s["maps"], s["b"]).reshape(-1)
        b = s["b"].to(torch.complex128)
        return _cg64(lambda u: _apply64(N, dense, s["maps"], u), b, case["iters"]).reshape(-1)
    if kind == "backproject":
        return _backproject64(N, s["trj"], s["data"], s["U"], s["maps"], s["mask"], case["dcf"])
    if kind == "forward":
        kc = s["trj"].reshape(-1, d)
        frame = torch.arange(case["nt"], device=DEV).repeat_interleave(s["trj"].shape[1])
        U64 = s["U"].to(torch.complex128)[:, frame]
        y = torch.empty((case["coils"], kc.shape[0]), dtype=torch.complex128, device=DEV)
        for c in range(case["coils"]):
            x = s["maps"][c].to(torch.complex128) * s["x"].to(torch.complex128)
            y[c] = (_sum_at_samples(kc, x) * U64).sum(0)
        return y.reshape((case["coils"],) + tuple(s["trj"].shape[:2]))
    if kind == "build":
        lam, km = _kernel64(N, s["trj"], s["U"])
        return lam, km + 1
    if kind == "cartesian":
        q = _cart_cells(s["trj"], N)
        K, V = case["K"], math.prod(N)
        U64 = s["U"].to(torch.complex128)
        frame = torch.arange(case["nt"], device=DEV)[:, None].expand_as(q).reshape(-1)
        q = q.reshape(-1)
        dense = torch.zeros((K * (K + 1) // 2, V), dtype=torch.complex128, device=DEV)
        for k in range(K):
            for j in range(k + 1):
                dense[j + k * (k + 1) // 2].index_add_(0, q, (U64[j].conj() * U64[k])[frame])
        b = torch.zeros((K,) + N[::-1], dtype=torch.complex128, device=DEV)
        axes = tuple(range(-d, 0))
        for c in range(case["coils"]):
            y = s["data"][c].reshape(-1).to(torch.complex128)
            for k in range(K):
                g = torch.zeros(V, dtype=torch.complex128, device=DEV)
                g.index_add_(0, q, y * U64[k].conj()[frame])
                b[k] += s["maps"][c].conj() * torch.fft.fftshift(torch.fft.ifftn(g.reshape(N[::-1]), dim=axes), dim=axes)
        x = _cg64(lambda u: _apply64(N, dense, s["maps"], u, double=False), b, case["iters"])
        return b, x.reshape(-1)
    # calibrate: region, one K = 1 solve per coil, centred transform
    q = max(N) // 32
    calib = tuple(_smooth_up(v // q) for v in N)
    scale = torch.tensor([np.float32(a / b) for a, b in zip(N, calib)], device=DEV)
    trj = s["trj"] * scale
    mask = ((s["trj"].abs() * scale) < 0.5).all(-1)
    one = torch.ones((1, case["nt"]), dtype=torch.float32, device=DEV)
    lam, km = _kernel64(calib, trj, one, mask)
    dense = torch.zeros((1, math.prod(2 * v for v in calib)), dtype=torch.float64, device=DEV)
    dense[:, km] = lam.T
    b = _backproject64(calib, trj, s["data"], one, None, mask)[:, 0]
    x = torch.stack([_cg64(lambda u: _apply64(calib, dense, None, u), b[c][None], case["iters"])[0]
                     for c in range(b.shape[0])])
    axes = tuple(range(-d, 0))
    kbp = torch.fft.fftshift(torch.fft.fftn(torch.fft.fftshift(x, dim=axes), dim=axes), dim=axes)
    return x, kbp
