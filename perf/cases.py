"""Timed cases of the reconstruction engine: the operators and short solves a
reconstruction program calls, through the C ABI with operands in HBM.

listed() names the cases, draw() gives more of the same ranges, prepare()
makes what a program holds before the call, run() is one call, work() the
bytes and operations it cannot do without and exact() its result in 64 bits
(plain torch).

Geometry: variable-density spirals (kx, ky in cycles/FOV, J interleaves x S
samples, turned by a seeded angle), stacks of them in 3D, smooth field maps
from Gaussian blobs, smooth ring-array coil sensitivities with unit sum of
squares, k-space data from the analytic Fourier transform of seeded ellipses
(the coils' phase and position vary) plus noise 40 dB below it.
"""
from __future__ import annotations

import ctypes as C
import math
import random
import sys
from pathlib import Path

import numpy as np
import torch

sys.path.insert(0, str(Path(__file__).resolve().parent.parent / "impatient-mri_amd"))

from impatient._lib import Context, NudftJob, call  # noqa: E402

DEV = "cuda"
F32, F64, C128 = torch.float32, torch.float64, torch.complex128
_ctx = None


def ctx():
    """The program's one context (stream and workspaces)."""
    global _ctx
    if _ctx is None:
        _ctx = Context(0)
    return _ctx


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # the smallest call: adjoint of one 64^2 single-coil slice (8 x 1024 spiral)
        dict(name="fhd_64_1coil", kind="fhd", Ny=64, Nx=64, Nz=1, coils=1, J=8, S=1024,
             t_ms=5.0, hz=100.0),
        # 3D stack of spirals, 4 coils: the partition-separable adjoint
        dict(name="fhd_64x64x16_4coil", kind="fhd", Ny=64, Nx=64, Nz=16, coils=4, J=8, S=1024,
             t_ms=5.0, hz=100.0),
        # ragged sizes: a cropped matrix and an interleave count and length that
        # divide nothing
        dict(name="fhd_250x234_8coil", kind="fhd", Ny=250, Nx=234, Nz=1, coils=8, J=31, S=4093,
             t_ms=8.0, hz=150.0),
        # the largest 2D adjoint: 512^2, 32 coils, 48 x 8192 spiral (once per
        # reconstruction, and the benchmark's step)
        dict(name="fhd_512_32coil", kind="fhd", Ny=512, Nx=512, Nz=1, coils=32, J=48, S=8192,
             t_ms=10.0, hz=200.0),
        # adjoints of a slice series of uneven sizes in one batched call
        dict(name="fhd_slices_8coil", kind="batch", sizes="128,128,256,256,384,384", coils=8,
             t_ms=8.0, hz=150.0),
        # forward operator (simulation, and each brute-force iteration)
        dict(name="forward_256_8coil", kind="forward", Ny=256, Nx=256, Nz=1, coils=8, J=32,
             S=4096, t_ms=8.0, hz=150.0),
        # Toeplitz kernels of a trajectory: once per trajectory, L + 1 planes
        dict(name="q_512", kind="q", Ny=512, Nx=512, J=48, S=8192, t_ms=10.0, L=10),
        # the normal operator, applied once per CG iteration: 2D many coils, 3D
        dict(name="apply_512_32coil", kind="apply", Ny=512, Nx=512, Nz=1, coils=32, J=48, S=8192,
             t_ms=10.0, hz=200.0, L=10),
        dict(name="apply_256x256x32_4coil", kind="apply", Ny=256, Nx=256, Nz=32, coils=4, J=32,
             S=4096, t_ms=8.0, hz=150.0, L=8),
        # a few CG iterations on a small slice (one pass of a TV or restart
        # loop): many short kernels and the host loop
        dict(name="cg_128_8coil", kind="cg", Ny=128, Nx=128, Nz=1, coils=8, J=16, S=2048,
             t_ms=8.0, hz=150.0, L=8, iters=3),
        # the gridding estimate of the adjoint (the solver's -toeplitzGridding)
        dict(name="fhd_gridding_512_32coil", kind="grid", Ny=512, Nx=512, Nz=1, coils=32, J=48,
             S=8192, t_ms=10.0, hz=200.0, L=10, os=1.375),
        # brute-force CG on the small single-coil slice: forward and adjoint
        # in turn with a host loop
        dict(name="bruteforce_64_1coil", kind="bforce", Ny=64, Nx=64, Nz=1, coils=1, J=8, S=1024,
             t_ms=5.0, hz=100.0, cg_num=4),
    ]


# image sizes whose 2x grids the Toeplitz passes transform (2^k and 3 2^k)
_FFT_SIZES = (32, 48, 64, 96, 128, 192, 256, 384, 512)


def _log(rng, a, b):
    return int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))


def _traj(rng, N):
    """Interleaves and samples for about N^2 U(0.7, 1.5) samples."""
    S = _log(rng, 12 * N ** 0.9, 20 * N)
    J = max(2, round(N * N * rng.uniform(0.7, 1.5) / S))
    return J, S


def draw(rng: random.Random):
    kind = rng.choice(["fhd", "fhd", "fhd", "fhd3", "batch", "forward", "q", "apply", "apply3",
                       "cg", "grid", "bforce"])
    hz, t_ms = round(rng.uniform(50, 220), 1), round(rng.uniform(4, 11), 2)
    if kind in ("fhd", "forward"):
        Ny = _log(rng, 48, 480 if kind == "fhd" else 320)
        Nx = max(32, int(Ny * rng.uniform(0.8, 1.0)))
        J, S = _traj(rng, Ny)
        return dict(kind=kind, Ny=Ny, Nx=Nx, Nz=1, coils=_log(rng, 1, 32), J=J, S=S, t_ms=t_ms,
                    hz=hz)
    if kind == "fhd3":
        N = _log(rng, 32, 96)
        J, S = _traj(rng, N)
        return dict(kind="fhd", Ny=N, Nx=N, Nz=2 * _log(rng, 4, 16), coils=_log(rng, 1, 8), J=J,
                    S=S, t_ms=t_ms, hz=hz)
    if kind == "batch":
        sizes = [_log(rng, 64, 384) for _ in range(rng.randint(2, 5))]
        return dict(kind="batch", sizes=",".join(map(str, sizes)), coils=rng.randint(3, 16),
                    t_ms=t_ms, hz=hz)
    if kind == "q":
        Ny = _log(rng, 48, 480)
        J, S = _traj(rng, Ny)
        return dict(kind="q", Ny=Ny, Nx=max(32, int(Ny * rng.uniform(0.8, 1.0))), J=J, S=S,
                    t_ms=t_ms, L=rng.randint(3, 12))
    if kind in ("apply", "cg"):
        Ny = rng.choice(_FFT_SIZES)
        J, S = _traj(rng, Ny)
        c = dict(kind=kind, Ny=Ny, Nx=rng.choice([Ny, Ny, max(32, Ny // 2)]), Nz=1,
                 coils=_log(rng, 1, 32), J=J, S=S, t_ms=t_ms, hz=hz, L=rng.randint(3, 10))
        return dict(c, iters=3) if kind == "cg" else c
    if kind == "apply3":
        N = rng.choice((32, 48, 64, 96, 128, 192))
        J, S = _traj(rng, N)
        return dict(kind="apply", Ny=N, Nx=N, Nz=rng.choice((8, 16, 32)), coils=_log(rng, 1, 8),
                    J=J, S=S, t_ms=t_ms, hz=hz, L=rng.randint(3, 8))
    if kind == "grid":
        N = 2 * _log(rng, 32, 240)
        J, S = _traj(rng, N)
        return dict(kind="grid", Ny=N, Nx=N, Nz=1, coils=_log(rng, 1, 32), J=J, S=S, t_ms=t_ms,
                    hz=hz, L=rng.randint(3, 10), os=rng.choice([1.25, 1.375, 1.5, 2.0]))
    N = _log(rng, 32, 96)
    J, S = _traj(rng, N)
    return dict(kind="bforce", Ny=N, Nx=N, Nz=1, coils=_log(rng, 1, 8), J=J, S=S, t_ms=t_ms,
                hz=hz, cg_num=4)


# --------------------------------------------------------------------- inputs
def _f32(a):
    return a.to(F32).reshape(-1).contiguous()


def _coords(Ny, Nx, Nz):
    """Voxel positions in FOV units, image index (y Nx + x) Nz + z."""
    ax = [(torch.arange(n, dtype=F64, device=DEV) - n // 2) / n for n in (Ny, Nx, Nz)]
    Y, X, Z = torch.meshgrid(*ax, indexing="ij")
    return X.reshape(-1), Y.reshape(-1), (Z.reshape(-1) if Nz > 1 else None)


def _spiral(rs, Ny, Nx, Nz, J, S, t_ms):
    tau = torch.arange(S, dtype=F64, device=DEV) / S
    r = (0.5 - 5e-7) * tau ** 1.5
    turns = max(Ny, Nx) / (2 * J)
    j = torch.arange(J, dtype=F64, device=DEV)[:, None]
    th = 2 * math.pi * (turns * tau[None] + j / J + rs.uniform())
    # real gradients leave the trajectory a little off centre
    kx = (Nx * r * torch.cos(th)).reshape(-1) + rs.uniform(0.2, 0.5)
    ky = (Ny * r * torch.sin(th)).reshape(-1) - rs.uniform(0.2, 0.5)
    t = (tau * t_ms * 1e-3).repeat(J)
    if Nz == 1:
        return _f32(kx), _f32(ky), None, _f32(t)
    kz = torch.arange(-(Nz // 2), Nz - Nz // 2, dtype=F64, device=DEV)
    return (_f32(kx.repeat(Nz)), _f32(ky.repeat(Nz)), _f32(kz.repeat_interleave(len(kx))),
            _f32(t.repeat(Nz)))


def _field(rs, X, Y, hz):
    f = torch.zeros_like(X)
    for _ in range(4):
        cx, cy = rs.uniform(-0.35, 0.35, 2)
        a = rs.choice([-1.0, 1.0]) * rs.uniform(0.5, 1.0)
        f += a * torch.exp(-((X - cx) ** 2 + (Y - cy) ** 2) / (2 * rs.uniform(0.08, 0.25) ** 2))
    return _f32(f * (2 * math.pi * hz) / f.abs().max())


def _sens(rs, X, Y, n):
    """Re and Im [n * N] of the coil maps; None for a single coil (S = 1)."""
    if n == 1:
        return None, None
    a = 2 * math.pi * (torch.arange(n, dtype=F64, device=DEV) / n + rs.uniform())
    d2 = (X[None] - 0.45 * torch.cos(a)[:, None]) ** 2 + (Y[None] - 0.45 * torch.sin(a)[:, None]) ** 2
    m = torch.exp(-d2 / (2 * 0.4 ** 2))
    m /= m.square().sum(0, keepdim=True).sqrt()
    ph = torch.from_numpy(rs.uniform(0, 2 * math.pi, n)).to(DEV)[:, None] + 0.5 * X[None] - Y[None]
    return _f32(m * torch.cos(ph)), _f32(m * torch.sin(ph))


def _ellipses(rs):
    return [(1.0, 0.34, 0.44, 0.0, 0.0)] + [
        (rs.uniform(-0.3, 0.4), *rs.uniform(0.03, 0.12, 2), *rs.uniform(-0.2, 0.2, 2))
        for _ in range(7)]


def _image(rs, X, Y, Z):
    v = torch.zeros_like(X)
    for A, a, b, x, y in _ellipses(rs):
        q = ((X - x) / a) ** 2 + ((Y - y) / b) ** 2
        v += A * ((q if Z is None else q + (Z / 0.45) ** 2) <= 1)
    ph = rs.uniform(-1, 1, 2)
    ph = ph[0] * X + ph[1] * Y
    return _f32(v * torch.cos(ph)), _f32(v * torch.sin(ph))


def _data(rs, seed, kx, ky, kz, n, nvox):
    """k-space data [n * M]: ellipse spectra, shifted and turned per coil, plus noise."""
    kx, ky = kx.double(), ky.double()
    out = torch.zeros(n, len(kx), dtype=C128, device=DEV)
    base = torch.zeros(len(kx), dtype=C128, device=DEV)
    for A, a, b, x, y in _ellipses(rs):
        q = (2 * math.pi * torch.sqrt((a * kx) ** 2 + (b * ky) ** 2)).clamp_min(1e-6)
        base += torch.polar(2 * A * math.pi * a * b * torch.special.bessel_j1(q) / q,
                            -2 * math.pi * (kx * x + ky * y))
    if kz is not None:
        base = base * torch.exp(-0.5 * (kz.double() / 2) ** 2)
    for c in range(n):
        sx, sy = rs.uniform(-0.05, 0.05, 2)
        out[c] = base * torch.polar(torch.full_like(kx, rs.uniform(0.5, 1.0)),
                                    rs.uniform(0, 6.28) - 2 * math.pi * (kx * sx + ky * sy))
    out *= nvox
    g = torch.Generator(device=DEV).manual_seed(int(seed) + 17)
    noise = torch.randn(2, *out.shape, dtype=F64, device=DEV, generator=g)
    out += 0.01 / math.sqrt(2) * out.abs().square().mean().sqrt() * torch.complex(noise[0], noise[1])
    return _f32(out.real), _f32(out.imag)


def _problem(case, seed, what):
    """Named float32 tensors on the GPU."""
    rs = np.random.RandomState(int(seed) % (1 << 32))
    Ny, Nx, Nz, n = case["Ny"], case["Nx"], case.get("Nz", 1), case.get("coils", 1)
    p = dict(zip(("kx", "ky", "kz", "t"), _spiral(rs, Ny, Nx, Nz, case["J"], case["S"],
                                                  case["t_ms"])))
    X, Y, Z = _coords(Ny, Nx, Nz)
    p["x"], p["y"], p["z"] = _f32(X), _f32(Y), None if Z is None else _f32(Z)
    if "hz" in case:
        p["fm"] = _field(rs, X, Y, case["hz"])
        p["sr"], p["si"] = _sens(rs, X, Y, n)
    if "data" in what:
        p["dr"], p["di"] = _data(rs, seed, p["kx"], p["ky"], p["kz"], n, len(X))
    if "image" in what:
        p["ir"], p["ii"] = _image(rs, X, Y, Z)
    return p


def _seg(t, L):
    """tau and t0 in float32, as the solver's files carry them."""
    t0, t1 = np.float32(t[0].item()), np.float32(t[-1].item())
    return float(np.float32((t1 - t0) / np.float32(L))), float(t0)


# ------------------------------------------------------------ prepare and run
def _p(a, elems=0):
    return C.c_void_p(0 if a is None else a.data_ptr() + 4 * elems)


def _i(*v):
    return [C.c_int(int(x)) for x in v]


def _out(n):
    return torch.zeros(n, dtype=F32, device=DEV), torch.zeros(n, dtype=F32, device=DEV)


class _Plan:
    """A Toeplitz plan, destroyed with the state that holds it."""

    def __init__(self, c, p):
        Ny, Nx, Nz, L = c["Ny"], c["Nx"], c["Nz"], c["L"]
        self.h = C.c_void_p()
        nq = 4 * Ny * Nx * (2 * Nz if Nz > 1 else 1)
        qr, qi = _out((L + 1) * nq)
        tau, t0 = _seg(p["t"], L)
        torch.cuda.synchronize()
        call("imp_toeplitz_q", ctx().h, *_i(len(p["kx"])), _p(p["kx"]), _p(p["ky"]), _p(p["kz"]),
             _p(p["t"]), None, None, *_i(Nx, Ny, Nz, nq), None, None, None, *_i(L, 0), _p(qr),
             _p(qi))
        call("imp_toep_create", ctx().h, *_i(Ny, Nx, Nz, c["coils"], L), C.c_float(tau),
             C.c_float(t0), _p(qr), _p(qi), _p(p["fm"]), _p(p["sr"]), _p(p["si"]),
             C.c_float(LAMBDA), C.byref(self.h))
        ctx().synchronize()

    def __del__(self):
        if self.h:
            call("imp_toep_destroy", self.h)


LAMBDA = 1e-3


def _slice_cases(case):
    """The 2D problems of a batch: N x N, a spiral scaled with N."""
    out = []
    for N in (int(v) for v in case["sizes"].split(",")):
        J, S = max(2, N // 8 if N <= 256 else 40), 16 * N
        out.append(dict(Ny=N, Nx=N, Nz=1, coils=case["coils"], J=J, S=S, t_ms=case["t_ms"],
                        hz=case["hz"]))
    return out


def prepare(case, seed):
    k = case["kind"]
    if k == "batch":
        ps = [_problem(c, seed + 101 * i, "data") for i, c in enumerate(_slice_cases(case))]
        jobs = (NudftJob * len(ps))()
        outs = []
        for J, p in zip(jobs, ps):
            o = _out(len(p["x"]))
            outs.append(o)
            J.num_k, J.num_x, J.ncoils = len(p["kx"]), len(p["x"]), case["coils"]
            for f, v in (("kx", "kx"), ("ky", "ky"), ("t", "t"), ("x", "x"), ("y", "y"),
                         ("fm", "fm"), ("d_r", "dr"), ("d_i", "di"), ("s_r", "sr"), ("s_i", "si")):
                setattr(J, f, p[v].data_ptr())
            J.out_r, J.out_i = o[0].data_ptr(), o[1].data_ptr()
        s = dict(case=case, ps=ps, jobs=jobs, out=outs)
    else:
        p = _problem(case, seed, {"fhd": "data", "grid": "data", "bforce": "data", "cg": "image",
                                  "forward": "image", "apply": "image", "q": ""}[k])
        n = len(p["x"])
        if k == "forward":
            o = _out(case["coils"] * len(p["kx"]))
        elif k == "q":
            o = _out((case["L"] + 1) * 4 * n)
        else:
            o = _out(n)
        s = dict(case=case, p=p, out=o)
        if k in ("apply", "cg"):
            s["plan"] = _Plan(case, p)
    ctx()
    torch.cuda.synchronize()
    return s


def run(s):
    c, k, h, o = s["case"], s["case"]["kind"], ctx().h, s["out"]
    if k == "batch":
        call("imp_nudft_adjoint_batch", h, C.c_int(len(s["jobs"])), s["jobs"], C.c_int(0))
        return o
    p = s["p"]
    nk, nx = len(p["kx"]), len(p["x"])
    if k == "fhd":
        call("imp_nudft_adjoint", h, *_i(nk, nx, c["coils"]), _p(p["kx"]), _p(p["ky"]),
             _p(p["kz"]), _p(p["t"]), _p(p["x"]), _p(p["y"]), _p(p["z"]), _p(p["fm"]), None, None,
             _p(p["dr"]), _p(p["di"]), _p(p["sr"]), _p(p["si"]), _p(o[0]), _p(o[1]))
    elif k == "forward":
        call("imp_nudft_forward", h, *_i(nk, nx, c["coils"]), _p(p["kx"]), _p(p["ky"]),
             _p(p["kz"]), _p(p["t"]), _p(p["x"]), _p(p["y"]), _p(p["z"]), _p(p["fm"]),
             _p(p["ir"]), _p(p["ii"]), _p(p["sr"]), _p(p["si"]), _p(o[0]), _p(o[1]))
    elif k == "q":
        call("imp_toeplitz_q", h, *_i(nk), _p(p["kx"]), _p(p["ky"]), None, _p(p["t"]), None, None,
             *_i(c["Nx"], c["Ny"], 1, 4 * nx), None, None, None, *_i(c["L"], 0), _p(o[0]), _p(o[1]))
    elif k == "apply":
        call("imp_toep_apply", s["plan"].h, _p(p["ir"]), _p(p["ii"]), _p(o[0]), _p(o[1]))
    elif k == "cg":
        # the image stands for F^H d: any right-hand side takes the same path
        call("imp_toep_cg", s["plan"].h, _p(p["ir"]), _p(p["ii"]), _p(o[0]), _p(o[1]),
             C.c_int(c["iters"]), C.c_double(0.0), C.c_int(1), None)
    elif k == "grid":
        call("imp_fhd_gridding", h, *_i(nk, c["coils"]), _p(p["kx"]), _p(p["ky"]), None,
             _p(p["t"]), *_i(c["Nx"], c["Ny"], 1), _p(p["fm"]), _p(p["dr"]), _p(p["di"]),
             _p(p["sr"]), _p(p["si"]), C.c_int(c["L"]), C.c_float(c["os"]), _p(o[0]), _p(o[1]))
    elif k == "bforce":
        # from the zero image, as the solver starts
        for v in o:
            call("imp_memset_d", h, _p(v), C.c_int(0), C.c_size_t(4 * nx))
        call("imp_bruteforce_cg", h, *_i(nk, nx, c["coils"]), _p(p["kx"]), _p(p["ky"]),
             _p(p["t"]), _p(p["x"]), _p(p["y"]), _p(p["fm"]), _p(p["dr"]), _p(p["di"]),
             _p(p["sr"]), _p(p["si"]), C.c_int(c["cg_num"]), C.c_float(LAMBDA), _p(o[0]), _p(o[1]))
    return o


# ----------------------------------------------------------------------- work
def work(case):
    """Operands read once, results written once.  Operations: the transforms
    of every segment and coil for the Toeplitz operator, the KB window for
    gridding, and for the NUDFTs one oversampled transform and a 10-point
    window per axis (a sum over all pairs is one way to evaluate them, not
    what they need)."""
    k = case["kind"]
    if k == "batch":
        w = [work(dict(c, kind="fhd")) for c in _slice_cases(case)]
        return {n: sum(v[n] for v in w) for n in ("bytes", "flops")}
    Ny, Nx, Nz, n = case["Ny"], case["Nx"], case.get("Nz", 1), case.get("coils", 1)
    vox, nk = Ny * Nx * Nz, case["J"] * case["S"] * Nz
    fft = lambda pts: 5.0 * pts * math.log2(pts)  # noqa: E731
    sens = 8 * n * vox if n > 1 else 0
    geo = 4 * (3 + (Nz > 1)) * (nk + vox)
    if k in ("fhd", "forward", "bforce"):
        its = 2 * case["cg_num"] - 1 if k == "bforce" else 1
        by = geo + sens + 8 * n * nk + 8 * vox
        fl = n * (4.0 * 100 * nk + 4 * fft(2 * Ny * Nx) * Nz) + 8.0 * n * vox
        return {"bytes": by + (its - 1) * 8 * (n * nk + vox), "flops": its * fl}
    if k == "grid":
        return {"bytes": 12 * nk + 8 * n * nk + sens + 12 * vox,
                "flops": n * (2 * 4.0 * 30 * nk + (case["L"] + 1) * fft(case["os"] ** 2 * vox))}
    L1 = case["L"] + 1
    if k == "q":
        return {"bytes": 12 * nk + 8 * L1 * 4 * vox,
                "flops": 2 * 4.0 * 100 * nk + L1 * fft(8 * vox)}
    grid = (8 if Nz > 1 else 4) * vox
    fl = n * L1 * (2 * fft(grid) + 2.0 * grid + 12 * vox)
    by = 4 * L1 * grid + sens + 4 * vox + 16 * vox
    its = case.get("iters", 1)
    return {"bytes": its * by, "flops": its * fl}


# ---------------------------------------------------------------------- exact
def _cx(r, i, n):
    return None if r is None else torch.complex(r.double(), i.double()).reshape(n, -1)


def _ph(p, rows, cols):
    """Phase in revolutions [voxel rows, sample cols]."""
    u = p["x"][rows, None].double() * p["kx"][None, cols].double()
    u.addr_(p["y"][rows].double(), p["ky"][cols].double())
    if p["z"] is not None:
        u.addr_(p["z"][rows].double(), p["kz"][cols].double())
    u.addr_(p["fm"][rows].double() / (2 * math.pi), p["t"][cols].double())
    return u


def _blocks(n, size):
    return [slice(a, min(n, a + size)) for a in range(0, n, size)]


def _adjoint(p, d, S):
    """[N] from data [C, M] and maps [C, N] or None."""
    nx, nk = len(p["x"]), d.shape[1]
    out = torch.empty(nx, dtype=C128, device=DEV)
    W = d.T.contiguous()
    for r in _blocks(nx, 8192):
        acc = 0
        for k in _blocks(nk, 32768):
            u = _ph(p, r, k).mul_(2 * math.pi)
            acc = acc + torch.polar(torch.ones_like(u), u) @ W[k]
        out[r] = acc.sum(1) if S is None else (acc * S[:, r].T.conj()).sum(1)
    return out


def _forward(p, img, S, n):
    nx, nk = len(p["x"]), len(p["kx"])
    V = (img.reshape(1, -1).expand(n, -1) if S is None else S * img.reshape(1, -1)).T.contiguous()
    out = torch.zeros(n, nk, dtype=C128, device=DEV)
    for k in _blocks(nk, 32768):
        for r in _blocks(nx, 8192):
            u = _ph(p, r, k).mul_(-2 * math.pi)
            out[:, k] += (torch.polar(torch.ones_like(u), u).T.contiguous() @ V[r]).T
    return out


def _hann(t, tau, l, t0):
    a = t.double() - tau * l - t0
    return torch.where(a.abs() < tau, 0.5 + 0.5 * torch.cos(math.pi * a / tau), 0.0)


def _q2d(kx, ky, t, Ny, Nx, L):
    """[L + 1, 2Ny, 2Nx] on the standard grid: sums over rows times columns."""
    tau, t0 = _seg(t, L)
    gx = torch.arange(-Nx, Nx, dtype=F64, device=DEV) / Nx
    gy = torch.arange(-Ny, Ny, dtype=F64, device=DEV) / Ny
    out = torch.zeros(L + 1, 2 * Ny, 2 * Nx, dtype=C128, device=DEV)
    for l in range(L + 1):
        a = _hann(t, tau, l, t0)
        k = torch.nonzero(a).reshape(-1)
        for b in _blocks(len(k), 65536):
            j = k[b]
            uy, ux = 2 * math.pi * gy[:, None] * ky[j].double(), 2 * math.pi * kx[j, None].double() * gx
            out[l] += torch.polar(a[j][None].expand_as(uy).contiguous(), uy) @ torch.polar(torch.ones_like(ux), ux)
    return out


def _operator(case, p):
    """v [N] -> A v in complex128."""
    Ny, Nx, Nz, L, n = case["Ny"], case["Nx"], case["Nz"], case["L"], case["coils"]
    m = case["J"] * case["S"]
    q = _q2d(p["kx"][:m], p["ky"][:m], p["t"][:m], Ny, Nx, L)
    N, ax = ((Ny, Nx), (0, 1)) if Nz == 1 else ((Ny, Nx, Nz), (0, 1, 2))
    if Nz > 1:
        gz = torch.arange(-Nz, Nz, dtype=F64, device=DEV) / Nz
        u = 2 * math.pi * gz[None] * p["kz"][::m, None].double()
        q = q[..., None] * torch.polar(torch.ones_like(u), u).sum(0)
    qf = [torch.fft.fftn(torch.fft.ifftshift(v)) for v in q]
    del q
    tau, t0 = _seg(p["t"], L)
    fm = p["fm"].double().reshape(N)
    S = _cx(p["sr"], p["si"], n)
    M, crop = tuple(2 * v for v in N), tuple(slice(0, v) for v in N)
    ph = [torch.polar(torch.ones_like(fm), fm * (tau * l + t0)) for l in range(L + 1)]

    def apply(v):
        v = v.reshape(N)
        out = torch.zeros_like(v)
        for c in range(n):
            sv = v if S is None else S[c].reshape(N) * v
            acc = torch.zeros_like(v)
            for l in range(L + 1):
                w = torch.fft.ifftn(torch.fft.fftn(ph[l].conj() * sv, s=M, dim=ax) * qf[l])
                acc += ph[l] * w[crop]
            out += acc if S is None else S[c].reshape(N).conj() * acc
        for d in range(len(N)):
            t = v - v.roll(-1, d)
            out += LAMBDA32 * (t - t.roll(1, d))
        return out.reshape(-1)
    return apply


LAMBDA32 = float(np.float32(LAMBDA))


def _dot(a, b):
    return torch.vdot(a, b).real.item()


def _kb(case, n):
    """Grid size, rounded oversampling and Beatty's beta of one axis (width 4)."""
    f = np.float32
    os = float(f(f(2) * f(np.ceil(f(f(case["os"]) * f(case["Nx"])) / f(2))) / f(case["Nx"])))
    g = int(np.ceil(f(f(os) * f(n))))
    return g + g % 2, os, math.pi * math.sqrt((os - 0.5) ** 2 * 64.0 / os ** 2 - 0.8)


def _window(k, n, G, os, beta):
    s = os * (k.double() + n / 2.0)
    g = s.floor()[:, None] + torch.arange(-4, 6, dtype=F64, device=DEV)
    d = (s[:, None] - g).abs() / os
    ok = (g >= 0) & (g < G) & (d <= 2)
    w = torch.special.i0(beta * (1 - (d / 2) ** 2).clamp_min(0).sqrt()) / 4
    return torch.where(ok, g, 0.0).long(), torch.where(ok, w, 0.0)


def _gridding(case, p):
    Ny, Nx, n, L = case["Ny"], case["Nx"], case["coils"], case["L"]
    tau, t0 = _seg(p["t"], L)
    ax = []
    for k, N in ((p["ky"], Ny), (p["kx"], Nx)):
        G, os, beta = _kb(case, N)
        i, w = _window(k, N, G, os, beta)
        e = beta ** 2 - (math.pi * 4 * (torch.arange(N, dtype=F64, device=DEV) - N // 2) / N) ** 2
        s = e.abs().sqrt()
        ax.append((G, os, i, w, torch.where(e > 0, torch.sinh(s), torch.sin(s)) / s))
    (Gy, oy, iy, wy, cy), (Gx, ox, ix, wx, cx) = ax
    d, S = _cx(p["dr"], p["di"], n), _cx(p["sr"], p["si"], n)
    fm = p["fm"].double()
    out = torch.zeros(Ny * Nx, dtype=C128, device=DEV)
    y0, x0 = Gy // 2 - Ny // 2, Gx // 2 - Nx // 2
    for l in range(L + 1):
        a = _hann(p["t"], tau, l, t0)
        j = torch.nonzero(a).reshape(-1)
        g = torch.zeros(Gy * Gx, n, 2, dtype=F64, device=DEV)
        for b in _blocks(len(j), 16384):
            jj = j[b]
            v = torch.view_as_real((d[:, jj] * a[jj]).T.contiguous())
            for ty in range(10):
                for tx in range(10):
                    w = wy[jj, ty] * wx[jj, tx]
                    if bool((w != 0).any()):
                        g.index_add_(0, iy[jj, ty] * Gx + ix[jj, tx], v * w[:, None, None])
        im = torch.view_as_complex(g).T.reshape(n, Gy, Gx)
        im = torch.fft.fftshift(torch.fft.ifft2(torch.fft.ifftshift(im, dim=(1, 2)), norm="forward"),
                                dim=(1, 2))[:, y0:y0 + Ny, x0:x0 + Nx]
        im = (im / (cy[:, None] * cx[None] * oy * ox)).reshape(n, -1)
        im = im.sum(0) if S is None else (im * S.conj()).sum(0)
        out += im * torch.polar(torch.ones_like(fm), fm * (t0 + l * tau))
    return out


def _parts(z):
    return z.real.reshape(-1).contiguous(), z.imag.reshape(-1).contiguous()


def exact(case, seed):
    """run()'s outputs in 64 bits."""
    k = case["kind"]
    if k == "batch":
        return [exact(dict(c, kind="fhd"), seed + 101 * i) for i, c in enumerate(_slice_cases(case))]
    n = case.get("coils", 1)
    p = _problem(case, seed, {"fhd": "data", "grid": "data", "bforce": "data", "cg": "image",
                              "forward": "image", "apply": "image", "q": ""}[k])
    S = _cx(p.get("sr"), p.get("si"), n)
    if k == "fhd":
        return _parts(_adjoint(p, _cx(p["dr"], p["di"], n), S))
    if k == "forward":
        return _parts(_forward(p, _cx(p["ir"], p["ii"], 1), S, n))
    if k == "q":
        return _parts(_q2d(p["kx"], p["ky"], p["t"], case["Ny"], case["Nx"], case["L"]))
    if k == "grid":
        return _parts(_gridding(case, p))
    if k in ("apply", "cg"):
        A, v = _operator(case, p), _cx(p["ir"], p["ii"], 1).reshape(-1)
        if k == "apply":
            return _parts(A(v))
        x, r, d = torch.zeros_like(v), v.clone(), v.clone()
        best, xb = _dot(r, r), x
        for _ in range(case["iters"]):
            q = A(d)
            rr = _dot(r, r)
            a = rr / _dot(d, q)
            x, r = x + a * d, r - a * q
            new = _dot(r, r)
            d = r + new / rr * d
            if new < best:
                best, xb = new, x
        return _parts(xb)
    # brute-force CG from zero: the normal equations with the difference term
    N = (case["Ny"], case["Nx"])

    def R(v):
        v = v.reshape(N)
        s = torch.zeros_like(v)
        for d in range(2):
            t = v - v.roll(-1, d)
            s += LAMBDA32 * (t - t.roll(1, d))
        return s.reshape(-1)
    y = _cx(p["dr"], p["di"], n)
    x = torch.zeros(len(p["x"]), dtype=C128, device=DEV)
    Af, d, old = torch.zeros_like(y), None, 0.0
    for _ in range(case["cg_num"] - 1):
        g = _adjoint(p, y - Af, S) - R(x)
        new = _dot(g, g)
        d = g if d is None else g + new / old * d
        old = new
        q = _forward(p, d, S, n)
        a = _dot(d, g) / (_dot(q.reshape(-1), q.reshape(-1)) + _dot(R(d), d))
        Af, x = Af + a * q, x + a * d
    return _parts(x)
