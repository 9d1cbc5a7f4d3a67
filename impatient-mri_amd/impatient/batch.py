"""Batched reconstruction of independent 2D slices of uneven sizes.

The slices (N x N, N in {128, 256, 384} for the 48-slice workload, 8 coils
each, spiral trajectories scaled per matrix size, field maps within
+-150 Hz) go through:

  1. all F^H d in one call (imp_nudft_adjoint_batch: large slices in separable
     form, the others in one persistent MFMA launch);
  2. Q_l once per size class (the trajectory is shared within a class) and a
     Toeplitz plan per slice (field map and coils are per slice);
  3. per slice: the learned warm start (network of the size class, trained
     weights when a model is given) with the zero-start fallback, then
     circulant-preconditioned CG to the tolerance with one HIP graph per
     iteration (IMP_CG_GRAPH); the slices run on several contexts (streams)
     from as many host threads, each keeping one plan per size class.

The schedule knobs (the NUDFT batch's workgroups per CU, and the pass-E
coils per workgroup of each size class) are picked by the Autotuner: it
times each candidate on the first slices of a class with the library's
kernel timer and keeps the fastest.

No counterpart in the reference beyond its per-slice host loop
(main_mri.cu:771-904, one slice after another, each rebuilding everything).
"""
from __future__ import annotations

import ctypes as C
import time
from dataclasses import dataclass

import numpy as np

from . import ops, synth
from ._lib import (CGStats, Context, IMP_CG_BEST_ITERATE, IMP_CG_FALLBACK_ZERO, IMP_CG_GRAPH,
                   IMP_CG_PRECOND, IMP_CG_TRUE_RESIDUAL, IMP_CG_USE_X0, call, ptr)

SIZES = (128, 256, 384)
# samples per interleave x interleaves per matrix size (spiral scaled with N)
TRAJ = {128: (16, 2048), 256: (32, 4096), 384: (40, 6144)}


@dataclass
class Slice:
    prob: synth.Problem
    d: np.ndarray             # [C, M] k-space data


def make_slices(n=48, seed=20260104, coils=8, L=8, max_hz=150.0, snr_db=40.0, ctx=None):
    """Seeded slice set: sizes drawn from SIZES, per-slice phantom draw and
    field map, data from the GPU forward NUDFT + noise."""
    from .learn import random_phantom
    rng = np.random.default_rng(seed)
    sizes = rng.choice(SIZES, n)
    out = []
    for i, N in enumerate(sizes):
        N = int(N)
        J, S = TRAJ[N]
        p = synth.make_problem(f"slice{i}_{N}", N, 1, coils, J, S, 8e-3, max_hz, 5, L,
                               seed + 1000 * N)   # geometry and coils shared per size class
        X = p.x.reshape(N, N).astype(np.float64)
        Y = p.y.reshape(N, N).astype(np.float64)
        r = np.random.default_rng(seed + 17 * i + 1)
        p.rho = random_phantom(r, X, Y).reshape(-1)
        p.fm = synth.field_map(r, X, Y, 5, max_hz).astype(np.float32).reshape(-1)
        d = ops.nudft_forward(ctx, p.kx, p.ky, None, p.t, p.x, p.y, None, p.fm, p.rho, p.sens,
                              coils)
        out.append(Slice(p, synth.add_noise(np.asarray(d).reshape(coils, -1), snr_db, seed + i)))
    return out


class Autotuner:
    """Times schedule candidates with the library kernel timer and keeps the
    fastest per key (size class / batch signature)."""

    def __init__(self, ctx: Context):
        self.ctx = ctx
        self.choice = {}
        self.trials = {}

    def _ms(self, name, fn):
        call("imp_profile_enable", self.ctx.h, C.c_int(1))
        call("imp_profile_reset", self.ctx.h)
        fn()
        tot, n = C.c_double(), C.c_int()
        call("imp_profile_read", self.ctx.h, name.encode(), C.byref(tot), C.byref(n))
        call("imp_profile_enable", self.ctx.h, C.c_int(0))
        return tot.value

    def pick(self, key, candidates, run, kernel):
        """run(candidate) executes one timed instance; returns the choice."""
        if key not in self.choice:
            t = {c: self._ms(kernel, lambda c=c: run(c)) for c in candidates}
            self.trials[key] = t
            self.choice[key] = min(t, key=t.get)
        return self.choice[key]


def _plan(ctx, p, qr, qi):
    L = p.ntime_segs
    t32 = p.t.astype(np.float32)
    tau = float(np.float32((t32[-1] - t32[0]) / np.float32(L)))
    h = C.c_void_p()
    fm = ctx.to_device(np.ascontiguousarray(p.fm, np.float32))
    sr = ctx.to_device(np.ascontiguousarray(p.sens.real.reshape(-1), np.float32))
    si = ctx.to_device(np.ascontiguousarray(p.sens.imag.reshape(-1), np.float32))
    call("imp_toep_create", ctx.h, C.c_int(p.Ny), C.c_int(p.Nx), C.c_int(1), C.c_int(p.ncoils),
         C.c_int(L), C.c_float(tau), C.c_float(float(t32[0])), ptr(qr), ptr(qi), ptr(fm),
         ptr(sr), ptr(si), C.c_float(p.lam), C.byref(h))
    return h, (fm, sr, si)


def reconstruct(ctx: Context, slices, tol=1e-5, max_iter=500, model=None, tuner=None, log=print,
                keep_images=False, streams=3):
    """Batched reconstruction; returns per-slice records and totals
    (keep_images: each record also holds its F^H d "b" and image "x" as
    host arrays, copied after the slice's timing ends)."""
    tuner = tuner or Autotuner(ctx)
    t_all = time.perf_counter()
    # 1. F^H d of every slice in one call (autotuned chunking of its launch of
    # the smaller slices)
    jobs = [dict(kx=s.prob.kx, ky=s.prob.ky, t=s.prob.t, x=s.prob.x, y=s.prob.y, fm=s.prob.fm,
                 d=s.d, sens=s.prob.sens) for s in slices]
    key = ("fhd_batch", tuple(sorted({s.prob.Nx for s in slices})), len(slices))
    scale = tuner.pick(key, (2, 4, 8, 16),
                       lambda c: ops.nudft_adjoint_batch(ctx, jobs, chunk_scale=c),
                       "k_nudft_mfma_batch")
    t0 = time.perf_counter()
    bs = ops.nudft_adjoint_batch(ctx, jobs, chunk_scale=scale)
    ctx.synchronize()
    t_fhd = time.perf_counter() - t0
    # 2. Q_l per size class
    t0 = time.perf_counter()
    classes = {}
    for s in slices:
        N = s.prob.Nx
        if N not in classes:
            qr, qi = ops.toeplitz_q_device(ctx, s.prob.kx, s.prob.ky, s.prob.t, N, N,
                                           s.prob.ntime_segs)
            classes[N] = dict(qr=qr, qi=qi)
    ctx.synchronize()
    t_q = time.perf_counter() - t0
    # 3. per slice: learned start and graph-captured PCG.  Slices run on
    # `streams` contexts (one HIP stream each) from as many host threads, so
    # one slice's small kernels and per-iteration read-back overlap another's
    # work.  Each worker keeps one plan per size class (the trajectory, Q_l
    # and coils are shared within a class; imp_toep_set_fieldmap switches
    # the field map) and preallocated vectors: no device allocation or free
    # (which would synchronise the device) per slice.
    from concurrent.futures import ThreadPoolExecutor
    first = {}
    for i, s in enumerate(slices):
        first.setdefault(s.prob.Nx, i)
    # pass-E schedule of each size class, tuned on the main context (once:
    # the tuner keeps its choice for later batches)
    cpg_of = {}
    for N, i in first.items():
        if ("pass_e", N) in tuner.choice:
            cpg_of[N] = tuner.choice[("pass_e", N)]
            continue
        p = slices[i].prob
        h, keep = _plan(ctx, p, classes[N]["qr"], classes[N]["qi"])
        br, bi = ctx.alloc((p.nvox,)), ctx.alloc((p.nvox,))
        xr, xi = ctx.alloc((p.nvox,)), ctx.alloc((p.nvox,))
        cpg0 = C.c_int()
        call("imp_toep_get_schedule", h, C.byref(cpg0))
        cands = sorted({c for c in (cpg0.value, 2 * cpg0.value, p.ncoils) if c <= p.ncoils})
        cpg_of[N] = tuner.pick(("pass_e", N), cands,
                               lambda c: (call("imp_toep_set_schedule", h, C.c_int(c)),
                                          call("imp_toep_apply", h, ptr(br), ptr(bi), ptr(xr),
                                               ptr(xi))),
                               "toep_pass_e")
        call("imp_toep_destroy", h)
    nw = max(1, min(streams, len(slices)))
    workers = [ctx] + [Context(ctx.device) for _ in range(nw - 1)]
    # every worker's plans, vectors and networks are made here, before the
    # threads start: an allocation or a synchronous copy on one thread while
    # another records its CG graph would invalidate that capture
    wstate = [dict() for _ in workers]
    for i, s in enumerate(slices):
        w, N, p = i % nw, s.prob.Nx, s.prob
        if N in wstate[w]:
            continue
        c = workers[w]
        h, keep = _plan(c, p, classes[N]["qr"], classes[N]["qi"])
        call("imp_toep_set_schedule", h, C.c_int(cpg_of[N]))
        v = {k: c.alloc((p.nvox,)) for k in ("br", "bi", "xr", "xi", "zr", "zi")}
        net = None
        if model is not None:
            net = ops.CNN(c, N, N, seed=1)
            net.set_params(model)
        wstate[w][N] = dict(h=h, keep=keep, fm=c.alloc((p.nvox,)), net=net, **v)
    for c in workers:
        c.synchronize()

    flags0 = IMP_CG_BEST_ITERATE | IMP_CG_TRUE_RESIDUAL | IMP_CG_PRECOND | IMP_CG_GRAPH

    def solve(i):
        w = i % nw
        s, b = slices[i], bs[i]
        p = s.prob
        N = p.Nx
        t0 = time.perf_counter()
        S = wstate[w][N]
        h = S["h"]
        S["fm"].upload(np.ascontiguousarray(p.fm, np.float32))
        call("imp_toep_set_fieldmap", h, ptr(S["fm"]))
        S["br"].upload(np.ascontiguousarray(b.real, np.float32))
        S["bi"].upload(np.ascontiguousarray(b.imag, np.float32))
        flags = flags0
        if S["net"] is not None:
            call("imp_toep_precond_apply", h, ptr(S["br"]), ptr(S["bi"]), ptr(S["zr"]),
                 ptr(S["zi"]))
            S["net"].forward_device(S["zr"], S["zi"], S["xr"], S["xi"])
            flags |= IMP_CG_USE_X0 | IMP_CG_FALLBACK_ZERO
        st = CGStats()
        call("imp_toep_cg", h, ptr(S["br"]), ptr(S["bi"]), ptr(S["xr"]), ptr(S["xi"]),
             C.c_int(max_iter), C.c_double(tol), C.c_int(flags), C.byref(st))
        t_slice = time.perf_counter() - t0
        r = st.as_dict()
        r.update(N=N, slice_s=t_slice, cpg=cpg_of[N], stream=w)
        if keep_images:
            r.update(b=np.asarray(b), x=S["xr"].get() + 1j * S["xi"].get())
        return r

    # slices of one worker run in order on its stream; workers in parallel
    def run_worker(w):
        return [(i, solve(i)) for i in range(w, len(slices), nw)]
    t0 = time.perf_counter()
    with ThreadPoolExecutor(max_workers=nw) as pool:
        parts = list(pool.map(run_worker, range(nw)))
    t_solve = time.perf_counter() - t0
    recs = [r for _, r in sorted((x for part in parts for x in part), key=lambda x: x[0])]
    for w, st_ in enumerate(wstate):
        for S in st_.values():
            call("imp_toep_destroy", S["h"])
            if S["net"] is not None:
                S["net"].close()
    for c in workers[1:]:
        c.close()
    t_total = time.perf_counter() - t_all
    log(f"batch: {len(slices)} slices in {t_total:.3f} s ({len(slices) / t_total:.1f} slices/s); "
        f"F^H d {t_fhd * 1e3:.1f} ms (one call, chunk scale {scale}), Q {t_q * 1e3:.1f} ms, "
        f"solves {t_solve * 1e3:.1f} ms on {nw} streams")
    return dict(slices=recs, total_s=t_total, fhd_s=t_fhd, q_s=t_q, solve_s=t_solve,
                streams=nw, nudft_chunk_scale=scale,
                tuner=dict((str(k), v) for k, v in tuner.trials.items()))


def main(argv=None):
    import argparse
    import json
    ap = argparse.ArgumentParser(description="48-slice batched reconstruction (sizes 128/256/384)")
    ap.add_argument("--slices", type=int, default=48)
    ap.add_argument("--model", default=None, help="trained warm-start model (.npz)")
    ap.add_argument("--tol", type=float, default=1e-5)
    ap.add_argument("--streams", type=int, default=3,
                    help="contexts (HIP streams) the per-slice solves run on")
    ap.add_argument("--repeat", type=int, default=2,
                    help="passes over the batch with one autotuner; the first includes its trials")
    args = ap.parse_args(argv)

    def log(m):
        print(f"[batch] {m}", flush=True)

    ctx = Context(0)
    t0 = time.perf_counter()
    sl = make_slices(args.slices, ctx=ctx)
    log(f"{len(sl)} slices synthesised in {time.perf_counter() - t0:.1f} s")
    params = None
    if args.model:
        from .learn import load_model
        params, _, _ = load_model(args.model)
    tuner = Autotuner(ctx)
    passes = [reconstruct(ctx, sl, tol=args.tol, model=params, tuner=tuner, log=log,
                          streams=args.streams)
              for _ in range(max(1, args.repeat))]
    res = passes[-1]
    recs = res["slices"]
    by = {}
    for r in recs:
        by.setdefault(r["N"], []).append(r)
    summary = {
        "slices": len(recs), "passes": len(passes),
        "first_pass_s": round(passes[0]["total_s"], 4),
        "total_s": round(res["total_s"], 4),
        "slices_per_s": round(len(recs) / res["total_s"], 2),
        "fhd_batch_s": round(res["fhd_s"], 4), "q_s": round(res["q_s"], 4),
        "solve_s": round(res["solve_s"], 4), "streams": res["streams"],
        "converged": int(sum(r["converged"] for r in recs)),
        "max_true_rel_residual": max(r["true_rel_residual"] for r in recs),
        "per_size": {N: {"count": len(v),
                         "mean_iterations": round(float(np.mean([r["iterations"] for r in v])), 1),
                         "mean_slice_s": round(float(np.mean([r["slice_s"] for r in v])), 4),
                         "start_used": int(sum(r["start_used"] for r in v))}
                     for N, v in sorted(by.items())},
        "autotune": {"nudft_chunk_scale": res["nudft_chunk_scale"], "trials_ms": res["tuner"]},
        "note": "total_s and per-size figures are the last pass (schedules already tuned); "
                "first_pass_s includes the autotuner's trial launches",
    }
    print(json.dumps(summary), flush=True)
    ctx.close()
    return 0


if __name__ == "__main__":
    import sys
    sys.exit(main())
