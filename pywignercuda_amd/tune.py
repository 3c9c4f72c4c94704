"""Autotuner: times every launch variant of the fused sweeps on the local GPU and
writes the fastest per (precision, regime, sweep, grid size) to tuning.json.

    python -m pywignercuda_amd.tune [--sizes 128,256,512,1024,2048] [--reps 50]

Regimes: "single" (one Wigner function, timed as whole steps of the graph-replayed
step loop, per-step microseconds in the *_us entries) and "batch" (an ensemble of
equal grids holding about 1 GiB, enough to fill the GPU).  The plans read the table
at creation (Wigner2D / WignerEnsemble, argument variants=None).
"""
from __future__ import annotations

import argparse
import json
import time
from pathlib import Path

import numpy as np

from . import _lib
from .wigner2d import TUNING_FILE, Wigner2D, WignerEnsemble


def _time(fn, reps):
    import torch

    fn()
    torch.cuda.synchronize()
    s, e = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    s.record()
    for _ in range(reps):
        fn()
    e.record()
    e.synchronize()
    return s.elapsed_time(e) / reps * 1e3  # us


def _better(v, t, best):
    """Whether variant v (time t) replaces best = (variant, time): the default variant 0 is
    timed first and is replaced only by a variant at least 1% faster (run-to-run noise)."""
    if best is None:
        return True
    return t < best[1] * (0.99 if best[0] == 0 else 1.0)


def _variants(table):
    L = _lib.lib()
    return range(L.wh_variant_info(table, -1, None, None))


def _step_us(p, W, steps):
    """Time per step of the graph-replayed step loop: each sweep then reads what the
    other wrote, as in a real run.  The plan's graphs must already be captured."""
    import torch

    torch.cuda.synchronize()
    t0 = time.perf_counter()
    p.run(W, steps, use_graph=True)
    torch.cuda.synchronize()
    return (time.perf_counter() - t0) / steps * 1e6


def _pick(p, W, table, steps, rounds=5):
    """Fastest variant of one table, timed in alternating rounds (variants often differ by
    1-2%, about the drift between two runs); the per-variant time is the best round."""
    times = {}
    for _ in range(rounds):
        for v in _variants(table):
            args = [-1, -1, -1]
            args[table] = v
            try:
                p.set_variants(*args)
            except _lib.WignerHipError:
                continue
            p.run(W, 4, use_graph=True)  # graph capture for this variant
            t = _step_us(p, W, steps)
            times[v] = min(t, times.get(v, t))
    best = None
    for v in sorted(times):
        if _better(v, times[v], best):
            best = (v, times[v])
    if best is not None:
        args = [-1, -1, -1]
        args[table] = best[0]
        p.set_variants(*args)
    return best


def tune_single(prec, N, reps, cl=False, xvar=None):
    """Variant of each sweep for one Wigner function, timed as whole steps of the step loop
    (x sweep first with the default p sweep, then the p sweep with the chosen x sweep);
    cl: the Caldeira-Leggett p sweep, with the x sweep fixed at xvar."""
    kw = dict(potential="0.5*pow(x,2) + 0.1*pow(x,4)", dpotential="x + 0.4*pow(x,3)", mask=True, precision=prec)
    if cl:
        kw.update(gamma=0.1, damping="CaldeiraLeggett", fp_damping="fabs(p)", D_theta=0.1)
    p = Wigner2D(N, N, 10.0, 10.0, 1.0, 1.0, 0.01, variants=(0, 0, 0), **kw)
    x, pp = p.x_host[None, :], p.p_host[:, None]
    W = p.to_device(np.exp(-((x - 1.0) ** 2) - pp ** 2))
    steps = max(100, 2 * reps)
    out = {}
    if cl and xvar is not None:
        p.set_variants(xvar, -1, -1)
    for table, name in ((0, "x"), (2 if cl else 1, "pcl" if cl else "p")):
        if cl and table == 0:
            continue
        out[name] = _pick(p, W, table, steps)
    p.close()
    return out


def tune_batch(prec, N, reps, cl=False):
    """Variant of each sweep for an ensemble; cl: of the Caldeira-Leggett p sweep, with the other
    sweeps as the table has them."""
    import torch

    bytes_per = N * N * (16 if prec == "fp64" else 8)
    n = max(2, min(512, (1 << 30) // bytes_per))
    m = dict(X=N, P=N, X_amp=10.0, P_amp=10.0, potential="0.5*pow(x,2) + 0.1*pow(x,4)",
             dpotential="x + 0.4*pow(x,3)")
    kw = {}
    if cl:
        m.update(fp_damping="fabs(p)", D_theta=0.1)
        kw.update(gamma=0.1, damping="CaldeiraLeggett")
    ens = WignerEnsemble([m] * n, 1.0, 1.0, 0.01, precision=prec, variants=None if cl else (0, 0, 0), **kw)
    states = [torch.zeros((N, N), dtype=ens.dtype, device=ens.device) for _ in range(n)]
    for s in states:
        s[0, 0] = 1.0
    out = {}
    for table, name in ((2, "pcl"),) if cl else ((0, "x"), (1, "p")):
        best = None
        for v in _variants(table):
            args = [-1, -1, -1]
            args[table] = v
            try:
                ens.set_variants(*args)
            except _lib.WignerHipError:
                continue
            t = _time(lambda: ens.run(states, 4, normalize_initial=False, use_graph=False), max(2, reps // 10))
            if _better(v, t, best):
                best = (v, t)
        out[name] = best
    ens.close()
    return out


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--sizes", default="128,256,512,1024,2048")
    ap.add_argument("--reps", type=int, default=50)
    ap.add_argument("--no-batch", action="store_true")
    ap.add_argument("--out", default=None, help="write the table here instead of the package's tuning.json")
    a = ap.parse_args()
    sizes = [int(s) for s in a.sizes.split(",")]
    table = json.loads(TUNING_FILE.read_text()) if TUNING_FILE.exists() else {}
    t0 = time.time()
    for prec in ("fp64", "fp32", "fp32fast"):
        single = table.setdefault(prec, {})
        batch = table.setdefault(prec + "_batch", {})
        for N in sizes:
            r = tune_single(prec, N, a.reps)
            rc = tune_single(prec, N, a.reps, cl=True, xvar=r["x"][0] if r.get("x") else None)
            for k, v in list(r.items()) + list(rc.items()):
                if v is not None:
                    single.setdefault(k, {})[str(N)] = v[0]
                    single.setdefault(k + "_us", {})[str(N)] = round(v[1], 2)
            print(f"{prec} {N}: single {r} cl {rc}", flush=True)
            if not a.no_batch:
                rb = {**tune_batch(prec, N, a.reps), **tune_batch(prec, N, a.reps, cl=True)}
                for k, v in rb.items():
                    if v is not None:
                        batch.setdefault(k, {})[str(N)] = v[0]
                        batch.setdefault(k + "_us", {})[str(N)] = round(v[1], 2)
                print(f"{prec} {N}: batch {rb}", flush=True)
    table["_meta"] = {"seconds": round(time.time() - t0, 1)}
    out = Path(a.out) if a.out else TUNING_FILE
    out.write_text(json.dumps(table, indent=1, sort_keys=True))
    print(f"wrote {out}")


if __name__ == "__main__":
    main()
