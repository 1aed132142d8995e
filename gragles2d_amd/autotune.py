"""Autotuner of the batched timestep: box-size bucket edges and, per bucket, the convolution
engine (circulant or GGX_CONV_FFT, which takes the strip products in FP64), picked by timing the real step on the device.

    python -m gragles2d_amd.autotune --workload batch-100k [--precision fp64] [--steps 5]

Candidates for the bucket edges are the built-in table, finer and coarser regular tables and
tables cut at quantiles of the workload's initial box sides (equal grain counts per bucket);
each is timed on stream-launched steps with the library's per-phase HIP events.  With the best
table, every populated bucket is then tried with the FFT engine, and keeps it when the step's
convolution phase gets faster.  The result is written to gragles2d_amd/tuned/<workload>_<prec>.json
and read back by `tuned_options` (bench.py uses it).  The choice changes only launch shapes and
the convolution's rounding, never the algorithm: every table gives the same results within the
parity bar (the circulant and FFT engines agree to ~1e-16).
"""
import argparse
import ctypes
import json
import os
import sys
import time

HERE = os.path.dirname(os.path.abspath(__file__))
TUNED = os.path.join(HERE, "tuned")
MAX_BOX = 512
MAX_BUCKETS = 16
DEFAULT_EDGES = [24, 32, 40, 48, 56, 64, 96, 128, 192, 256, 512]


def table_path(workload, precision):
    return os.path.join(TUNED, f"{workload}_{precision}.json")


def tuned_options(workload, precision):
    """{'bucket_edges': [...], 'fft_buckets': mask} from the committed table, or None."""
    path = table_path(workload, precision)
    if not os.path.exists(path):
        return None
    with open(path) as f:
        t = json.load(f)
    return {"bucket_edges": t["bucket_edges"], "fft_buckets": t["fft_buckets"], "path": path,
            "ms_per_step": t.get("ms_per_step")}


def _close(edges):
    """Ascending, unique, capped at MAX_BUCKETS entries, ending with MAX_BOX."""
    e = sorted({int(x) for x in edges if 1 <= x < MAX_BOX})
    while len(e) > MAX_BUCKETS - 1:   # merge the closest pair of lower edges
        k = min(range(len(e) - 1), key=lambda i: e[i + 1] - e[i])
        del e[k]
    return e + [MAX_BOX]


def candidates(sides):
    """Edge tables to time: built-in, regular steps of 4, 8 and 16 over the sides that occur, and
    quantile cuts of the sides (8, 10 and 12 buckets, rounded up to multiples of 4)."""
    import numpy as np
    lo, hi = int(np.min(sides)), int(np.max(sides))
    out = {"built-in": _close(DEFAULT_EDGES)}
    for step in (4, 8, 16):
        first = (lo + step - 1) // step * step
        out[f"step{step}"] = _close(list(range(first, hi + step, step)) + [128, 256])
    for k in (8, 10, 12):
        q = np.quantile(sides, np.linspace(0, 1, k + 1)[1:])
        out[f"quantile{k}"] = _close([int((v + 3) // 4 * 4) for v in q] + [hi, 128, 256])
    uniq, seen = {}, set()
    for name, e in out.items():
        if tuple(e) not in seen:
            seen.add(tuple(e))
            uniq[name] = e
    return uniq


def option_kw(tuned):
    """Keyword options of GrainHandler for a tuned table."""
    e = list(tuned["bucket_edges"])
    return {"bucket_edges": (ctypes.c_int * MAX_BUCKETS)(*(e + [0] * (MAX_BUCKETS - len(e)))),
            "fft_buckets": int(tuned["fft_buckets"])}


def time_step(G, N, s, net, prec, edges, fft_mask, warmup, steps):
    """ms per step and per-phase ms of stream-launched steps with this table."""
    h = G.GrainHandler(s, precision=prec, batching=N.BATCH_FUSED, persistent=1, use_graph=0,
                       **option_kw({"bucket_edges": edges, "fft_buckets": fft_mask}))
    h.set_simulation_parameter(net)
    h.step(warmup)
    h.sync()
    st0 = h.stats()
    t0 = time.perf_counter()
    h.step(steps)
    h.sync()
    sec = time.perf_counter() - t0
    st1 = h.stats()
    h.close()
    ph = {k: (getattr(st1, k) - getattr(st0, k)) / steps for k in ("comparison_ms", "convolution_ms", "levelset_ms")}
    return 1e3 * sec / steps, ph


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--workload", default="batch-100k")
    ap.add_argument("--precision", default="fp64", choices=["fp64", "fp32"])
    ap.add_argument("--steps", type=int, default=5)
    ap.add_argument("--warmup", type=int, default=2)
    ap.add_argument("--out", default=None)
    a = ap.parse_args()
    sys.path.insert(0, os.path.dirname(HERE))
    import numpy as np
    from gragles2d_amd import _native as N
    from gragles2d_amd import grainhdl as G
    from gragles2d_amd.configs import WORKLOADS

    w = WORKLOADS[a.workload]
    prec = N.PREC_FP64 if a.precision == "fp64" else N.PREC_FP32
    net = G.Network.generate(w.grains, w.seed, w.lognormal_sigma)
    kw = w.settings_kw()
    kw["number_of_particles"] = len(net)
    s = G.default_settings(**kw)
    # initial box sides of the workload (the sides the buckets will hold)
    probe = G.GrainHandler(s, precision=prec)
    probe.set_simulation_parameter(net)
    fr = probe.frame()
    sides = np.array([int(fr.info[g]["xmax"] - fr.info[g]["xmin"]) for g in range(1, fr.nslots)
                      if fr.info[g]["present"] and fr.info[g]["exists"]])
    probe.close()
    log = {"workload": w.name, "precision": a.precision, "device": "MI355X (gfx950)",
           "box_sides": {"min": int(sides.min()), "median": float(np.median(sides)), "max": int(sides.max())},
           "edge_candidates": {}, "fft_trials": {}}
    best = None
    for name, edges in candidates(sides).items():
        ms, ph = time_step(G, N, s, net, prec, edges, 0, a.warmup, a.steps)
        log["edge_candidates"][name] = {"edges": edges, "ms_per_step": ms, "phases_ms": ph}
        print(f"{name:12s} {ms:8.3f} ms/step  {edges}", flush=True)
        if best is None or ms < best[0]:
            best = (ms, name, edges, ph)
    ms0, name, edges, ph0 = best
    mask = 0
    conv = ph0["convolution_ms"]
    for b, e in enumerate(edges):
        lo = edges[b - 1] if b else 0
        if not np.any((sides > lo) & (sides <= e)):
            continue
        ms, ph = time_step(G, N, s, net, prec, edges, mask | (1 << b), a.warmup, a.steps)
        keep = ph["convolution_ms"] < conv
        log["fft_trials"][str(e)] = {"convolution_ms": ph["convolution_ms"], "kept": bool(keep)}
        print(f"  bucket <= {e:3d}: FFT convolution {ph['convolution_ms']:.3f} ms vs {conv:.3f} ms -> "
              f"{'FFT' if keep else 'circulant'}", flush=True)
        if keep:
            mask |= 1 << b
            conv = ph["convolution_ms"]
    ms, ph = time_step(G, N, s, net, prec, edges, mask, a.warmup, a.steps)
    log.update({"bucket_edges": edges, "fft_buckets": mask, "chosen": name, "ms_per_step": ms, "phases_ms": ph,
                "command": f"python -m gragles2d_amd.autotune --workload {a.workload} --precision {a.precision} "
                           f"--steps {a.steps} --warmup {a.warmup}"})
    out = a.out or table_path(w.name, a.precision)
    os.makedirs(os.path.dirname(out), exist_ok=True)
    with open(out, "w") as f:
        json.dump(log, f, indent=1)
    print(f"chose {name} {edges}, fft mask {mask:#x}: {ms:.3f} ms/step -> {out}", flush=True)


if __name__ == "__main__":
    main()
