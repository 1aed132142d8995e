"""Benchmark of the batched per-grain level-set timestep on one MI355X.

One step = one pass of the run_sim loop body over every live grain of the workload (default
batch-100k: 100019 grains of a lognormal power diagram, R = 6325, box sides ~16-110, FP64).
Inputs are resident in HBM before the timed region; the timed region is exactly --steps steps
between two device synchronisations.  Prints one JSON line.

  value           grid-point updates/s of the hipGraph-replayed step (the production launch mode)
  phases / roofline
                  the same network stepped with stream launches and HIP events around each phase
                  (on the library's stream): the level-set launches of a step (k_compare,
                  k_contour, k_alloc, k_redist) run back to back between two events, so their
                  summed duration and algorithmic bytes give the achieved HBM rate of the phase
  pergrain_value  the same kernels with one launch per grain (the reference's per-LSbox calls)
  cpu_baseline    the oracle (C++/OpenMP restatement of the reference's CPU path) on a bounded
                  sample of the same workload, on this host's cores
  adjoint         fwd+adj s/step on the differentiation workload (diff-500: 500 grains, 16
                  mobility bins, FP64): a recorded step, the readback of the grains' areas and
                  perimeters, and ggx_step_adjoint, against a plain step of the same trajectory
"""
import argparse
import json
import os
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

HBM_PEAK = 8.0e12  # MI355X HBM3E, bytes/s


def parse():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=20)
    ap.add_argument("--warmup", type=int, default=3)
    ap.add_argument("--workload", default="batch-100k")
    ap.add_argument("--precision", default="fp64", choices=["fp64", "fp32"])
    ap.add_argument("--graph", type=int, default=1, help="1: time the hipGraph-replayed step, 0: stream launches")
    ap.add_argument("--conv", default="auto", choices=["auto", "circulant", "fft"], help="convolution engine")
    ap.add_argument("--tuned", type=int, default=1, help="1: use the committed autotuner table when there is one")
    ap.add_argument("--phase-steps", type=int, default=5, help="stream-launched steps timed per phase (0 = skip)")
    ap.add_argument("--pergrain-steps", type=int, default=1, help="steps timed with one launch per grain (0 = skip)")
    ap.add_argument("--cpu-grains", type=int, default=3000, help="grains of the CPU baseline sample (0 = skip)")
    ap.add_argument("--cpu-steps", type=int, default=2)
    ap.add_argument("--adjoint-steps", type=int, default=20, help="fwd+adj iterations on diff-500 (0 = skip)")
    return ap.parse_args()


ENGINES = {"auto": 0, "circulant": 1, "fft": 2}
TUNED = None   # the committed autotuner table of the workload (bucket edges, FFT buckets), if any


def tuned_kw():
    """GrainHandler options of the tuned table ({} without one)."""
    if TUNED is None:
        return {}
    from gragles2d_amd.autotune import option_kw
    return option_kw(TUNED)


def make_handler(G, N, s, net, prec, **opts):
    opts.update(tuned_kw())
    h = G.GrainHandler(s, precision=prec, batching=N.BATCH_FUSED, **opts)
    h.set_simulation_parameter(net)
    return h


def timed_steps(h, warmup, steps):
    h.step(warmup)
    h.sync()
    st0 = h.stats()
    t0 = time.perf_counter()
    h.step(steps)
    h.sync()
    sec = time.perf_counter() - t0
    return st0, h.stats(), sec


def main():
    a = parse()
    if a.gpus != 1:
        print(f"bench.py: this build runs on one GPU only; --gpus {a.gpus} is not supported "
              "(the multi-GPU sharding is a design note, not an implementation)", file=sys.stderr)
        sys.exit(2)
    from gragles2d_amd import _native as N
    from gragles2d_amd import grainhdl as G
    from gragles2d_amd.configs import WORKLOADS

    w = WORKLOADS[a.workload]
    prec = N.PREC_FP64 if a.precision == "fp64" else N.PREC_FP32
    global TUNED
    if a.tuned:
        from gragles2d_amd.autotune import tuned_options
        TUNED = tuned_options(w.name, a.precision)
    net = G.Network.generate(w.grains, w.seed, w.lognormal_sigma)
    kw = w.settings_kw()
    kw["number_of_particles"] = len(net)
    s = G.default_settings(**kw)

    # headline: the captured step replayed (or stream launches with --graph 0)
    hdl = make_handler(G, N, s, net, prec, persistent=1, use_graph=a.graph, conv_engine=ENGINES[a.conv])
    st0, st1, sec = timed_steps(hdl, a.warmup, a.steps)
    upd = st1.grid_point_updates - st0.grid_point_updates
    value = upd / sec
    out = {
        "metric": "grid-point updates/s (batched timestep)",
        "value": value,
        "unit": "grid-point updates/s",
        "n_gpus": 1,
        "steps": a.steps,
        "warmup": a.warmup,
        "ms_per_step": 1e3 * sec / a.steps,
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f64" if prec == N.PREC_FP64 else "f32",
        "data": "synthetic (seeded lognormal power diagram)",
        "config": {"workload": w.name, "grains": len(net), "grid": G.derive(s).real_domain_size,
                   "launch": "hipGraph replay" if a.graph else "stream", "conv_engine": a.conv,
                   "buckets": (TUNED["bucket_edges"] if TUNED else "built-in"),
                   "fft_buckets": (TUNED["fft_buckets"] if TUNED else 0),
                   "live_grains_last_step": st1.live_grains,
                   "max_box": st1.max_box, "grid_points_per_step": upd / a.steps},
    }
    hdl.close()

    if a.phase_steps > 0:
        out.update(phase_split(G, N, s, net, prec, w, a))
    if a.pergrain_steps > 0:
        pg = G.GrainHandler(s, precision=prec, batching=N.BATCH_PERGRAIN, conv_engine=ENGINES[a.conv],
                            **tuned_kw())
        pg.set_simulation_parameter(net)
        p0, p1, pgs = timed_steps(pg, 1, a.pergrain_steps)
        pv = (p1.grid_point_updates - p0.grid_point_updates) / pgs
        out["pergrain_value"] = pv
        out["batched_over_pergrain"] = value / pv
        pg.close()
    if a.adjoint_steps > 0:
        out["adjoint"] = adjoint_timing(a.adjoint_steps)
    if a.cpu_grains > 0:
        out["cpu_baseline"] = cpu_baseline(w, a.cpu_grains, a.cpu_steps)
    print(json.dumps(out), flush=True)


def adjoint_timing(iters, warm=16):
    """fwd+adj seconds per step on diff-500 after `warm` steps: each iteration records a step,
    reads every grain's area and perimeter, and runs the adjoint with the cotangent of the
    squared mean-area and boundary-length loss; the plain step of the same trajectory is timed
    beside it (stream launches, synchronised)."""
    import numpy as np
    from gragles2d_amd import adjoint as ADJ
    T = ADJ.Trajectory("diff-500", steps=warm + 1)
    bins = ADJ.seeded_bins(1004)
    hdl = T.handler(bins)
    hdl.step(1)
    hdl.sync()
    t0 = time.perf_counter()
    for _ in range(iters):
        hdl.step(1)
        hdl.sync()
    plain = (time.perf_counter() - t0) / iters
    fwd = adj = 0.0
    for _ in range(iters):
        t0 = time.perf_counter()
        hdl.record_next_step()
        hdl.step(1)
        area, per, alive = ADJ.grain_measures(hdl)
        t1 = time.perf_counter()
        n = max(int(alive.sum()), 1)
        ga = np.where(alive, 2 * (area[alive].sum() / n) / n, 0.0)   # d/dA of (mean area)^2
        gp = np.full(area.shape, 2 * (per.sum() / 2) / 2)              # d/dP of (length)^2
        hdl.step_adjoint(ga, gp)
        t2 = time.perf_counter()
        fwd += t1 - t0
        adj += t2 - t1
    hdl.close()
    return {"workload": "diff-500", "grains": len(T.net), "dtype": "f64", "iterations": iters,
            "plain_step_s": plain, "recorded_step_s": fwd / iters, "adjoint_s": adj / iters,
            "fwd_adj_s_per_step": (fwd + adj) / iters}


LEVEL_KERNELS = ("k_compare", "k_contour", "k_alloc", "k_redist")


def phase_split(G, N, s, net, prec, w, a):
    """Per-phase device time of stream-launched steps (HIP events on the library's stream) and
    the roofline of the dominant HBM-bound kernel from them."""
    h = make_handler(G, N, s, net, prec, persistent=1, use_graph=0, conv_engine=ENGINES[a.conv])
    st0, st1, sec = timed_steps(h, a.warmup, a.phase_steps)
    h.close()
    k = a.phase_steps
    phases = {name: (getattr(st1, name) - getattr(st0, name)) / k for name in
              ("comparison_ms", "convolution_ms", "levelset_ms")}
    phases = {"lists_ms": phases["comparison_ms"], "convolution_ms": phases["convolution_ms"],
              "level_ms": phases["levelset_ms"]}
    conv_b = (st1.conv_bytes - st0.conv_bytes) / k
    level_b = (st1.algorithmic_bytes - st0.algorithmic_bytes) / k - conv_b
    aniso = not w.isotropic
    if aniso or phases["level_ms"] >= phases["convolution_ms"]:
        # anisotropic networks: the convolution phase also holds the velocity corrector (k_aniso,
        # bound by its per-pixel projection, not by HBM), so the roofline line is the level-set phase's
        kern, byts, ms = LEVEL_KERNELS, level_b, phases["level_ms"]
    else:
        fft = a.conv == "fft" or s.convolution_mode != 2
        strips = fft and prec == N.PREC_FP64
        kern, byts, ms = (("k_box_rows", "k_box_columns") if strips else ("k_conv_fft",) if fft else ("k_conv_tiles",)), conv_b, phases["convolution_ms"]
    achieved = byts / (ms * 1e-3)
    precision = "fp64" if prec == N.PREC_FP64 else "fp32"
    if aniso:
        phases["convolution_ms includes"] = "k_aniso (the velocity corrector)"
    return {
        "phases_ms_per_step": phases,
        "stream_ms_per_step": 1e3 * sec / k,
        "algorithmic_bytes_per_step": {"convolution": conv_b, "level": level_b},
        "roofline": {"kernel": " + ".join(kern), "bound": "hbm", "achieved": achieved / 1e9, "peak": HBM_PEAK / 1e9,
                     "unit": "GB/s", "frac": achieved / HBM_PEAK,
                     "traffic": measured_traffic(w.name, precision, kern)},
    }


def measured_traffic(workload, precision, kernels):
    """HBM bytes per step of the kernels' launches from the committed rocprofv3 --pmc summary
    (FETCH_SIZE and WRITE_SIZE, scaled by what the counters read for a copy of known size);
    None when no summary exists for this workload and precision."""
    path = os.path.join(ROOT, "profiles", f"traffic_{workload.replace('-', '')}_{precision}.json")
    if not os.path.exists(path):
        return None
    with open(path) as f:
        t = json.load(f)
    prefixes = tuple(f"ggx::{k}" for k in kernels)
    hits = [e["hbm_bytes"] for name, e in t.get("per_step", {}).items() if name.startswith(prefixes)]
    return sum(hits) if hits else None


def cpu_model():
    try:
        with open("/proc/cpuinfo") as f:
            for line in f:
                if line.startswith("model name"):
                    return line.split(":", 1)[1].strip()
    except OSError:
        pass
    return "unknown"


def cpu_threads():
    env = os.environ.get("OMP_NUM_THREADS", "")
    n = len(os.sched_getaffinity(0))
    return min(n, int(env)) if env.isdigit() and int(env) > 0 else n


def cpu_baseline(w, ngrains, steps):
    """The oracle (C++/OpenMP FP64 restatement of the reference's timestep) on a bounded sample
    of the same workload: a network of `ngrains` grains with the same points per grain, border
    and size distribution, timed over `steps` steps after one untimed step."""
    from gragles2d_amd import grainhdl as G
    from oracle.pyoracle import Oracle

    threads = cpu_threads()
    net = G.Network.generate(ngrains, w.seed, w.lognormal_sigma)
    kw = w.settings_kw()
    kw["number_of_particles"] = len(net)
    d = G.derive(G.default_settings(**kw))
    o = Oracle(d.real_domain_size, w.border, d.dt, len(net), analysis_timestep=kw["analysis_timestep"], nthreads=threads,
               aniso=w.aniso())
    for i in range(len(net)):
        gid, pts, q = net.grain(i)
        o.add_grain(gid, pts, q)
    o.init()
    o.step()
    t_before = o.timers()
    upd, sec = 0, 0.0
    for _ in range(steps):
        for g in range(1, len(net) + 1):
            inf = o.info(g)
            if inf.present and inf.exists:
                upd += (inf.xmax - inf.xmin) ** 2
        t0 = time.perf_counter()
        o.step()
        sec += time.perf_counter() - t0
    t_after = o.timers()
    phases = {k: 1e3 * (t_after[k] - t_before[k]) / steps for k in t_after}
    return {"value": upd / sec, "unit": "grid-point updates/s", "cores": threads, "kind": "port",
            "cpu": cpu_model(), "ms_per_step": 1e3 * sec / steps, "phases_ms_per_step": phases,
            "sample": f"{len(net)}-grain network of the same workload (ppg {w.points_per_grain}, border {w.border}, "
                      f"sigma {w.lognormal_sigma}), {steps} steps after one untimed step, {threads} OpenMP threads"}


if __name__ == "__main__":
    main()
