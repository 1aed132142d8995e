"""What the performance of this framework is measured on: the work a simulation program has it do,
through the public entry points (GrainHandler, Trajectory, ggx_convolve_boxes).

Kinds of case:
  run     a whole short simulation: context, network load, every pass of the loop, the frame read
          back (the small networks, where launches, latency and loading count)
  steps   a simulation under way: `steps` passes of the loop on a loaded network, then the grains'
          table read back for the statistics (the large networks; the state moves on from pass to pass)
  diff    the differentiation workload: a trajectory, its loss and the backward pass to the 16
          mobility bins
  boxes   the batched convolution on caller-owned device buffers, ragged box sides
"""
import ctypes
import math

import numpy as np
import torch

from gragles2d_amd import _native as N
from gragles2d_amd import adjoint as ADJ
from gragles2d_amd import grainhdl as G

INFO = np.dtype([(name, np.int32) for name, _ in N.GrainInfo._fields_[:16]] +
                [(name, np.float64) for name, _ in N.GrainInfo._fields_[16:]])


def _net(kind, name=None, *, grains, ppg=20, border=7, sigma=0.0, steps, fp32=False, graph=True, mode=2, aniso=0):
    """A network case: grain count, NumberOfPointsPerGrain, DomainBorderSize, lognormal spread of
    the grain sizes, passes, field type, launch mode, ConvolutionMode, UseMobilityModel (0: isotropic)."""
    c = dict(kind=kind, grains=grains, ppg=ppg, border=border, sigma=sigma, steps=steps, fp32=fp32, graph=graph,
             mode=mode, aniso=aniso)
    return dict(c, name=name) if name else c


def _boxes(name=None, *, count, lo, hi, mode, noalloc=False):
    """A convolution batch: box count, smallest and largest side, ConvolutionMode, the entry point."""
    c = dict(kind="boxes", count=count, lo=lo, hi=hi, mode=mode, noalloc=noalloc)
    return dict(c, name=name) if name else c


def listed():
    return [
        # plain-100: the quick look at a small network, all 21 passes of its 20 timesteps, default options
        _net("run", "plain-100 run", grains=100, steps=21, graph=False),
        # iso-2k: an everyday study, all 201 passes with a wide margin, captured steps
        _net("run", "iso-2k run", grains=2000, border=20, steps=201),
        # aniso-10k: Read-Shockley energies, sigmoid mobility and junction drag on a production network
        _net("steps", "aniso-10k", grains=10000, steps=20, aniso=1),
        # batch-100k: the headline network in FP64
        _net("steps", "batch-100k fp64", grains=100000, sigma=0.35, steps=20),
        # a mid-size lognormal network in FP32, where areas are wanted and 1e-5 is enough
        _net("steps", "batch-30k fp32", grains=30000, sigma=0.35, steps=40, fp32=True),
        # few grains, finely resolved: boxes of 70 to 300 points
        _net("steps", "fine-200", grains=200, ppg=60, border=10, sigma=0.35, steps=50),
        # the Laplace symbol, which only the FFT engine convolves
        _net("steps", "laplace-5k", grains=5000, sigma=0.35, steps=60, mode=0),
        # diff-500: the 128-step trajectory with its loss and gradient
        _net("diff", "diff-500 loss+grad", grains=500, steps=128, graph=False, aniso=4),
        # a handful of boxes convolved, as a test or a post-processing script does: launches and set-up
        _boxes("boxes-24 gaussian", count=24, lo=16, hi=64, mode=2),
        # every box of a network convolved at once, ragged sides
        _boxes("boxes-6k richardson", count=6000, lo=16, hi=128, mode=1),
        # wide boxes through the entry point that allocates nothing
        _boxes("boxes-96 wide", count=96, lo=130, hi=256, mode=0, noalloc=True),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["run", "steps", "steps", "aniso", "fine", "fft", "diff", "boxes"])
    if kind == "run":  # small isotropic networks from load to frame
        return _net("run", grains=_log(rng, 40, 2000), border=rng.choice([7, 7, 10, 20]), steps=rng.randint(20, 120),
                    fp32=rng.random() < 0.25, graph=rng.random() < 0.5)
    if kind == "steps":  # isotropic networks under way, mid-size to the headline's
        g = _log(rng, 1500, 95000)
        return _net("steps", grains=g, sigma=rng.choice([0.0, 0.35]), steps=max(8, min(60, 1200000 // g)),
                    fp32=rng.random() < 0.4, graph=rng.random() < 0.7)
    if kind == "aniso":
        g = _log(rng, 300, 12000)
        return _net("steps", grains=g, steps=max(12, min(60, 200000 // g)), fp32=rng.random() < 0.2,
                    aniso=rng.choice([1, 1, 2, 4]),
                    graph=rng.random() < 0.7)
    if kind == "fine":
        return _net("steps", grains=rng.randint(60, 300), ppg=rng.randint(45, 64), border=10, sigma=rng.choice([0.0, 0.35]),
                    steps=rng.randint(20, 50), graph=rng.random() < 0.7)
    if kind == "fft":
        g = _log(rng, 400, 8000)
        return _net("steps", grains=g, sigma=rng.choice([0.0, 0.35]), steps=max(15, min(60, 200000 // g)),
                    mode=rng.choice([0, 0, 1]), graph=rng.random() < 0.7)
    if kind == "diff":
        return _net("diff", grains=rng.randint(150, 700), steps=rng.randint(24, 128), graph=False, aniso=4)
    if rng.random() < 0.3:
        return _boxes(count=_log(rng, 8, 96), lo=130, hi=rng.randint(140, 256), mode=rng.randint(0, 2),
                      noalloc=rng.random() < 0.5)
    return _boxes(count=_log(rng, 8, 6000), lo=rng.randint(8, 30), hi=rng.randint(33, 128), mode=rng.randint(0, 2),
                  noalloc=rng.random() < 0.3)


def _settings_kw(case, grains):
    kw = dict(number_of_particles=grains, number_of_points_per_grain=case["ppg"], number_of_timesteps=case["steps"] - 1,
              analysis_timestep=10, plot_interval=1, domain_border_size=case["border"], microstructure_gen_mode=0,
              convolution_mode=case["mode"], is_isotropic_network=0 if case["aniso"] else 1, breakup_number=0,
              discrete_sampling_rate=31, grain_scheduler=0, lattice_type=0)
    if case["aniso"]:
        ds = (3.0 * 2 + 2.0 * 2) / int(math.sqrt(case["grains"]) * case["ppg"])
        kw.update(research_mode=0, use_mobility_model=case["aniso"], triple_point_drag=0.5 / ds,
                  constant_sector_radius=3.0, interpolating_sector_radius=2.0)
    return kw


def _handler(case, net, settings):
    h = G.GrainHandler(settings, precision=N.PREC_FP32 if case["fp32"] else N.PREC_FP64, use_graph=int(case["graph"]))
    if case["aniso"] == 4:
        h.set_mobility_bins(ADJ.seeded_bins(case["grains"]))
    h.set_simulation_parameter(net)
    return h


def _table(case, t):
    """The grains' table (info_all) as columns with room for the few grains that a power diagram
    gives beyond the count asked for, so that every seed's outputs have one shape."""
    out = {name: np.zeros(int(1.02 * case["grains"]) + 64, INFO[name]) for name in INFO.names}
    for name in INFO.names:
        out[name][:len(t)] = t[name]
    return out


def _fields(case, seed):
    """Boxes of the case's sides in an order of the seed's: signed distances of a disc of random
    centre and radius, clamped to the band, as a step meets them."""
    n = np.random.default_rng(case["count"] + case["lo"]).integers(case["lo"], case["hi"] + 1, case["count"])
    n[0] = case["hi"]
    rng = np.random.default_rng(seed)
    n = rng.permutation(n.astype(np.int64))
    delta = 0.035
    out = []
    for side in n.tolist():
        y, x = np.mgrid[0:side, 0:side]
        cx, cy, r = rng.uniform(0.35, 0.65) * side, rng.uniform(0.35, 0.65) * side, rng.uniform(0.2, 0.4) * side
        out.append(np.clip((r - np.hypot(x - cx, y - cy)) * 0.005, -delta, delta).reshape(-1))
    return n, np.concatenate(out)


DT, R = 2.2e-5, 200  # the time step and grid of a 100-grain network


def prepare(case, seed):
    if case["kind"] == "boxes":
        n, flat = _fields(case, seed)
        off = np.concatenate([[0], np.cumsum(n * n)[:-1]])
        d = torch.device("cuda:0")
        src = torch.from_numpy(flat).to(d)
        return dict(case=case, lib=N.load(), n=torch.from_numpy(n.astype(np.int32)).to(d), off=torch.from_numpy(off).to(d),
                    src=src, dst=torch.empty_like(src), max_n=int(n.max()))
    net = G.Network.generate(case["grains"], seed, case["sigma"])
    if case["kind"] == "diff":
        t = ADJ.Trajectory("diff-500", steps=case["steps"])
        t.net = net
        t.settings = dict(_settings_kw(case, len(net)), number_of_timesteps=case["steps"])
        return dict(case=case, trajectory=t, bins=torch.from_numpy(ADJ.seeded_bins(seed)), target=(1.0 / len(net), 30.0))
    settings = G.default_settings(**_settings_kw(case, len(net)))
    if case["kind"] == "run":
        return dict(case=case, net=net, settings=settings)
    h = _handler(case, net, settings)
    h.step(2)  # under way: both buffer parities met, the corrector on
    h.sync()
    return dict(case=case, handler=h)


def run(state):
    case = state["case"]
    if case["kind"] == "boxes":
        call = state["lib"].ggx_convolve_boxes_noalloc if case["noalloc"] else state["lib"].ggx_convolve_boxes
        rc = call(case["count"], state["n"].data_ptr(), state["off"].data_ptr(), state["src"].data_ptr(),
                  state["dst"].data_ptr(), state["max_n"], case["mode"], DT, R,
                  ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
        N.check(rc, "ggx_convolve_boxes")
        return state["dst"]
    if case["kind"] == "diff":
        bins = state["bins"].clone().requires_grad_(True)
        t = state["trajectory"]
        h = t.handler(state["bins"].numpy())
        loss = t.loss(bins, state["target"], h)
        loss.backward()
        out = dict(loss=loss.detach(), grad=bins.grad, table=_table(case, np.frombuffer(h.info_all(), dtype=INFO)))
        h.close()
        return out
    if case["kind"] == "run":
        h = _handler(case, state["net"], state["settings"])
        if case["graph"]:
            h.step(case["steps"])
        else:
            h.run_sim(case["steps"])  # pass by pass, with the surviving grains counted after each
        f = h.frame()
        # every live grain's field, grain after grain, in an array of one size for every seed
        phi, o = np.zeros(int(3 * (1.3 * case["ppg"] + 2 * case["border"]) ** 2 * case["grains"])), 0
        for g in np.flatnonzero(f.info["exists"]).tolist():
            if g > 0:
                v = f.phi(g).reshape(-1)
                phi[o:o + v.size] = v
                o += v.size
        out = dict(table=_table(case, f.info), phi=phi)
        h.close()
        return out
    h = state["handler"]
    h.step(case["steps"])
    return _table(case, np.frombuffer(h.info_all(), dtype=INFO))


def work(case):
    """Compulsory traffic and arithmetic: per step every box point's field read and written and its
    IDLocal written; two separable passes of n multiply-adds per point (2 n log2 n butterflies for
    the FFT).  The side of an average box is 1.3 points-per-grain spacings plus the two margins."""
    if case["kind"] == "boxes":
        pts = case["count"] * (case["lo"] ** 2 + case["lo"] * case["hi"] + case["hi"] ** 2) / 3.0
        return {"bytes": 16.0 * pts, "flops": 20.0 * pts * math.log2(case["hi"])}
    n = 1.3 * case["ppg"] + 2 * case["border"]
    pts = case["grains"] * n * n * case["steps"]
    per = 4.0 * n if case["mode"] == 2 else 20.0 * math.log2(n)
    return {"bytes": pts * (2 * (4 if case["fp32"] else 8) + 4), "flops": pts * per}


def _symbol(n, mode):
    """The convolution's symbol over the half spectrum (row frequency j, column frequency i)."""
    nsq = float(R) * R
    j = np.arange(n, dtype=np.float64)[:, None]
    i = np.arange(n // 2 + 1, dtype=np.float64)[None, :]
    if mode == 2:
        i2, j2 = np.minimum(i, n - i), np.minimum(j, n - j)
        return np.exp(-math.sqrt(2 / math.pi) * (i2 * i2 + j2 * j2) * 4.0 * DT * nsq / (n * n) * math.pi ** 2)
    g = 2.0 * (2.0 - np.cos(2 * np.pi * i / n) - np.cos(2 * np.pi * j / n)) * nsq
    if mode == 0:
        return 1.0 / (1.0 + DT * g)
    return (4.0 / (1 + 1.5 * DT / 40 * g) ** 40 - 1.0 / (1 + 3.0 * DT / 40 * g) ** 40) / 3.0


def exact(case, seed):
    """The convolutions by numpy's FFT.  A simulation's outputs hang on thousands of discrete
    decisions per step (contours, winners, removals): they have no value but the step's own."""
    if case["kind"] != "boxes":
        return None
    n, flat = _fields(case, seed)
    out, o, sym = np.empty_like(flat), 0, {}
    for side in n.tolist():
        if side not in sym:
            sym[side] = _symbol(side, case["mode"])
        f = flat[o:o + side * side].reshape(side, side)
        out[o:o + side * side] = np.fft.irfft2(np.fft.rfft2(f) * sym[side], s=(side, side)).reshape(-1)
        o += side * side
    return torch.from_numpy(out)
