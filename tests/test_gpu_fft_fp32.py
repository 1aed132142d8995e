"""FP32 steps on the FFT engine (k_conv_fft), which every FP32 bucket with a Laplace symbol, with the
engine asked for or picked by the tuned table takes: half spectra in LDS (sides up to 128) and in global
slots (above).  The bar of the FP32 path: the same grains survive, and every grain's area is within 1e-5 of
the FP64 oracle's or within 30 times what float storage alone does to that grain.
"""
import numpy as np
import pytest

from gragles2d_amd import _native as N
from gragles2d_amd import grainhdl as G

from .gpu_helpers import make_oracle, make_pair, settings_for
from .test_gpu_parity import COND_FACTOR, FP32_MIN_CELLS, FP32_TOL

pytestmark = pytest.mark.gpu

CASES = [(100, 20, 7, 0.35, 8), (6, 60, 40, 0.0, 4), (40, 60, 10, 0.35, 4)]


def _areas(net, steps, ppg, gb, mode, **opts):
    gpu, o = make_pair(net, ppg=ppg, gb=gb, precision=N.PREC_FP32, mode=mode, oracle_threads=8, **opts)
    r = make_oracle(net, ppg, gb, 8, keep_compared=False, mode=mode)
    for _ in range(steps):
        gpu.step(1)
        assert o.step() == 0
        r.round_fields_to_float()
        assert r.step() == 0
    fr, cell, worst = gpu.frame(), gpu.derived.h ** 2, 0.0
    for g in range(1, len(net) + 1):
        gi, oi, ri = fr.info[g], o.info(g), r.info(g)
        assert bool(gi["present"] and gi["exists"]) == bool(oi.present and oi.exists), g
        if oi.present and oi.exists:
            scale = max(oi.volume, FP32_MIN_CELLS * cell)
            err = abs(gi["volume"] - oi.volume) / scale
            cond = abs(ri.volume - oi.volume) / scale if (ri.present and ri.exists) else float("inf")
            worst = max(worst, err)
            assert err <= max(FP32_TOL, COND_FACTOR * cond), (g, err, cond)
    print(f"mode {mode}: max area error {worst:.1e}", flush=True)


@pytest.mark.parametrize("n,ppg,gb,sigma,steps", CASES)
@pytest.mark.parametrize("mode", [0, 1])
def test_laplace_steps(n, ppg, gb, sigma, steps, mode):
    _areas(G.Network.generate(n, 600 + n, sigma), steps, ppg, gb, mode)


@pytest.mark.parametrize("n,ppg,gb,sigma,steps", CASES)
@pytest.mark.parametrize("opts", [dict(conv_engine=N.CONV_FFT), dict(fft_buckets=0x2AA)])
def test_gaussian_steps_on_the_engine(n, ppg, gb, sigma, steps, opts):
    _areas(G.Network.generate(n, 600 + n, sigma), steps, ppg, gb, 2, **opts)


def _run(net, ppg, gb, mode, steps, **opts):
    h = G.GrainHandler(settings_for(len(net), ppg, gb, mode), **opts)
    h.set_simulation_parameter(net)
    h.step(steps)
    return h


@pytest.mark.parametrize("n,ppg,gb,sigma,steps", CASES)
@pytest.mark.parametrize("opts", [dict(batching=N.BATCH_PERGRAIN), dict(persistent=0), dict(use_graph=1)])
def test_launch_modes_give_the_same_bits(n, ppg, gb, sigma, steps, opts):
    net = G.Network.generate(n, 600 + n, sigma)
    ha = _run(net, ppg, gb, 0, steps, precision=N.PREC_FP32)
    hb = _run(net, ppg, gb, 0, steps, precision=N.PREC_FP32, **opts)
    a, b = ha.frame(), hb.frame()
    for g in range(1, len(net) + 1):
        assert a.info[g].tobytes() == b.info[g].tobytes(), g
        if a.info[g]["exists"]:
            assert np.array_equal(a.phi(g), b.phi(g)) and np.array_equal(a.idlocal(g), b.idlocal(g)), g


@pytest.mark.parametrize("mode", [0, 1])
def test_fp64_fallback_agrees_with_the_strips(mode):
    # one-grain launches under 16000 bytes of LDS: the boxes whose strips are above that take the FFT
    net = G.Network.generate(30, 1000)
    ha = _run(net, 20, 7, mode, 3, batching=N.BATCH_PERGRAIN)
    hb = _run(net, 20, 7, mode, 3, batching=N.BATCH_PERGRAIN, lds_budget=16000)
    a, b = ha.frame(), hb.frame()
    sides = [a.info[g]["xmax"] - a.info[g]["xmin"] for g in range(1, len(net) + 1) if a.info[g]["exists"]]
    assert max(sides) > 54, max(sides)   # 288 n bytes and more of a strip of columns
    for g in range(1, len(net) + 1):
        assert bool(a.info[g]["exists"]) == bool(b.info[g]["exists"]), g
        if a.info[g]["exists"]:
            assert float(np.max(np.abs(a.phi(g) - b.phi(g)))) <= 1e-10, g
