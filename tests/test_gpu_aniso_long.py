"""The velocity corrector on contours longer than it stages in LDS (above 320 points), against the oracle:
existence and boxes exactly, fields to 1e-10 after every step, and one-grain launches bit for bit."""
import numpy as np
import pytest

from gragles2d_amd import _native as N
from gragles2d_amd import grainhdl as G

from .gpu_helpers import ANISO, make_pair, settings_for

pytestmark = pytest.mark.gpu

STAGED = 320
NETS = [(4, 11, 110, 0.0, 1), (6, 15, 80, 0.3, 1), (5, 14, 90, 0.0, 4)]  # grains, seed, points per grain, sigma, model


def _aniso(model):
    a = dict(ANISO, mobility_model=model)
    if model == 4:
        a["mobility_bins"] = [0.2 + 0.05 * b for b in range(16)]
    return a


@pytest.mark.parametrize("n,seed,ppg,sigma,model", NETS)
def test_long_contours_match_the_oracle(n, seed, ppg, sigma, model):
    net = G.Network.generate(n, seed, sigma)
    gpu, o = make_pair(net, ppg=ppg, gb=9, aniso=_aniso(model), oracle_threads=8)
    longer = 0
    for t in range(4):
        if t > 0:
            info = gpu.info_all()
            longer += sum(info[g].contour_len > STAGED for g in range(1, len(net) + 1) if info[g].exists and info[g].motion_regular)
        gpu.step(1)
        assert o.step() == 0
        f, worst = gpu.frame(), 0.0
        for g in range(1, len(net) + 1):
            gi, oi = f.info[g], o.info(g)
            assert bool(gi["present"] and gi["exists"]) == bool(oi.present and oi.exists), (t, g)
            if oi.present and oi.exists:
                assert (gi["xmin"], gi["xmax"], gi["ymin"], gi["ymax"]) == (oi.xmin, oi.xmax, oi.ymin, oi.ymax), (t, g)
                worst = max(worst, float(np.max(np.abs(f.phi(g) - o.phi(g)))))
        print(f"step {t}: max|dphi| {worst:.1e}", flush=True)
        assert worst <= 1e-10, t
    assert longer > 0


@pytest.mark.parametrize("prec", [N.PREC_FP64, N.PREC_FP32])
@pytest.mark.parametrize("n,seed,ppg,sigma,model", NETS)
def test_launch_modes_give_the_same_bits(n, seed, ppg, sigma, model, prec):
    net = G.Network.generate(n, seed, sigma)
    runs = []
    for opts in (dict(), dict(batching=N.BATCH_PERGRAIN), dict(use_graph=1)):
        h = G.GrainHandler(settings_for(len(net), ppg, 9, 2, aniso=_aniso(model)), precision=prec, **opts)
        if model == 4:
            h.set_mobility_bins(_aniso(4)["mobility_bins"])
        h.set_simulation_parameter(net)
        h.step(4)
        runs.append((h, h.frame()))
    a = runs[0][1]
    for _, b in runs[1:]:
        for g in range(1, len(net) + 1):
            assert a.info[g].tobytes() == b.info[g].tobytes(), g
            if a.info[g]["exists"]:
                assert np.array_equal(a.phi(g), b.phi(g)) and np.array_equal(a.idlocal(g), b.idlocal(g)), g
