"""A context's lds_budget on the GPU: one-grain launches under a budget give the bits of the same run
without one (the convolution of a box whose register tiles are above the budget takes the strips)."""
import numpy as np
import pytest

from gragles2d_amd import _native as N
from gragles2d_amd import grainhdl as G

from .gpu_helpers import settings_for

pytestmark = pytest.mark.gpu


def _run(net, steps, ppg, gb, **kw):
    h = G.GrainHandler(settings_for(len(net), ppg, gb), **kw)
    h.set_simulation_parameter(net)
    h.step(steps)
    return h


def _same(a, b, ids):
    fa, fb = a.frame(), b.frame()
    for g in ids:
        assert fa.info[g].tobytes() == fb.info[g].tobytes(), g
        if fa.info[g]["exists"]:
            assert np.array_equal(fa.phi(g), fb.phi(g)) and np.array_equal(fa.idlocal(g), fb.idlocal(g)), g
            assert np.array_equal(fa.contour(g), fb.contour(g)), g


@pytest.mark.parametrize("prec", [N.PREC_FP64, N.PREC_FP32])
@pytest.mark.parametrize("n,ppg,gb,budget", [(30, 20, 7, 26000), (6, 60, 40, 70000)])
def test_one_grain_launches_under_a_budget_give_the_same_bits(prec, n, ppg, gb, budget):
    net = G.Network.generate(n, 970 + n)
    a = _run(net, 3, ppg, gb, precision=prec, batching=N.BATCH_PERGRAIN)
    b = _run(net, 3, ppg, gb, precision=prec, batching=N.BATCH_PERGRAIN, lds_budget=budget)
    _same(a, b, range(1, len(net) + 1))
