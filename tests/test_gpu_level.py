"""The level-set kernels at the sizes where their work splits change, against the oracle (the bar of
gpu_helpers: fields 1e-10, everything discrete exact) and against one-grain launches bit for bit.

Box sides around 64 (one bit word per row or two, one wave or four per grain, the tile of one wave
or two), around 128 (three bit words, the FP64 tile no longer fits LDS) and close to the largest side; a grain pinched to a point, whose contour passes saddles (walked, not ranked).
"""
import numpy as np
import pytest

from gragles2d_amd import _native as N
from gragles2d_amd import grainhdl as G

from .gpu_helpers import FIELD_EPS, compare_step, failures, make_pair

pytestmark = pytest.mark.gpu


def _parity(net, steps, ppg, gb, **kw):
    gpu, o = make_pair(net, ppg=ppg, gb=gb, oracle_threads=8, **kw)
    ids = range(1, len(net) + 1)
    worst, sides = 0.0, set()
    for t in range(steps):
        info = gpu.info_all()
        sides |= {info[g].xmax - info[g].xmin for g in ids if info[g].exists}
        gpu.step(1)
        assert o.step() == 0
        rep = compare_step(gpu, o, ids, field_eps=max(FIELD_EPS, 2 * worst))
        worst = max(worst, rep["_max_phi_err"])
        assert not failures(rep), (t, failures(rep))
    assert worst <= 1e-10
    return sides


@pytest.mark.parametrize("n,ppg,gb,lo,hi", [(40, 34, 9, 63, 65), (24, 80, 10, 126, 131)])
def test_box_sides_around_the_splits(n, ppg, gb, lo, hi):
    sides = _parity(G.Network.generate(n, 900 + n), 4, ppg, gb)
    assert min(sides) <= lo and max(sides) >= hi, sorted(sides)


def test_box_sides_around_the_splits_anisotropic():
    aniso = dict(research_mode=0, mobility_model=1, triple_point_drag=0.5 * 34 * 6 / 10.0, constant_sector_radius=3.0,
                 interpolating_sector_radius=2.0)
    sides = _parity(G.Network.generate(40, 940), 4, 34, 9, aniso=aniso)
    assert min(sides) <= 63 and max(sides) >= 65, sorted(sides)


def test_largest_box_sides():
    # two grains on a 480-point domain: boxes close to the largest side, eight bit words per row
    two = [np.array([[0, 0], [0.5, 0], [0.5, 1], [0, 1], [0, 0]], float),
           np.array([[0.5, 0], [1, 0], [1, 1], [0.5, 1], [0.5, 0]], float)]
    sides = _parity(G.Network.from_polygons(two), 2, 340, 10)
    assert max(sides) >= 480, sorted(sides)


def _hourglass(pinch):
    """Grain 1: two triangles that meet in the domain's centre; grains 2 and 3 fill the rest."""
    c = 0.5
    glass = np.array([[0, 0], [1, 0], [c + pinch, c], [1, 1], [0, 1], [c - pinch, c], [0, 0]], float)
    left = np.array([[0, 0], [c - pinch, c], [0, 1], [0, 0]], float)
    right = np.array([[1, 0], [1, 1], [c + pinch, c], [1, 0]], float)
    return G.Network.from_polygons([glass, left, right])


@pytest.mark.parametrize("pinch", [0.0, 0.004, 0.02])
@pytest.mark.parametrize("ppg", [25, 70])
def test_pinched_grain(pinch, ppg):
    _parity(_hourglass(pinch), 4, ppg, 7)


@pytest.mark.parametrize("prec", [N.PREC_FP64, N.PREC_FP32])
@pytest.mark.parametrize("n,ppg,gb", [(40, 34, 9), (20, 80, 10)])
def test_one_grain_launches_give_the_same_bits(prec, n, ppg, gb):
    # a one-grain launch sizes its LDS for that grain's side, a batched one for the bucket's largest
    net = G.Network.generate(n, 950 + n)
    s = G.default_settings(number_of_particles=len(net), number_of_points_per_grain=ppg, domain_border_size=gb,
                           convolution_mode=2, is_isotropic_network=1, analysis_timestep=1)
    a = G.GrainHandler(s, precision=prec, batching=N.BATCH_FUSED)
    b = G.GrainHandler(s, precision=prec, batching=N.BATCH_PERGRAIN)
    for h in (a, b):
        h.set_simulation_parameter(net)
        h.step(3)
    fa, fb = a.frame(), b.frame()
    for g in range(1, len(net) + 1):
        assert fa.info[g].tobytes() == fb.info[g].tobytes(), g
        if fa.info[g]["exists"]:
            assert np.array_equal(fa.phi(g), fb.phi(g)) and np.array_equal(fa.idlocal(g), fb.idlocal(g))
            assert np.array_equal(fa.contour(g), fb.contour(g))
            assert np.array_equal(fa.neighbours(g)[1], fb.neighbours(g)[1])
