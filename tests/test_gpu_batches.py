"""ggx_convolve_boxes with max_n far above the sides, and with more strips than a launch has workgroups:
the bits of the call whose max_n is the largest side (a strip's products do not know max_n)."""
import numpy as np
import pytest

from .test_gpu_fft import DT, R, _batch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("count,lo,hi,max_n", [(40, 3, 33, 512), (3000, 3, 40, 128), (20000, 2, 9, 16), (7, 65, 130, 300)])
@pytest.mark.parametrize("mode", [0, 1, 2])
def test_max_n_above_the_sides_gives_the_same_bits(mode, count, lo, hi, max_n):
    rng = np.random.default_rng(count + mode)
    fields = [rng.uniform(-0.05, 0.05, (n, n)) for n in rng.integers(lo, hi + 1, count)]
    rc, got = _batch(fields, mode, max_n=max_n)
    rd, want = _batch(fields, mode)
    assert rc == 0 and rd == 0
    assert all(np.array_equal(a, b) for a, b in zip(got, want))


def test_more_strips_than_workgroups_match_the_oracle():
    from oracle.pyoracle import convolve
    rng = np.random.default_rng(77)
    fields = [rng.uniform(-0.05, 0.05, (n, n)) for n in rng.integers(1, 41, 6000)]
    rc, got = _batch(fields, 1, max_n=64)
    assert rc == 0
    for k in list(range(0, 6000, 61)) + [5999]:
        assert float(np.max(np.abs(got[k] - convolve(fields[k], 1, DT, R)))) <= 1e-12
