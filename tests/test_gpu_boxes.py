"""The standalone batch's strip products at the edges of their tiles, lines and launches against the
oracle's convolution.

The bound: four products of up to n terms each, summed in blocks of eight, on fields of magnitude
F: with |H| <= sqrt 2 and the symbol's 1 / n^2 an element of the result carries at most
4 * (8 + n / 8) * 2^-53 relative rounding of sums no larger than 4 F, below 2e-13 F at n = 512; 1e-12 F leaves room for the oracle's own error.
"""
import numpy as np
import pytest

from .test_gpu_fft import DT, R, _batch

pytestmark = pytest.mark.gpu

# one tile / one line more or less than 4, 8, 16; a wave's second, third and fourth tile; a second
# round of sixteen tiles; strips beyond the default LDS limit; the largest side
SIDES = [1, 3, 4, 5, 7, 8, 9, 15, 17, 63, 65, 129, 193, 255, 257, 300, 511, 512]


@pytest.mark.parametrize("mode", [0, 1, 2])
def test_strip_products_match_the_oracle(mode):
    from oracle.pyoracle import convolve
    rng = np.random.default_rng(40 + mode)
    fields = [rng.uniform(-0.05, 0.05, (n, n)) + 0.02 for n in SIDES]
    rc, got = _batch(fields, mode)
    assert rc == 0
    for f, g in zip(fields, got):
        err = float(np.max(np.abs(g - convolve(f, mode, DT, R))))
        print(f"mode {mode} n {f.shape[0]}: max|diff| {err:.2e}", flush=True)
        assert err <= 1e-12 * 0.07
