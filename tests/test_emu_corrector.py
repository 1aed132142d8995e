"""The velocity corrector on contours that it does not stage in LDS (k_sectors' arc lengths by one lane,
k_aniso's reads in place), in the CPU emulator against the oracle; one network has shorter ones beside them."""
import pytest

from .test_emu_limits import limits  # noqa: F401


@pytest.mark.parametrize("args", ["6 2 15 9 80 0.3 1 0", "5 2 14 9 90 0 4 1"])
def test_corrector_on_long_contours(limits, args):  # noqa: F811
    limits("corrector " + args)
