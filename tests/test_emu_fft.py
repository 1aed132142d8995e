"""The FFT engine (k_conv_fft) in the CPU emulator: FP32 steps with a Laplace symbol or with the engine
asked for run it always, FP64 steps where the lds_budget is too small for the strip products."""
import os
import re
import subprocess

import pytest

from .test_emu_limits import EMU, ENV, limits  # noqa: F401


def test_every_form_matches_the_oracle(limits):  # noqa: F811
    limits("engine")


@pytest.mark.parametrize("cmode", [0, 1])
def test_fp64_steps_whose_strips_are_above_the_budget(limits, cmode):  # noqa: F811
    # boxes of 30 to 62 points under 16000 bytes: the largest take the FFT with global slots
    limits(f"budget 6 2 1001 7 20 0 0 16000 {cmode}")


@pytest.mark.parametrize("net,engine,cmode,pergrain", [
    ("6 2 1001 7 20", 0, 0, 0), ("6 2 1001 7 20", 0, 1, 0), ("6 2 1001 7 20", 2, 2, 0),  # half spectra in LDS
    ("6 2 1001 7 20", 0, 0, 1), ("6 2 1001 7 20", 2, 2, 1),
    ("6 2 3 40 60", 0, 0, 0),                                                             # sides 150-226: global slots
])
def test_fp32_steps(limits, net, engine, cmode, pergrain):  # noqa: F811
    # everything discrete that the FP32 run is held to, and the areas: within 1e-5 of the oracle's
    r = subprocess.run([os.path.join(EMU, "emu_parity")] + f"{net} 0.0 1 {pergrain} 0.0 1 {engine} {cmode}".split(),
                       capture_output=True, text=True, timeout=900, env=ENV)
    out = r.stdout + r.stderr
    assert "ERROR: AddressSanitizer" not in out and "runtime error" not in out, out[-4000:]
    assert r.returncode == 0 and "PARITY OK" in out, out[-3000:]
    areas = [float(x) for x in re.findall(r"max rel dvol (\S+)", out)]
    assert len(areas) == 2 and max(areas) <= 1e-5, areas
