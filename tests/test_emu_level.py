"""The level-set kernels in the CPU emulator (tests/emu: real barriers, exact-size LDS, ASan and
UBSan) at the box sides where their work splits change: around 64 (one bit word per row or two, one
wave or four per grain) and above 128, isotropic and anisotropic, against the oracle."""
import os
import subprocess

import pytest

EMU = os.path.join(os.path.dirname(os.path.abspath(__file__)), "emu")
ENV = dict(os.environ, ASAN_OPTIONS="detect_leaks=1:abort_on_error=0", UBSAN_OPTIONS="halt_on_error=1")


@pytest.mark.parametrize("args", [
    "5 3 1023 9 34 0.0",                       # sides around 64
    "5 3 1022 9 34 0.0 0 0 0.0 1 0 2 1",       # the same, Read-Shockley energies and sectors
    "5 2 1023 9 34 0.0 1",                     # FP32
    "3 2 1024 20 128 0.0",                     # above 128
])
def test_emulated_box_sides_around_the_splits(args):
    r = subprocess.run(["make", "-s", "-C", EMU], capture_output=True, text=True, timeout=900)
    assert r.returncode == 0, r.stderr[-4000:]
    r = subprocess.run([os.path.join(EMU, "emu_parity")] + args.split(), capture_output=True, text=True, timeout=900, env=ENV)
    out = r.stdout + r.stderr
    assert "ERROR: AddressSanitizer" not in out and "runtime error" not in out, out[-4000:]
    assert r.returncode == 0 and "PARITY OK" in out, out[-3000:]
