"""The library at its limits in the CPU emulator (tests/emu: real barriers, exact-size LDS, ASan and
UBSan)."""
import os
import subprocess

import pytest

EMU = os.path.join(os.path.dirname(os.path.abspath(__file__)), "emu")
ENV = dict(os.environ, ASAN_OPTIONS="detect_leaks=1:abort_on_error=0", UBSAN_OPTIONS="halt_on_error=1")


@pytest.fixture(scope="module")
def limits():
    r = subprocess.run(["make", "-s", "-C", EMU], capture_output=True, text=True, timeout=900)
    assert r.returncode == 0, r.stderr[-4000:]

    def run(args):
        r = subprocess.run([os.path.join(EMU, "emu_limits")] + args.split(), capture_output=True, text=True, timeout=900, env=ENV)
        out = r.stdout + r.stderr
        assert "ERROR: AddressSanitizer" not in out and "runtime error" not in out, out[-4000:]
        assert r.returncode == 0 and "LIMITS OK" in out, out[-3000:]
    return run


@pytest.mark.parametrize("args", [
    "6 2 1001 7 20 0",        # FP64, sides up to 62: the register tiles alone would take 34.9 KB of 24.6
    "6 2 1001 7 20 1",        # FP32
    "6 2 1001 7 20 1 0 20000",
    "6 2 1001 7 20 0 1",      # anisotropic
    "2 1 7 9 90 0",           # sides 142 and 145 under 44.5 KB: the strips
])
def test_lds_budget_is_kept_and_nothing_it_allowed_is_refused(limits, args):
    limits("budget " + args)


@pytest.mark.parametrize("args", [
    "64 3 16 128 2",    # one strip of eight there, more work items than workgroups
    "100 1 40 64 0",
    "20 5 16 256 1",    # one strip of sixteen, a workgroup per work item
])
def test_batch_spreads_over_the_dies_whatever_max_n(limits, args):
    limits("batch " + args)


def test_fft_workspace_is_there_only_where_the_fft_runs(limits):
    limits("workspace")
