"""Implicit chemistry with a wave per cell on the CPU (tests/emu/run_chem.py): its
LDS indexing under AddressSanitizer, its wave operations and barriers, and its
results against the oracle."""
import os
import subprocess
import sys

import pytest

from test_emu_kernels import HERE, emu_lib  # noqa: F401

pytestmark = pytest.mark.slow


@pytest.mark.parametrize("args", [("air", "0x10", "0x11", "0", "1"), ("cells30", "0x10", "0x11"), ("cells30", "0"),
                                  ("cells30", "1")])
def test_wave_kernel_in_bounds(emu_lib, args):  # noqa: F811
    asan = subprocess.run(["gcc", "-print-file-name=libasan.so"], capture_output=True, text=True).stdout.strip()
    env = dict(os.environ, HTR_AMD_LIBRARY=emu_lib, LD_PRELOAD=asan, ASAN_OPTIONS="detect_leaks=0",
               UBSAN_OPTIONS="print_stacktrace=1")
    r = subprocess.run([sys.executable, os.path.join(HERE, "emu", "run_chem.py"), *args], env=env, capture_output=True,
                       text=True, timeout=900)
    assert r.returncode == 0, (r.stdout[-2000:], r.stderr[-3000:])
    assert "ERROR: AddressSanitizer" not in r.stderr and "runtime error" not in r.stderr, r.stderr[-3000:]
    assert len([ln for ln in r.stdout.splitlines() if ln.startswith("CASE ")]) == len(args) - 1
