"""Diffusion along one direction at the edges of the blocks' lines, on the CPU
(tests/emu/run_lines.py), bit for bit against the oracle."""
import os
import subprocess
import sys

import pytest

from test_emu_kernels import HERE, emu_lib  # noqa: F401

pytestmark = pytest.mark.slow


def test_diffusion_lines_at_edges(emu_lib):  # noqa: F811
    asan = subprocess.run(["gcc", "-print-file-name=libasan.so"], capture_output=True, text=True).stdout.strip()
    env = dict(os.environ, HTR_AMD_LIBRARY=emu_lib, LD_PRELOAD=asan, ASAN_OPTIONS="detect_leaks=0",
               UBSAN_OPTIONS="print_stacktrace=1")
    r = subprocess.run([sys.executable, os.path.join(HERE, "emu", "run_lines.py")], env=env, capture_output=True,
                       text=True, timeout=900)
    assert r.returncode == 0, (r.stdout[-2000:], r.stderr[-3000:])
    assert "ERROR: AddressSanitizer" not in r.stderr and "runtime error" not in r.stderr, r.stderr[-3000:]
    assert len([ln for ln in r.stdout.splitlines() if ln.startswith("CASE ")]) == 26
