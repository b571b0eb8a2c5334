"""The kernel source compiled for the CPU against the HIP emulation with failures
and stream order (tests/emu_faults/hip; nothing fails unless it is armed), once a
session, and its child processes under AddressSanitizer and UBSan."""
import functools
import os
import shutil
import subprocess
import sys
import tempfile

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
SRC = os.path.join(os.path.dirname(HERE), "htr-solver_amd", "csrc", "htr_all.hip")


@functools.lru_cache(maxsize=None)
def _build():
    folder = tempfile.TemporaryDirectory(prefix="htr_emu_")
    out = os.path.join(folder.name, "libhtr_emu.so")
    cmd = ["g++", "-x", "c++", "-std=c++20", "-O1", "-g", "-fPIC", "-shared", "-I", os.path.join(HERE, "emu_faults"),
           "-ffp-contract=off", "-Wno-unused-function", "-Wno-attributes",
           "-fsanitize=address,undefined", "-fno-sanitize-recover=undefined", "-o", out, SRC, "-lpthread"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-4000:]
    return out, folder


def run_child(script, *args):
    """The CASE lines that a child process prints."""
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    asan = subprocess.run(["gcc", "-print-file-name=libasan.so"], capture_output=True, text=True).stdout.strip()
    env = dict(os.environ, HTR_AMD_LIBRARY=_build()[0], LD_PRELOAD=asan, ASAN_OPTIONS="detect_leaks=0",
               UBSAN_OPTIONS="print_stacktrace=1")
    r = subprocess.run([sys.executable, os.path.join(HERE, script), *args], env=env, capture_output=True, text=True,
                       timeout=900)
    assert r.returncode == 0, (r.stdout[-2000:], r.stderr[-3000:])
    assert "ERROR: AddressSanitizer" not in r.stderr and "runtime error" not in r.stderr, r.stderr[-3000:]
    return [ln for ln in r.stdout.splitlines() if ln.startswith("CASE ")]
