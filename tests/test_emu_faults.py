"""What library calls that fail on the way leave behind, on the CPU: the kernel
source compiled against the HIP emulation with failures and stream order
(tests/emu_faults/hip), under AddressSanitizer and UBSan."""
import os
import shutil
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
SRC = os.path.join(os.path.dirname(HERE), "htr-solver_amd", "csrc", "htr_all.hip")

pytestmark = pytest.mark.slow


@pytest.fixture(scope="module")
def fault_lib(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    out = str(tmp_path_factory.mktemp("faults") / "libhtr_faults.so")
    cmd = ["g++", "-x", "c++", "-std=c++20", "-O1", "-g", "-fPIC", "-shared", "-I", os.path.join(HERE, "emu_faults"),
           "-ffp-contract=off", "-Wno-unused-function", "-Wno-attributes",
           "-fsanitize=address,undefined", "-fno-sanitize-recover=undefined", "-o", out, SRC, "-lpthread"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-4000:]
    return out


@pytest.mark.parametrize("which", ["side_streams", "teno_memory", "rhs_memory", "mixture_upload"])
def test_failed_calls(fault_lib, which):
    asan = subprocess.run(["gcc", "-print-file-name=libasan.so"], capture_output=True, text=True).stdout.strip()
    env = dict(os.environ, HTR_AMD_LIBRARY=fault_lib, LD_PRELOAD=asan, ASAN_OPTIONS="detect_leaks=0",
               UBSAN_OPTIONS="print_stacktrace=1")
    r = subprocess.run([sys.executable, os.path.join(HERE, "emu_faults", "run_faults.py"), which], env=env,
                       capture_output=True, text=True, timeout=900)
    assert r.returncode == 0, (r.stdout[-2000:], r.stderr[-3000:])
    assert "ERROR: AddressSanitizer" not in r.stderr and "runtime error" not in r.stderr, r.stderr[-3000:]
    assert any(ln.startswith("CASE " + which) for ln in r.stdout.splitlines())
