"""What library calls that fail on the way leave behind, on the CPU: the kernel
source compiled against the HIP emulation with failures and stream order
(tests/emu_faults/hip), under AddressSanitizer and UBSan."""
import os

import pytest

from emu_build import run_child

pytestmark = pytest.mark.slow


@pytest.mark.parametrize("which", ["side_streams", "teno_memory", "rhs_memory", "mixture_upload"])
def test_failed_calls(which):
    cases = run_child(os.path.join("emu_faults", "run_faults.py"), which)
    assert any(ln.startswith("CASE " + which) for ln in cases)
