"""Implicit chemistry with a wave per cell on the CPU (tests/emu/run_chem.py): its
LDS indexing under AddressSanitizer, its wave operations and barriers, and its
results against the oracle."""
import os

import pytest

from emu_build import run_child

pytestmark = pytest.mark.slow


@pytest.mark.parametrize("args", [("air", "0x10", "0x11", "0", "1"), ("cells30", "0x10", "0x11"), ("cells30", "0")])
def test_wave_kernel_in_bounds(args):
    assert len(run_child(os.path.join("emu", "run_chem.py"), *args)) == len(args) - 1
