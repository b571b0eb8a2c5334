"""Diffusion along one direction at the edges of the blocks' lines, on the CPU
(tests/emu/run_lines.py), bit for bit against the oracle."""
import os

import pytest

from emu_build import run_child

pytestmark = pytest.mark.slow


def test_diffusion_lines_at_edges():
    assert len(run_child(os.path.join("emu", "run_lines.py"))) == 26
