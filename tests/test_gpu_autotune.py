"""The autotuned tilings of the block passes, through the library's own classes:
what is timed is stored for the method and the sample type of the solve that
looks it up."""
import os
import subprocess

import pytest

pytestmark = pytest.mark.gpu

EXE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp", "block_schedule_check")


def test_a_tuned_tiling_is_found_by_the_solve_it_was_timed_for():
    assert os.path.exists(EXE), "build with make -C parode_amd/csrc"
    out = subprocess.run([EXE], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0, out.stdout + out.stderr
