"""The index ranges of the block responses' products, without a GPU: every
operand and result of a wide map's table, tree and top products lies in the
buffer that is carved for it, for every number of blocks up to the capacity."""
import os
import subprocess

EXE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp", "block_ranges_check")


def test_products_stay_inside_their_buffers():
    assert os.path.exists(EXE), "build with make -C parode_amd/csrc"
    out = subprocess.run([EXE], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0, out.stdout + out.stderr
