"""LG_GEMM_TILE_WIDTH, read once per process, makes 256-row tiles 128 (the kernel of gemm_fast.hip), 192 or 256 features wide: the same bits in
every layout and epilogue, since every output above 256 rows is one sum in the order of k."""
import json
import os
import subprocess
import sys

import pytest

from tests import gemm_width_child

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.parametrize("width", ["2", "3", "4"])
def test_the_width_of_256_row_tiles_changes_no_bit(dev, width):
    child = subprocess.run([sys.executable, "-m", "tests.gemm_width_child"], cwd=ROOT, env=dict(os.environ, LG_GEMM_TILE_WIDTH=width),
                           stdout=subprocess.PIPE, stderr=subprocess.PIPE, text=True, timeout=100)
    assert child.returncode == 0, child.stderr[-2000:]
    assert json.loads(child.stdout.strip().splitlines()[-1]) == gemm_width_child.outputs()
