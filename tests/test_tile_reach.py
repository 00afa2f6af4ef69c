"""gam_set_tile changes the launches of every tiled stage that a step launches on its own,
the column kernels of large blocks among them."""
import subprocess

import pytest

from tests.emu import build_emu


@pytest.mark.parametrize("defs", [(), ("EMF_COL_MIN=0",)], ids=["edges", "edge_columns"])
def test_tiles_reach_the_launches(defs):
    r = subprocess.run([build_emu.build(defs=defs, main="tile_reach.cpp")], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr
