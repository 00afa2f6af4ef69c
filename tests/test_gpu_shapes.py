"""Kernels whose launch or algorithm depends on the block's extents, against the
oracle at the extents where they can go wrong: columns of several interfaces
per thread with a short last one, columns of a single interface, thin and
ragged boxes, and the two ways of a cell's volume (folded cells keep the
reference's quadrature).

One step: the FP64 parity bar, 1e-12 normwise.  Volumes and centres: sums of
1728 separately rounded terms on either side, 1728 x 2^-53 = 2e-13 each, so
1e-12 normwise."""
import os
import subprocess
import sys

import numpy as np
import pytest

import oracle
from kaiju_amd import configs
from tests.helpers import app_from_oracle, compare_state, relerr, say

TOL_STEP = 1e-12
TOL_METRIC = 1e-12


def _cases():
    bw = configs.blast_wave
    out = {
        "columns_of_4_ragged": bw((96, 72, 65)),
        "columns_thin_k": bw((17, 130, 9)),
        "columns_thin_i": bw((9, 40, 150), rmeth="8CENT", doBoris=True, Ca=6.0),
        "columns_hydro": bw((24, 90, 12), doMHD=False),
        "box_25d": configs.orszag_tang((61, 43, 1)),
        "box_flat_boris": configs.orszag_tang((130, 70, 3), doBoris=True, Ca=3.0),
    }
    for k, s in out.items():
        s.name = k
    return out


CASES = _cases()


@pytest.mark.gpu
@pytest.mark.parametrize("name", list(CASES))
def test_one_step(name):
    say(f"[shapes] {name}")
    oc = oracle.OracleCase(CASES[name])
    oc.step(1)
    with app_from_oracle(oc) as app:
        assert app.steps(2) == 0
        oc.step(2)
        e = compare_state(app, oc, 0)
        say(f"   {e}")
        assert max(e["Gas"], e["magFlux"], e["Bxyz"]) <= TOL_STEP, e
        assert abs(app.Model.dt - oc.m.dt) <= TOL_STEP * oc.m.dt


@pytest.mark.gpu
@pytest.mark.parametrize("amp", [0.2, 0.9])
@pytest.mark.parametrize("mirror", [False, True])
def test_volumes_of_skewed_and_folded_cells(amp, mirror):
    """Corners moved at random by up to amp cells: 0.2 leaves det J of one sign in most
    cells, 0.9 folds most of them.  mirror: left-handed cells."""
    say(f"[volumes] {amp} {mirror}")
    spec = configs.orszag_tang((12, 9, 7))
    oc = oracle.OracleCase(spec, setup=False)
    oc.gen_corners()
    rng = np.random.default_rng(17)
    xyz = oc.grid["xyz"]
    d = 2.0 * np.pi / 12
    xyz += amp * d * rng.uniform(-0.5, 0.5, size=xyz.shape)
    if mirror:
        xyz[..., 0] *= -1.0
    oc.metric()
    from kaiju_amd.gamera import GamApp
    with GamApp(spec) as app:
        app.set_corners(xyz)
        g = app.get_grid(only=("volume", "xyzcc", "face", "xfc"))
    for k in g:
        assert relerr(g[k], oc.grid[k]) <= TOL_METRIC, k
    vol, ref = g["volume"], oc.grid["volume"]
    assert np.max(np.abs(vol - ref) / ref) <= TOL_METRIC


def test_shapes_on_cpu_emulation():
    """The same checks on the CPU emulation of the kernels, in bounds under AddressSanitizer."""
    from tests.emu import build_emu
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    for asan, expr in ((False, "thin or 25d or volumes"), (True, "thin_k or 25d or volumes")):
        env = dict(os.environ, KAIJU_EMU_LIB=build_emu.build(asan=asan))
        if asan:
            env.update(LD_PRELOAD=build_emu.asan_runtime(), ASAN_OPTIONS="detect_leaks=0:abort_on_error=1")
        r = subprocess.run([sys.executable, "-m", "pytest", "-q", "-p", "no:cacheprovider", "-m", "gpu", os.path.abspath(__file__),
                            "-k", expr], cwd=root, env=env, capture_output=True, text=True, timeout=900)
        assert r.returncode == 0, r.stdout[-3000:] + r.stderr[-2000:]
