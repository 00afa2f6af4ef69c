"""gam_get_work's face velocities are the last step's, whatever came after it that did not
step: the step fills those its EMFs read, the call the rest, from that step's
predictor state and geometry.  The same operations, the same bits."""
import numpy as np
import pytest

from kaiju_amd import configs
from tests.helpers import say


@pytest.mark.gpu
@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("what", ["geometry", "capture", "packed_capture", "halted", "halted_replay"])
def test_face_velocities_of_the_last_step(what, precision):
    from kaiju_amd.ensemble import Ensemble
    from kaiju_amd.gamera import GamApp, gen_corners
    spec = configs.blast_wave((12, 9, 5), precision=precision)
    say(f"[vf] {what} precision {precision}")
    app = GamApp(spec)
    app.InitModel()
    assert app.steps(3) == 0
    if what.startswith("halted"):
        c = app.get_clock()
        c.dt0 = 1e6 * c.dt
        app.set_clock(c)
        assert app.steps(1) == 1
    if what != "geometry":
        want = app.get_work(2)
    else:
        with GamApp(spec) as twin:
            twin.InitModel()
            assert twin.steps(3) == 0
            want = twin.get_work(2)
    assert np.abs(want).max() > 0
    xyz = gen_corners(spec)
    xyz[..., 0] *= 1.0 + 0.3 * xyz[..., 1]
    app.set_corners(np.asfortranarray(xyz))
    if what == "halted":
        assert app.steps(2) == 1
    if what in ("geometry", "halted"):
        got = app.get_work(2)
        app.close()
    else:
        with Ensemble([spec], tune=False, nsteps=2, apps=[app], packed=what == "packed_capture") as ens:
            if what == "halted_replay":
                assert ens.run(2) == 1
            got = app.get_work(2)
    assert np.array_equal(got, want)


def test_face_velocities_on_cpu_emulation():
    from tests.emu import build_emu
    from tests.test_emu import _run
    assert " passed" in _run(build_emu.build(asan=False), {}, "velocities_of", 300, "test_gpu_face_velocities.py")
