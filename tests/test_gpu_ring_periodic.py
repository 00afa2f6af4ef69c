"""The ring average with six periodic faces (a handle's default boundaries): the fused
step restores the field about the axis (RingFlux2FieldFix, gridutils.F90:298-300) after
its boundary pass as the separate calls do: the same operations, the same bits."""
import numpy as np
import pytest

from tests.helpers import app_from_oracle, say


@pytest.mark.gpu
@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("n,chunks", [((16, 12, 32), (8, 16)), ((11, 10, 24), (6,))])
def test_ringed_periodic_block_fused_step_equals_separate_calls(n, chunks, precision):
    from tests.test_ring import _hatched
    say(f"[ring] six periodic faces {n} chunks {chunks} precision {precision}")
    _, oc = _hatched(n, precision=precision, chunks=chunks)
    with app_from_oracle(oc) as a, app_from_oracle(oc) as b:
        for x in (a, b):
            x.set_bcs(("periodic",) * 6)
            assert x.get_ring() == chunks
        for _ in range(2):
            assert a.stepGamera(fused=True) == b.stepGamera(fused=False)
        for w in (0, 1):
            sa, sb = a.get_state(w), b.get_state(w)
            for k in ("Gas", "magFlux", "Bxyz"):
                assert np.array_equal(sa[k], sb[k]), (w, k)
        assert a.Model.dt == b.Model.dt and a.Model.ts == b.Model.ts


def test_ringed_periodic_block_on_cpu_emulation():
    from tests.emu import build_emu
    from tests.test_emu import _run
    assert " passed" in _run(build_emu.build(asan=False), {}, "ringed", 300, "test_gpu_ring_periodic.py")
