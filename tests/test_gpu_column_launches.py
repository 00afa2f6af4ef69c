"""The separate launches of a step, with any tiles, and the merged ones of small blocks: the
same operations in the same order, so the same bits; background field, Boris
correction, boundaries, ring average and learned correction included.

Small blocks take the merged launches by themselves and the separate ones (k_vf, k_emf,
k_emf_jcol, k_flux, k_flux_col) under stage timers.  A build with EMF_COL_MIN=0 runs the
I and K edges on k_emf_col there, which only large blocks do otherwise."""
import dataclasses

import numpy as np
import pytest

import oracle
from kaiju_amd import configs
from tests.helpers import DIPOLE, DevF32, app_from_oracle, relerr, say, small_cases
from tests.test_gpu_parity import TILE_SETS

CASES = {s.name: s for s in small_cases()}


def _same_bits(oc, steps):
    with app_from_oracle(oc) as a:
        st = a.steps(steps)
        s1, w1 = a.get_state(0), [a.get_work(w) for w in range(3)]
        for tiles in ({}, *TILE_SETS):
            with app_from_oracle(oc) as b:
                b.set_timing(True)
                for stage, t in tiles.items():
                    b.set_tile(stage, *t)
                assert b.steps(steps) == st
                s2 = b.get_state(0)
                for k in ("Gas", "magFlux", "Bxyz"):
                    assert np.array_equal(s1[k], s2[k]), (k, tiles)
                for w in range(3):
                    assert np.array_equal(w1[w], b.get_work(w)), (w, tiles)
                assert a.Model.dt == b.Model.dt


@pytest.mark.gpu
@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("name", list(CASES))
def test_separate_and_merged_launches_agree(name, precision):
    say(f"[launches] {name} precision {precision}")
    s = CASES[name]
    _same_bits(oracle.OracleCase(dataclasses.replace(s, model=dataclasses.replace(s.model, precision=precision))), 2)


@pytest.mark.gpu
@pytest.mark.parametrize("precision", [0, 1])
def test_separate_and_merged_launches_agree_on_the_axis_block(precision):
    from tests.test_ring import _hatched
    say(f"[launches] axis block precision {precision}")
    _same_bits(_hatched((16, 12, 32), precision=precision)[1], 2)


@pytest.mark.gpu
@pytest.mark.parametrize("mkw", [{}, dict(precision=1, rmeth="8CENT", doBoris=True, Ca=6.0)], ids=["fp64", "fp32_8cent_boris"])
@pytest.mark.parametrize("what", ["background", "correction"])
def test_large_block_of_periods_with_background_or_correction(what, mkw):
    """A block of 41 x 33 x 35 cells with its own arrays of a background field or a
    correction, and one of 4 x 5 x 5 copies of it (over EMF_COL_MIN zones): positions apart,
    the copies are exact, so the bars are those of the plain blocks: 6 terms of up to 205
    cell sizes in the cell-centred field, 1.4e-13, twice a step for two steps, 1e-12
    normwise; FP32 bulk a few tens of 2^-24 in a chain, 1e-5."""
    from kaiju_amd.gamera import GamApp
    n, rep = (41, 33, 35), (4, 5, 5)
    say(f"[periods] {what} {mkw}")
    tol = 1e-5 if mkw.get("precision") else 1e-12

    def tile(a, position=False, rep=rep):   # arrays with ghosts, faces one longer
        for ax in range(3):
            ng = (a.shape[ax] - n[ax]) // 2
            q = np.arange(n[ax] * rep[ax] + a.shape[ax] - n[ax]) - ng
            a = np.take(a, ng + q % n[ax], axis=ax)
            if position:
                a[:, :, :, ax] += (q // n[ax]).reshape([-1 if d == ax else 1 for d in range(3)] + [1] * (a.ndim - 4))
        return np.asfortranarray(a)

    def flat(o):   # (i, j, k, 8) to the device layout, i fastest of the cells
        return np.ascontiguousarray(o.transpose(2, 1, 0, 3)).reshape(-1, 8)

    spec = configs.blast_wave(n, **mkw)
    with GamApp(spec) as small:
        small.InitModel()
        pos = ("xyz", "xyzcc", "xfc")
        grid = {k: np.round(v * 2.0**44) / 2.0**44 if k in pos else v for k, v in small.get_grid().items()}
        small.set_grid({k: tile(v, k in pos, (1, 1, 1)) for k, v in grid.items()})
        big_spec = configs.blast_wave(tuple(q * r for q, r in zip(n, rep)), **mkw)
        with GamApp(big_spec) as big:
            big.set_grid({k: tile(v, k in pos) for k, v in grid.items()})
            if what == "background":
                small.background_dipole(DIPOLE["M0"], DIPOLE["xc"], DIPOLE["bu"])
                bg = small.get_background()
                small.set_background({k: tile(v, rep=(1, 1, 1)) for k, v in bg.items()})
                big.set_background({k: tile(v) for k, v in bg.items()})
            else:
                o = np.random.default_rng(8).normal(size=small.G + (8,))
                ds, db = DevF32(flat(o)), DevF32(flat(tile(o)))
                small.set_correction(ds.ptr, 0.05)
                big.set_correction(db.ptr, 0.05)
            assert small.steps(1) == 0
            for w in (0, 1):
                st = small.get_state(w)
                big.put_state(w, st["time"], *[tile(st[q]) for q in ("Gas", "magFlux", "Bxyz")])
            big.set_clock(small.get_clock())
            big._sync_model()
            assert small.steps(2) == 0
            assert big.steps(2) == 0
            assert abs(big.Model.dt - small.Model.dt) <= tol * small.Model.dt
            g = big_spec.nG
            xs, ys = small.get_state(0), big.get_state(0)
            for q in ("Gas", "magFlux", "Bxyz"):
                x, y = tile(xs[q]), ys[q]
                act = tuple(slice(g, d - g) for d in x.shape[:3])
                e = relerr(y[act], x[act])
                say(f"   {q}: {e:.1e}")
                assert e <= tol
            if what == "correction":
                small.set_correction(None)
                big.set_correction(None)
                ds.free()
                db.free()


@pytest.mark.parametrize("kind", ["edges", "edge_columns"])
def test_launches_on_cpu_emulation(kind):
    """edge_columns: with AddressSanitizer, the corrected steps too."""
    from tests.emu import build_emu
    from tests.test_emu import _run
    expr = "agree and (bw or cyl or axis or 25d or exten or nolfm)"
    if kind == "edges":
        assert " passed" in _run(build_emu.build(asan=False), {}, expr, 900, "test_gpu_column_launches.py")
        return
    lib = build_emu.build(asan=True, defs=("EMF_COL_MIN=0",))
    env = {"LD_PRELOAD": build_emu.asan_runtime(), "ASAN_OPTIONS": "detect_leaks=0:abort_on_error=1"}
    assert " passed" in _run(lib, env, "agree and (dipole or axis or odd or thin or 25d)", 900, "test_gpu_column_launches.py")
    assert " passed" in _run(lib, env, "corrected_step", 900, "test_learned.py")
