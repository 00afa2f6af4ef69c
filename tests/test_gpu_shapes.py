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
    """The merged launches of small blocks, and the separate ones (the flux columns,
    and the EMF columns of large blocks where EMF_COL_MIN is 0)."""
    say(f"[shapes] {name}")
    oc = oracle.OracleCase(CASES[name])
    oc.step(1)
    with app_from_oracle(oc) as app, app_from_oracle(oc) as sep:
        assert app.steps(2) == 0
        sep.set_timing(True)
        assert sep.steps(2) == 0
        oc.step(2)
        for a in (app, sep):
            e = compare_state(a, oc, 0)
            say(f"   {e}")
            assert max(e["Gas"], e["magFlux"], e["Bxyz"]) <= TOL_STEP, e
            assert abs(a.Model.dt - oc.m.dt) <= TOL_STEP * oc.m.dt


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


@pytest.mark.gpu
@pytest.mark.parametrize("mkw", [{}, dict(precision=1, rmeth="8CENT", doBoris=True, Ca=6.0)], ids=["fp64", "fp32_8cent_boris"])
def test_large_block_of_periods(mkw):
    """A block large enough for the EMF columns (more than EMF_COL_MIN zones, no extent a
    multiple of 8) that repeats a small periodic block, with the same metrics (positions
    in multiples of 2^-44, so that whole periods add exactly), does what the small
    one does in its merged launches.  The same operations but for the absolute positions
    in the cell-centred field's sums: 6 terms of up to 205 cell sizes, 6 x 205 x 2^-53 =
    1.4e-13, twice a step for two steps: 1e-12 normwise.  FP32 bulk: 2^-24 and
    a few tens of operations in a chain, 1e-5."""
    from kaiju_amd.gamera import GamApp
    n, rep = (41, 33, 35), (4, 5, 5)
    say(f"[periods] {mkw}")
    tol = 1e-5 if mkw.get("precision") else 1e-12

    def tile(a, position=False, rep=rep):   # arrays with ghosts, faces one longer
        for ax in range(3):
            ng = (a.shape[ax] - n[ax]) // 2
            q = np.arange(n[ax] * rep[ax] + a.shape[ax] - n[ax]) - ng
            a = np.take(a, ng + q % n[ax], axis=ax)
            if position:   # components (x, y, z) along the 4th axis, unit period
                a[:, :, :, ax] += (q // n[ax]).reshape([-1 if d == ax else 1 for d in range(3)] + [1] * (a.ndim - 4))
        return np.asfortranarray(a)

    with GamApp(configs.blast_wave(n, **mkw)) as small:
        small.InitModel()
        pos = ("xyz", "xyzcc", "xfc")
        grid = {k: np.round(v * 2.0**44) / 2.0**44 if k in pos else v for k, v in small.get_grid().items()}
        small.set_grid({k: tile(v, k in pos, (1, 1, 1)) for k, v in grid.items()})   # ghost cells as the cells they repeat
        assert small.steps(1) == 0
        big_spec = configs.blast_wave(tuple(q * r for q, r in zip(n, rep)), **mkw)
        with GamApp(big_spec) as big:
            big.set_grid({k: tile(v, k in pos) for k, v in grid.items()})
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
                assert relerr(y[act], x[act]) <= tol


@pytest.mark.gpu
@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("n", [(9, 40, 2), (17, 6, 30)])
def test_ghosts_of_a_halted_step(n, precision):
    """A periodic fused step whose CalcDT halts leaves the ghost cells that its update
    skips as the separate calls leave them: the same copies and sums, the same bits."""
    from kaiju_amd.gamera import GamApp
    say(f"[halt] {n} precision {precision}")
    out = []
    for fused in (True, False):
        with GamApp(configs.blast_wave(n, precision=precision)) as app:
            app.InitModel()
            assert app.steps(2) == 0
            st = app.get_state(0)
            gas, c = st["Gas"], tuple(app.nG + q // 2 for q in n)
            gas[c + (1,)] = 1e12 * gas[c + (0,)]
            gas[c + (4,)] += 0.5 * 1e24 * gas[c + (0,)]
            app.put_state(0, st["time"], gas, st["magFlux"], st["Bxyz"])
            ts = app.Model.ts
            assert (app.steps(3) if fused else app.stepGamera(fused=False)) != 0
            assert app.Model.ts == ts + 1
            out.append(app.get_state(0))
    for q in ("Gas", "magFlux", "Bxyz"):
        assert np.array_equal(out[0][q], out[1][q], equal_nan=True), q


EMU_EXPR = {"all": "one_step and (thin or 25d) or volumes or halted", "asan": "one_step and 25d or volumes or halted", "cols": "one_step and not ragged"}


@pytest.mark.parametrize("kind", list(EMU_EXPR))
def test_shapes_on_cpu_emulation(kind, tmp_path):
    """The same checks on the CPU emulation of the kernels, in bounds under
    AddressSanitizer; cols: the EMF columns at every size."""
    from tests.emu import build_emu
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    lib = build_emu.build(asan=kind == "asan") if kind != "cols" else str(tmp_path / "libgamera_emu.so")
    env = dict(os.environ, KAIJU_EMU_LIB=lib)
    if kind == "asan":
        env.update(LD_PRELOAD=build_emu.asan_runtime(), ASAN_OPTIONS="detect_leaks=0:abort_on_error=1")
    if kind == "cols":
        subprocess.run([build_emu._cxx(), "-std=c++17", "-O1", "-fPIC", "-shared", "-DGAM_EMU", "-DEMF_COL_MIN=0", "-ffp-contract=off",
                        "-fno-fast-math", "-fsanitize=address", "-fno-omit-frame-pointer", "-x", "c++", "-I",
                        os.path.join(root, "include"), "-I", build_emu.CSRC, "-I", build_emu.HERE,
                        os.path.join(build_emu.CSRC, "gam_api.hip"), "-o", lib], check=True)
        env.update(LD_PRELOAD=build_emu.asan_runtime(), ASAN_OPTIONS="detect_leaks=0:abort_on_error=1")
    r = subprocess.run([sys.executable, "-m", "pytest", "-q", "-p", "no:cacheprovider", "-m", "gpu", os.path.abspath(__file__),
                        "-k", EMU_EXPR[kind]], cwd=root, env=env, capture_output=True, text=True, timeout=900)
    assert r.returncode == 0, r.stdout[-3000:] + r.stderr[-2000:]
