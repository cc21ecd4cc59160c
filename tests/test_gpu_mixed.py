"""The mixed form (CAD_PRECISION_MIXED): FP64 BiCGSTAB right-preconditioned by
an FP32 aggregation multigrid V-cycle, stopped on the true relative residual.

It is not bit-compatible with the reference (a different preconditioner, so a
different iterate), so it is judged by what the solve must deliver: the true
relative residual ||BB - A PT|| / ||BB|| at CGEPSR, recomputed in FP64, and
fields within 1e-6 relative of the reference's, the bound the mixed form is
held to.
"""
import numpy as np
import pytest

import fixtures as fx
from helpers import assert_close, assert_same_int, assert_vel_close

pytestmark = pytest.mark.gpu

CASES = ["tiny", "beach_small", "corner3d"]
KEYS = ("rho0", "grz0", "anu0", "scmvp", "flower", "fupper", "plower", "cgpara", "cgepsa",
        "cgepsr", "cgdiv", "icgtyp", "icgmax", "wbub", "idrop")
STATE = ("UU", "VV", "WW", "PP", "FF", "BCU", "BCV", "BCW", "BCP", "NF", "INDC")


def _ctx(pkg, st, dtnow, **extra):
    numi, numj, numk = st["GGV"].shape
    p = fx.deck_params(st["DECK"])
    p.update(fx.solver_params(st))
    c = pkg.capi.Context(numi, numj, numk, st["INDB"].shape[1])
    c.set_params(**{k: p[k] for k in KEYS}, dtnow=dtnow, precision=pkg.capi.PRECISION_MIXED, **extra)
    c.upload_static(st)
    return c, p


@pytest.mark.parametrize("case", CASES)
def test_mixed_solve_on_reference_systems(pkg, case):
    """The reference's own Poisson systems: true residual at CGEPSR in far
    fewer iterations than MILU-BiCGSTAB, PT within 1e-6 of the reference's."""
    st = fx.static(case)
    for s in fx.steps(case):
        r = fx.step(case, s)
        if "ps_in" not in r:
            continue
        print(f"{case} step {s}", flush=True)
        c, p = _ctx(pkg, st, float(r["v1_in"]["DTNOW"][0]))
        with c:
            a = {k: r["v1_in"][k] for k in STATE}
            a["BCF"] = r["f1_in"]["BCF"]
            c.upload_state(a)
            c.upload_matrix(r["ps_in"], r["ps_in"]["INDC"])
            info = c.vpsol()
            res = c.poisson_residual()
            pt = c.download_pt()
        ref_itr = int(r["ps_out"]["ICGITR"][0])
        print(f"  ITR {info['icgitr']} (reference {ref_itr}) true residual {res:.2e}", flush=True)
        # the stop test: ||r|| <= CGEPSR ||BB|| + CGEPSA (the reference's
        # structure, with the true residual in place of the preconditioned one)
        bn = info["cgbnrm"]
        assert res * bn <= (p["cgepsr"] * bn + p["cgepsa"]) * (1.0 + 1e-6), (s, res, bn)
        assert abs(info["cgxnrm"] - res) <= 1e-3 * res + 1e-30
        assert 0 < info["icgitr"] <= max(ref_itr, 20)
        assert_close(f"{case} step {s} PT", pt, r["ps_out"]["PT"], 1e-6)


def test_mixed_free_run_dam_break(pkg):
    """100 steps of the 64x16x48 dam break in the mixed form from the
    reference's initial state: flags equal and velocity, pressure and F
    within 1e-6 of the reference's step 100."""
    case = "dam_a"
    st = fx.static(case)
    r1 = fx.step(case, 1)
    c, _ = _ctx(pkg, st, float(r1["v1_in"]["DTNOW"][0]))
    with c:
        a = {k: r1["v1_in"][k] for k in STATE}
        a["BCF"] = r1["f1_in"]["BCF"]
        c.upload_state(a)
        worst = 0.0
        for s in range(1, 101):
            info = c.step()
            bn = info["cgbnrm"]
            worst = max(worst, c.poisson_residual() * bn / (1.0e-10 * bn + 1.0e-15))
        out = c.download_state()
    ref = fx.step(case, 100)["f1_out"]
    print(f"mixed dam break: worst residual / tolerance {worst:.3f}, last ITR {info['icgitr']}",
          flush=True)
    assert worst <= 1.0 + 1e-6
    assert_same_int("step 100 NF", out["NF"], ref["NF"])
    assert_vel_close("step 100 velocity", out, ref, 1e-6)
    for k in ("PP", "FF"):
        assert_close(f"step 100 {k}", out[k], ref[k], 1e-6)


@pytest.mark.parametrize("case", ["wave_open", "tdoor"])
def test_mixed_form_with_boundary_and_timer_door_models(pkg, tmp_path, case):
    """The mixed form under the models around the step: the wave flume with
    a radiation end (1000 steps) and the droplet deck with both TimerDoor
    models (300 steps), run from the deck through driver.run: flags equal and
    fields within 1e-6 of the reference's last step."""
    st = fx.static(case)
    tr = fx.trajectory(case)
    last = int(tr["STEP"][-1])
    deck = str(st["DECK"]) + f"\nFILE RSL STEP {last} {last} 1\n"
    if "FILE_MTB" in st:
        (tmp_path / "run.mtb").write_text(str(st["FILE_MTB"]))
    res = pkg.driver.run(deck, "run", tmp_path, precision=pkg.capi.PRECISION_MIXED)
    assert res["nnow"] == last
    rec = [r for r in pkg.rsl.read(tmp_path / "run.rsl")][1:][-1]
    ref = fx.step(case, last)["f1_out"]
    print(f"{case}: mixed run to step {last}", flush=True)
    assert_same_int(f"step {last} NF", rec["NF"], ref["NF"])
    assert_vel_close(f"step {last} velocity", rec, ref, 1e-6)
    for k in ("PP", "FF"):
        assert_close(f"step {last} {k}", rec[k], ref[k], 1e-6)


def test_mixed_falls_back_to_milu_bicgstab(pkg):
    """With the mixed form's own iterations capped at one, its solve cannot
    converge by itself: the reference's MILU-BiCGSTAB finishes it from the
    current iterate, to the true residual at CGEPSR, PT within 1e-6 of the
    reference's."""
    case = "corner3d"
    st = fx.static(case)
    s = fx.steps(case)[-1]
    r = fx.step(case, s)
    c, p = _ctx(pkg, st, float(r["v1_in"]["DTNOW"][0]))
    with c:
        a = {k: r["v1_in"][k] for k in STATE}
        a["BCF"] = r["f1_in"]["BCF"]
        c.upload_state(a)
        c.upload_matrix(r["ps_in"], r["ps_in"]["INDC"])
        c.set_krylov_cap(1)
        info = c.vpsol()
        res = c.poisson_residual()
        pt = c.download_pt()
        stats = c.mixed_stats()
    print(f"fallback: ITR {info['icgitr']} stats {stats} true residual {res:.2e}", flush=True)
    assert stats["fallbacks"] == 1 and stats["fallback_iters"] > 0
    assert info["icgitr"] == 1 + stats["fallback_iters"]
    bn = info["cgbnrm"]
    assert res * bn <= (p["cgepsr"] * bn + p["cgepsa"]) * (1.0 + 1e-6)
    assert_close(f"{case} step {s} PT", pt, r["ps_out"]["PT"], 1e-6)


# interior cells: whole solve in one workgroup with two rows of a colour a thread,
# six, four; levels above it, odd extents; a coarsest level beyond it (two
# lines and one line thick); over 2^20 cells; a half line just over 64 positions
SHAPES = [(8, 8, 8), (25, 16, 12), (32, 16, 8), (97, 21, 13), (40, 33, 37), (300, 2, 40), (2, 130, 70),
          (260, 70, 66), (129, 5, 4)]


@pytest.mark.parametrize("shape", SHAPES)
def test_mixed_solve_over_level_shapes(pkg, shape):
    """A Poisson system with a fixed value above a ragged surface, on grids whose
    levels end in each kind of coarsest solve: three solves in a row (the
    surface of the second is lower, the third is the first again) as captured
    iterations and, with kernel timing on, as launches of their own give the
    same bits; the true residual holds and no solve falls back.  Grids that
    coarsen need few iterations, which a wrong row, correction or restriction
    would not give."""
    ni, nj, nk = (n + 2 for n in shape)
    rs = np.random.default_rng(ni + nj)
    systems = []
    for level in (0.8, 0.5, 0.8):
        indc = np.full((ni, nj, nk), -1, np.int32, order="F")
        top = np.clip((level * shape[2] + rs.integers(-1, 2, shape[:2])).astype(int), 1, shape[2])
        indc[1:-1, 1:-1, 1:-1] = np.where(np.arange(shape[2]) < top[:, :, None], 0, -1)
        on = indc == 0
        mat = {k: np.zeros((ni, nj, nk), order="F") for k in pkg.capi.MATRIX}
        for a, (lo, up) in enumerate((("ALI", "AUI"), ("ALJ", "AUJ"), ("ALK", "AUK"))):
            mat[lo][...] = np.where(on & np.roll(on, 1, axis=a), -1.0, 0.0)
            mat[up][...] = np.where(on & np.roll(on, -1, axis=a), -1.0, 0.0)
        above = on & ~np.roll(on, -1, axis=2)
        mat["AD"][...] = np.where(on, above * 2.0 - sum(mat[k] for k in ("ALI", "AUI", "ALJ", "AUJ", "ALK", "AUK")), 0.0)
        mat["BB"][...] = np.where(on, rs.standard_normal((ni, nj, nk)), 0.0)
        systems.append((mat, indc))
    lay = pkg.layout.from_text(pkg.configs.dam_break(*shape, col_x=0.01, col_z=0.01).deck)
    outs = []
    for timing in (0, 1):
        with pkg.capi.Context(ni, nj, nk, lay.numb) as c:
            c.upload_static(lay.static_arrays())
            c.upload_state(lay.raw_state())
            c.set_params(cgpara=0.95, icgtyp=1, cgepsa=0.0, cgepsr=1e-10, cgdiv=1e30, icgmax=2000,
                         precision=pkg.capi.PRECISION_MIXED)
            c.set_kernel_timing(timing)
            for mat, indc in systems:
                print(f"mixed {shape} timing {timing}", flush=True)
                c.upload_matrix(mat, indc)
                info = c.vpsol()
                outs.append((info["icgitr"], c.poisson_residual(), c.download_pt()))
            assert c.mixed_stats()["fallbacks"] == 0, shape
    print(f"  ITR {[o[0] for o in outs]} residuals {[o[1] for o in outs]}", flush=True)
    for a, b in zip(outs[:3], outs[3:]):
        assert a[0] == b[0] and np.array_equal(a[2], b[2]), shape
        assert a[1] <= 1e-10 * (1 + 1e-6), (shape, a[1])
        if min(shape) >= 4:
            assert a[0] <= 24, (shape, a[0])
