"""The pipelined MILU sweeps (one launch per sweep, wavefront tiles of 8x8
lines) against the hyperplane schedule (one launch per plane I+J+K) and the
reference.

Both schedules evaluate every cell's recurrence on the same operands in the same
order, so the Poisson solution, the iteration count and every field after whole
steps must agree bit for bit between them; against the reference the solver's
usual bar applies (same ITR, PT to 1e-10 relative).  The grids cover one tile,
ragged tiles in J and K, and (buildings tank) many tiles with obstacles and a
free surface, so tiles with no active cell and partial I ranges occur.
"""
import numpy as np
import pytest

import fixtures as fx
import pyoracle as po
from helpers import assert_close

pytestmark = pytest.mark.gpu

TOL = 1.0e-10
CASES = ["tiny", "beach_small", "corner3d"]


def _params(st, rec):
    p = fx.deck_params(st["DECK"])
    p.update(fx.solver_params(st))
    p["dtnow"] = float(rec["DTNOW"][0])
    keys = ("rho0", "grz0", "anu0", "dtnow", "scmvp", "flower", "fupper", "plower", "cgpara",
            "cgepsa", "cgepsr", "cgdiv", "icgtyp", "icgmax", "wbub", "idrop")
    return {k: p[k] for k in keys if k in p}


def _state(rec, bcf):
    a = {k: rec[k] for k in ("UU", "VV", "WW", "PP", "FF", "BCU", "BCV", "BCW", "BCP", "NF", "INDC")}
    a["BCF"] = bcf
    return a


def _solve(pkg, st, r, schedule):
    numi, numj, numk = st["GGV"].shape
    with pkg.capi.Context(numi, numj, numk, st["INDB"].shape[1]) as c:
        c.set_params(**_params(st, r["v1_in"]))
        c.upload_static(st)
        c.upload_state(_state(r["v1_in"], r["f1_in"]["BCF"]))
        c.set_sweep_schedule(schedule)
        c.upload_matrix(r["ps_in"], r["ps_in"]["INDC"])
        info = c.vpsol()
        return info, c.download_pt()


PIPELINED = ["SWEEP_PIPELINED", "SWEEP_PIPELINED_8X8", "SWEEP_PIPELINED_16X4"]


@pytest.mark.parametrize("sched", PIPELINED)
@pytest.mark.parametrize("case", CASES)
def test_schedules_agree_on_reference_systems(pkg, case, sched):
    st = fx.static(case)
    for s in fx.steps(case):
        r = fx.step(case, s)
        print(f"case {case} step {s} {sched}", flush=True)
        ip, pp = _solve(pkg, st, r, getattr(pkg.capi, sched))
        ih, ph = _solve(pkg, st, r, pkg.capi.SWEEP_HYPERPLANE)
        for k in ("cgbnrm", "cgxnrm", "icgitr"):
            assert ip[k] == ih[k], (k, ip[k], ih[k])
        assert np.array_equal(pp, ph), f"{case} step {s}: PT differs between schedules"
        assert ip["icgitr"] == int(r["ps_out"]["ICGITR"][0])
        assert_close(f"{case} step {s} PT", pp, r["ps_out"]["PT"], TOL)


def _run_steps(pkg, lay, state, flags, schedule, nsteps):
    ni, nj, nk = lay.shape
    with pkg.capi.Context(ni, nj, nk, lay.numb) as c:
        p = lay.params()
        c.set_params(**{k: v for k, v in p.items() if k in c.params})
        c.upload_static(lay.static_arrays())
        c.upload_state(state)
        c.init_state(lay.deck.wvlvl, lay.deck.uini, flags)
        c.set_sweep_schedule(schedule)
        infos = [c.step() for _ in range(nsteps)]
        return infos, c.download_state(), c.download_pt()


@pytest.mark.parametrize("sched", PIPELINED)
@pytest.mark.parametrize("shape", [(48, 40, 36), (70, 19, 45)])
def test_schedules_agree_over_steps(pkg, shape, sched):
    ni, nj, nk = shape
    case = pkg.configs.buildings_tank(ni, nj, nk, nbuild=6, seed=3, eps_r=1.0e-10,
                                      name=f"buildings_{ni}x{nj}x{nk}")
    lay = pkg.layout.from_text(case.deck)
    state = lay.raw_state()
    case.ic(lay.XX, lay.ZZ, lay.NF0, state)
    print(f"buildings {shape} {sched}", flush=True)
    ip, sp, pp = _run_steps(pkg, lay, dict(state), 0, getattr(pkg.capi, sched), 4)
    ih, sh, ph = _run_steps(pkg, lay, dict(state), 0, pkg.capi.SWEEP_HYPERPLANE, 4)
    for k in ("icgitr", "cgbnrm", "cgxnrm", "fsum", "fcut", "nums"):
        assert [i[k] for i in ip] == [i[k] for i in ih], k
    assert all(i["icgitr"] > 0 for i in ip)
    assert np.array_equal(pp, ph), "PT differs between schedules"
    for k in sp:
        assert np.array_equal(sp[k], sh[k]), f"{k} differs between schedules"


ALL_SCHEDULES = PIPELINED + ["SWEEP_HYPERPLANE"]


def _milu_check(pkg, mat, indc, prm, sched, ys):
    ni, nj, nk = mat["AD"].shape
    with pkg.capi.Context(ni, nj, nk, 0) as c:
        c.set_params(**prm)
        c.set_sweep_schedule(getattr(pkg.capi, sched))
        c.upload_matrix(mat, indc)
        assert c.milu_factor() == 1
        outs = [c.milu_apply(y) for y in ys]
    dd, ok = po.mzdcmp(mat, indc, prm["cgpara"], prm["icgtyp"])
    assert ok == 1
    for y, x in zip(ys, outs):
        ref = po.mzminv(mat, dd, y, indc)
        bad = np.flatnonzero((x != ref).ravel(order="F"))
        assert bad.size == 0, f"{sched}: {bad.size} cells differ, first at {bad[:5]}"


@pytest.mark.parametrize("sched", ALL_SCHEDULES)
@pytest.mark.parametrize("case", CASES)
def test_milu_apply_bitexact_with_oracle(pkg, case, sched):
    """x = M^-1 y on the reference's Poisson matrices equals the serial MILU
    sweeps of the oracle (vf_mzdcmp.f, vf_mzfrwd.f, vf_mzbkwd.f) bit for bit."""
    st = fx.static(case)
    rs = np.random.default_rng(7)
    for s in fx.steps(case)[:2]:
        r = fx.step(case, s)
        print(f"case {case} step {s} {sched}", flush=True)
        mat = r["ps_in"]
        prm = _params(st, r["v1_in"])
        ys = [mat["BB"], rs.standard_normal(mat["AD"].shape)]
        _milu_check(pkg, mat, mat["INDC"], prm, sched, ys)


@pytest.mark.parametrize("sched", ALL_SCHEDULES)
def test_milu_apply_bitexact_many_tiles(pkg, sched):
    """The same on a buildings tank with obstacles and a free surface: many
    tiles, ragged edges, empty tiles and partial I ranges."""
    case = pkg.configs.buildings_tank(70, 38, 45, nbuild=6, seed=3, eps_r=1.0e-10, name="b70")
    lay = pkg.layout.from_text(case.deck)
    state = lay.raw_state()
    case.ic(lay.XX, lay.ZZ, lay.NF0, state)
    ni, nj, nk = lay.shape
    with pkg.capi.Context(ni, nj, nk, lay.numb) as c:
        p = lay.params()
        c.set_params(**{k: v for k, v in p.items() if k in c.params})
        c.upload_static(lay.static_arrays())
        c.upload_state(state)
        c.init_state(lay.deck.wvlvl, lay.deck.uini, 0)
        c.predictor()
        c.vpcoef()
        mat = c.download_matrix()
        indc = c.download_state()["INDC"]
    prm = {k: v for k, v in p.items() if k in ("cgpara", "icgtyp", "cgepsa", "cgepsr", "cgdiv", "icgmax")}
    rs = np.random.default_rng(11)
    _milu_check(pkg, mat, indc, prm, sched, [mat["BB"], rs.standard_normal(mat["AD"].shape)])


@pytest.mark.parametrize("shape", [(4, 3, 3), (9, 16, 4), (14, 17, 9), (21, 2, 40), (37, 49, 5), (600, 11, 6),
                                   (301, 21, 13), (33, 30, 46), (20, 44, 67), (130, 9, 33)])
def test_packed_sweeps_bitexact_with_oracle(pkg, shape):
    """The default schedule's packed sweeps at the edges of their tiles (16 x 4
    and 16 x 8 lines, stages of 8 steps, one and two walking waves a
    workgroup), on matrices with random couplings and activity: whole lines
    and tiles without an active cell, activity that ends anywhere in a stage,
    values on inactive cells of the right-hand side and the matrix that must
    not be read.  M^-1 y equals the oracle's serial sweeps bit for bit, twice in
    a row (the second call's mailboxes hold the first one's entries)."""
    ni, nj, nk = (n + 2 for n in shape)
    rs = np.random.default_rng(ni * 131 + nj)
    indc = np.full((ni, nj, nk), -1, np.int32, order="F")
    act = rs.random(shape) < 0.8
    act[:, rs.random(shape[1]) < 0.2, :] = False
    act[:, :, shape[2] * 3 // 4 + 1:] = False
    act[: shape[0] // 5] = False
    act[shape[0] // 2, shape[1] // 2, 0] = True
    indc[1:-1, 1:-1, 1:-1] = np.where(act, 0, -1)
    on = indc == 0
    mat = {k: np.zeros((ni, nj, nk), order="F") for k in pkg.capi.MATRIX}
    for a, (lo, up) in enumerate((("ALI", "AUI"), ("ALJ", "AUJ"), ("ALK", "AUK"))):
        w = -rs.random((ni, nj, nk))
        back = np.roll(on, 1, axis=a)
        mat[lo][...] = np.where(on & back, w, 0.0)
        mat[up][...] = np.roll(mat[lo], -1, axis=a)
    mat["AD"][...] = 6.5
    mat["BB"][...] = rs.standard_normal((ni, nj, nk))
    for k in ("AUI", "ALJ", "AD"):      # never read on inactive cells
        mat[k][1:-1, 1:-1, 1:-1][~act] = rs.standard_normal(int((~act).sum()))
    prm = dict(cgpara=0.95, icgtyp=1, cgepsa=1e-15, cgepsr=1e-10, cgdiv=1e30, icgmax=500)
    y = rs.standard_normal((ni, nj, nk))
    print(f"packed sweeps {shape}", flush=True)
    _milu_check(pkg, mat, indc, prm, "SWEEP_PIPELINED", [y, mat["BB"], y])


@pytest.mark.parametrize("shape", [(2, 2, 200), (3, 3, 400)])
def test_default_schedule_on_a_tall_column(pkg, shape):
    """A column much taller than wide is a chain of tiles with next to no walk, on
    which the packed sweeps take 1.4 times the 64-line tiles' time: the default
    schedule takes the latter there, and equals the fixed tile shapes bit for bit.
    (The bar of 1.15 lies between; the runs of one schedule differ by 1 %.)"""
    ni, nj, nk = (n + 2 for n in shape)
    indc = np.full((ni, nj, nk), -1, np.int32, order="F")
    indc[1:-1, 1:-1, 1:-1] = 0
    on = indc == 0
    mat = {k: np.zeros((ni, nj, nk), order="F") for k in pkg.capi.MATRIX}
    for a, (lo, up) in enumerate((("ALI", "AUI"), ("ALJ", "AUJ"), ("ALK", "AUK"))):
        mat[lo][...] = np.where(on & np.roll(on, 1, axis=a), -1.0, 0.0)
        mat[up][...] = np.where(on & np.roll(on, -1, axis=a), -1.0, 0.0)
    mat["AD"][...] = 6.5
    mat["BB"][...] = np.random.default_rng(5).standard_normal((ni, nj, nk))
    lay = pkg.layout.from_text(pkg.configs.dam_break(*shape, col_x=0.01, col_z=0.01).deck)
    ms, out = {}, {}
    with pkg.capi.Context(ni, nj, nk, lay.numb) as c:
        c.upload_static(lay.static_arrays())
        c.upload_state(lay.raw_state())
        c.set_params(cgpara=0.95, icgtyp=1, cgepsa=1e-15, cgepsr=1e-10, cgdiv=1e30, icgmax=500)
        c.upload_matrix(mat, indc)
        for name in ("SWEEP_PIPELINED", "SWEEP_PIPELINED_8X8", "SWEEP_PIPELINED_16X4"):
            print(f"tall column {shape} {name}", flush=True)
            c.set_sweep_schedule(getattr(pkg.capi, name))
            c.milu_factor()
            out[name] = c.milu_apply(mat["BB"])
            c.time_minv(5)
            ms[name] = sorted(c.time_minv(20) for _ in range(5))[2]
    print(ms, flush=True)
    assert all(np.array_equal(o, out["SWEEP_PIPELINED"]) for o in out.values())
    assert ms["SWEEP_PIPELINED"] <= 1.15 * min(ms.values()), ms
