"""cad_m1bcgs_noalloc, the solve on device-resident arrays that allocates
nothing, against the solve drop-in vf_m1bcgs_ on the same recorded Poisson
systems: the solution bit for bit, BNORM, XNORM and ITER equal.  Two calls in
a row, the second on a smaller grid and on another stream, with the work
arrays filled with NaN (the solve must clear what it reads), and the
refusals of sizes beyond the limit (no device call is made for those)."""
import numpy as np
import pytest

import fixtures as fx

WORK = ("DD", "XW", "YY", "R0", "RR", "PP", "AP", "AE")


def _params(case):
    st = fx.static(case)
    p = fx.deck_params(st["DECK"])
    p.update(fx.solver_params(st))
    return {k: p[k] for k in ("cgpara", "cgepsa", "cgepsr", "cgdiv", "icgtyp", "icgmax")}


def _flat(a):
    return np.asfortranarray(a).ravel(order="F")


@pytest.mark.gpu
def test_noalloc_solve_equals_the_dropin(pkg):
    import torch
    cap = pkg.capi
    calls = [("corner3d", fx.steps("corner3d")[-1], None), ("tiny", fx.steps("tiny")[-1], "side")]
    for case, s, stream_kind in calls:
        ps = fx.step(case, s)["ps_in"]
        p = _params(case)
        shape = ps["AD"].shape
        x0 = np.zeros(shape, order="F")
        print(f"vf_m1bcgs_ {case} step {s} {shape}", flush=True)
        xr, bnr, xnr, itr = cap.m1bcgs(ps, ps["INDC"], x0=x0, **p)
        dev = {k: torch.from_numpy(_flat(ps[k]).copy()).cuda() for k in cap.MATRIX}
        dev["INDC"] = torch.from_numpy(_flat(ps["INDC"]).astype(np.int32)).cuda()
        dev["X0"] = torch.from_numpy(_flat(x0).copy()).cuda()
        for k in WORK:
            dev[k] = torch.full((int(np.prod(shape)),), float("nan"), dtype=torch.float64,
                                device="cuda")
        torch.cuda.synchronize()
        side = torch.cuda.Stream() if stream_kind == "side" else None
        ptrs = {k: v.data_ptr() for k, v in dev.items()}
        print(f"cad_m1bcgs_noalloc {case} step {s} stream={stream_kind}", flush=True)
        rc, bn, xn, it = cap.m1bcgs_noalloc(ptrs, shape, stream=None if side is None else
                                            side.cuda_stream, **p)
        assert rc == 0, cap.lib().cad_last_error().decode()
        x = dev["X0"].cpu().numpy().reshape(shape, order="F")
        assert it == itr, (case, it, itr)
        assert bn == bnr and xn == xnr, (case, bn, bnr, xn, xnr)
        assert np.array_equal(x, xr), (case, np.abs(x - xr).max())
        assert it == int(fx.step(case, s)["ps_out"]["ICGITR"][0])


@pytest.mark.gpu
def test_noalloc_solve_with_and_without_room_for_the_packed_sweeps(pkg):
    """The packed sweeps' operands take 64 bytes a cell of their padded walks: a
    long grid fits the reserved part, 300 x 300 lines of 6 cells (40 padded) do
    not and use the natural-layout sweeps.  Both equal the drop-in bit for bit,
    one after the other on the same scratch."""
    import torch
    cap = pkg.capi
    for shape in ((66, 18, 30), (6, 300, 300), (130, 50, 12)):
        rs = np.random.default_rng(shape[0])
        indc = np.full(shape, -1, np.int32, order="F")
        indc[1:-1, 1:-1, 1:-1] = np.where(rs.random([n - 2 for n in shape]) < 0.9, 0, -1)
        on = indc == 0
        mat = {k: np.zeros(shape, order="F") for k in cap.MATRIX}
        for a, (lo, up) in enumerate((("ALI", "AUI"), ("ALJ", "AUJ"), ("ALK", "AUK"))):
            mat[lo][...] = np.where(on & np.roll(on, 1, axis=a), -rs.random(shape), 0.0)
            mat[up][...] = np.roll(mat[lo], -1, axis=a)
        mat["AD"][...] = 6.5
        mat["BB"][...] = np.where(on, rs.standard_normal(shape), 0.0)
        p = dict(cgpara=0.95, icgtyp=1, cgepsa=1e-15, cgepsr=1e-10, cgdiv=1e30, icgmax=500)
        x0 = np.zeros(shape, order="F")
        print(f"vf_m1bcgs_ {shape}", flush=True)
        xr, bnr, xnr, itr = cap.m1bcgs(mat, indc, x0=x0, **p)
        dev = {k: torch.from_numpy(_flat(mat[k]).copy()).cuda() for k in cap.MATRIX}
        dev["INDC"] = torch.from_numpy(_flat(indc)).cuda()
        for k in ("X0",) + WORK:
            dev[k] = torch.zeros(int(np.prod(shape)), dtype=torch.float64, device="cuda")
        torch.cuda.synchronize()
        print(f"cad_m1bcgs_noalloc {shape}", flush=True)
        rc, bn, xn, it = cap.m1bcgs_noalloc({k: v.data_ptr() for k, v in dev.items()}, shape, **p)
        assert rc == 0, cap.lib().cad_last_error().decode()
        assert itr > 0 and (it, bn, xn) == (itr, bnr, xnr), (shape, it, itr, bn, bnr, xn, xnr)
        assert np.array_equal(dev["X0"].cpu().numpy().reshape(shape, order="F"), xr), shape


def test_noalloc_refuses_grids_beyond_the_limit(pkg):
    cap = pkg.capi
    ptrs = {k: 4096 for k in list(cap.MATRIX) + ["X0", "INDC"] + list(WORK)}
    n = cap.NOALLOC_MAX_CELLS
    rc, *_ = cap.m1bcgs_noalloc(ptrs, (256, 128, n // (256 * 128) + 1))
    assert rc == -1
    assert "CAD_NOALLOC_MAX_CELLS" in cap.lib().cad_last_error().decode()
    rc, *_ = cap.m1bcgs_noalloc(ptrs, (3, 8, 8))
    assert rc == -1
    bad = dict(ptrs, DD=0)
    rc, *_ = cap.m1bcgs_noalloc(bad, (8, 8, 8))
    assert rc == -1 and "null" in cap.lib().cad_last_error().decode()
