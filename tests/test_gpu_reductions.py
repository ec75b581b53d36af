"""The device reductions over horizontal planes (profile statistics, state summary, slab means of
the large-scale forcing) at the shapes where their split over work-groups and four-cell groups can
go wrong: fewer cells than one work-group, rows that are not a multiple of four (or of a 128-byte
line) long, one row, many parts per level, more levels than there are work-groups to split.

Profiles, means and integrals are FP64 sums in another order than the numpy restatement's: two
orders of n terms differ by at most 2 n eps times the sum of the terms' magnitudes (n = 37 200
columns, 1.1e-16: 8e-12), so the bound is 1e-11 of the mean magnitude of what is summed -- not of
the sum, which cancels for the velocities.  The summary's extremes, locations and counts agree
exactly; planted NaN and Inf sit in the last, partial group of a row.  The forcing
through three steps against the FP64 oracle with the bound of test_gpu_parity (2e-3 of the change).
"""
import numpy as np
import pytest

import fe_profiles
import fe_py
import oracle_py
from test_gpu_parity import LSF_STRONG
from test_gpu_summary import _host_summary

pytestmark = pytest.mark.gpu
NH = 3



def _magnitudes(m):
    """Mean magnitudes of the terms behind the profile columns (largest over the levels), and of the
    summary's rows (per unit mass, raw)."""
    f = [m.interior(m.array("hydroFlds"))[k].astype(np.float64) for k in range(5)]
    f.append(m.interior(m.array("sgstkeScalars"))[0].astype(np.float64))
    if m.array("moistScalars") is not None:
        f += list(m.interior(m.array("moistScalars")).astype(np.float64))
    rho, (u, v, w, th) = f[0], [np.abs(x / f[0]) for x in f[1:5]]
    lev = lambda a: np.nanmax(a.mean(axis=(0, 1)))
    sq = lambda a, b: lev(a * b) + lev(a) * lev(b)
    e, q, l = [lev(np.abs(x / rho)) for x in f[5:8]] + [0.0] * (8 - len(f))
    cols = [lev(u), lev(v), lev(w), lev(th), sq(u, u), sq(u, w), sq(v, v), sq(v, w), sq(w, w),
            0.5 * (sq(u, u) + sq(v, v) + sq(w, w)), sq(th, w), e, q, l, 1.0, 1.0, 1.0]
    rows = [(rho, rho)] + [(x / rho, x) for x in f[1:5]] + [(np.ones(1), np.ones(1))] + [(x / rho, x) for x in f[5:]]
    ok = lambda a: np.abs(a[np.isfinite(a)])
    return np.array(cols), [(ok(a).mean(), ok(b).mean()) for a, b in rows]


def _compare(m, dev, ref, mags):
    dv = float(m.getf("dX")) * m.getf("dY") * m.getf("dZ") * m.geti("Nx") * m.geti("Ny") * m.geti("Nz")
    assert list(dev) == list(ref)
    for (row, r), (a, b) in zip(ref.items(), mags):
        d = dev[row]
        for c in ("max", "min"):
            assert np.float32(d[c]) == np.float32(r[c]), (row, c)
        for c in ("imax", "jmax", "kmax", "imin", "jmin", "kmin", "nan", "inf"):
            assert int(d[c]) == int(r[c]), (row, c, d[c], r[c])
        assert abs(d["mean"] - r["mean"]) <= 1e-11 * a, (row, d["mean"], r["mean"])
        if np.isfinite(r["integral"]):
            assert abs(d["integral"] - r["integral"]) <= 1e-11 * b * dv, (row, d["integral"], r["integral"])
        else:
            assert not np.isfinite(d["integral"]), row


SHAPES = [(5, 4, 6), (33, 3, 9), (130, 67, 5), (31, 96, 4), (200, 186, 7), (16, 12, 1100)]


@pytest.mark.parametrize("shape", SHAPES, ids=["x".join(map(str, s)) for s in SHAPES])
@pytest.mark.parametrize("moist", [False, True])
def test_profiles_and_summary(shape, moist, tmp_path):
    nx, ny, nz = shape
    base = fe_py.CFG2 if moist else fe_py.CFG0
    p = dict(base, Nx=nx, Ny=ny, Nz=nz, d_zeta=2.0 if nz > 100 else 20.0, dampingLayerDepth=20.0, NtBatch=1)
    m = fe_py.Model(p, str(tmp_path))
    try:
        fe_py.turbulent_state((m.array("hydroFlds"), m.array("sgstkeScalars")), seed=nx)
        if moist:
            fe_py.moist_state(m, seed=ny)
        m.upload()
        m.download()
        ref = fe_profiles.profiles(m.array("hydroFlds"), m.array("sgstkeScalars"), m.array("moistScalars"))
        got = m.profiles()
        cols, rows = _magnitudes(m)
        assert (np.abs(got - ref).max(axis=0) <= 1e-11 * cols).all()
        assert np.array_equal(m.profiles(), got)
        # p' of a plain upload is whatever the last batch left: zero here, on both sides
        _compare(m, m.state_summary(), _host_summary(m), rows)
        h = m.array("hydroFlds")
        h[1, NH + nx - 1, NH + ny - 1, NH] = np.nan
        h[4, NH + nx - 1, NH, NH + nz - 1] = np.inf
        m.upload()
        m.download()
        _compare(m, m.state_summary(), _host_summary(m), _magnitudes(m)[1])
    finally:
        m.close()


@pytest.mark.parametrize("shape", [(8, 8, 12), (33, 9, 10), (66, 50, 8)])
def test_slab_means(shape, tmp_path):
    nx, ny, nz = shape
    p = dict(fe_py.CFG2, Nx=nx, Ny=ny, Nz=nz, d_zeta=40.0, dt=0.05, NtBatch=3, lsf_horMnSubTerms=1, **LSF_STRONG)
    m = fe_py.Model(p, str(tmp_path))
    try:
        fe_py.turbulent_state((m.array("hydroFlds"), m.array("sgstkeScalars")), seed=5)
        fe_py.moist_state(m, seed=6)
        o = oracle_py.Oracle(p, 64)
        o.load_from_model(m)
        h0 = m.interior(m.array("hydroFlds")).astype(np.float64).copy()
        q0 = m.interior(m.array("moistScalars")).astype(np.float64).copy()
        m.L.fe_set_int(b"simTime_itRestart", 0)
        m.commence()
        o.steps(3)
        for name, oname, start in (("hydroFlds", "HYDRO", h0), ("moistScalars", "MOIST", q0)):
            g = m.interior(m.array(name)).astype(np.float64)
            r = m.interior(o.arr(oname)[:g.shape[0]])
            ax = (1, 2, 3)
            change = np.abs(r - start).max(axis=ax)
            assert (np.abs(g - r).max(axis=ax) <= 2e-3 * change + 1e-6 * np.abs(r).max(axis=ax)).all(), (name, shape)
        o.close()
    finally:
        m.close()
