"""Z segments of a stage launch start at their first level: what a level takes over from the one
below (p', the z fluxes through the lower face, SGS fluxes, rho K_m, eddy viscosities) is formed by
the segment's set-up.  Stage tendencies of launches split into segments -- two levels, the shortest,
to the largest, with short last segments -- against the unsplit launch, over every family of kernels
(flat and terrain-following, lateral halo storage, with and without a surface layer, prognostic TKE
and Smagorinsky, dry and moist, partial tiles).

Both form every value from the same operands by the same source expressions, so levels that start
no segment are equal bit for bit; at a segment's first level an instance of the compiler may fuse
one multiply-add otherwise, one rounding of 6e-8 in a term, bounded by 1e-6 of the field maximum.
"""
import numpy as np
import pytest

import fe_py
from test_topography import CLOSURES, hill, write_topo

pytestmark = pytest.mark.gpu
NH = 3

CASES = {
    "dry": (dict(fe_py.CFG0, Nx=70, Ny=19, Nz=23), False, (2, 6, 11)),
    "dry-no-surface": (dict(fe_py.CFG0, Nx=64, Ny=9, Nz=16, surflayerSelector=0), False, (2, 8)),
    "moist": (dict(fe_py.CFG2, Nx=65, Ny=12, Nz=21, d_zeta=60.0), True, (3, 10)),
    "smagorinsky": (dict(fe_py.CFG0, Nx=40, Ny=17, Nz=18, TKESelector=0), False, (2, 9)),
    "hill": (dict(fe_py.CFG0, Nx=66, Ny=18, Nz=20), False, (3, 10)),
    "hill-moist": (dict(fe_py.CFG0, Nx=66, Ny=18, Nz=20, **CLOSURES["moist"][0]), True, (2, 7)),
    "hill-smagorinsky": (dict(fe_py.CFG0, Nx=66, Ny=18, Nz=20, TKESelector=0), False, (4,)),
    "halo": (dict(fe_py.CFG0, Nx=64, Ny=24, Nz=16, amd_haloBuffer=1), False, (2, 8)),
}


@pytest.mark.parametrize("case", list(CASES))
def test_segments_start_at_their_first_level(case, tmp_path):
    params, moist, segs = CASES[case]
    if case.startswith("hill"):
        h = hill(params["Nx"], params["Ny"], 20.0, 60.0, 100.0)
        params = dict(params, d_xi=20.0, d_eta=20.0, d_zeta=20.0, topoFile=write_topo(str(tmp_path / "topo.bin"), h))

    def run(nseg):
        m = fe_py.Model(dict(params, NtBatch=1, amd_zSegments=nseg), str(tmp_path / f"s{nseg}"))
        try:
            assert (nseg == 1) == ("z-segments" not in m.L.fe_kernel_info().decode())
            fe_py.turbulent_state((m.array("hydroFlds"), m.array("sgstkeScalars")), seed=31)
            if moist:
                fe_py.moist_state(m, seed=32)
            m.upload()
            out = {}
            for st in (0, 2):
                m.build_frhs(st)
                for key in ("hydroFldsFrhs", "sgstkeScalarsFrhs", "moistScalarsFrhs"):
                    if m.array(key) is not None:
                        out[key, st] = m.interior(m.array(key)).astype(np.float64)
            return out
        finally:
            m.close()

    ref = run(1)
    nz = params["Nz"]
    for nseg in segs:
        got = run(nseg)
        zlen = -(-nz // nseg)
        zlen += zlen % 2
        starts = set(range(zlen, nz, zlen))
        assert starts
        for k, r in ref.items():
            d = np.abs(got[k] - r)
            assert np.isfinite(r).all() and np.isfinite(got[k]).all(), (case, nseg, k)
            assert np.all(d.max(axis=(1, 2, 3)) <= 1e-6 * np.abs(r).max(axis=(1, 2, 3))), (case, nseg, k, d.max(axis=(1, 2, 3)))
            levels = set(int(i[-1]) for i in np.argwhere(d > 0))
            assert levels <= starts, (case, nseg, k, sorted(levels), sorted(starts))
