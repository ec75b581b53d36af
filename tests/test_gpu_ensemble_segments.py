"""Default z segments of an ensemble: chosen for all members together (the segment length whose work
items end earliest on the persistent grid), unless a member's are set by amd_zSegments or
fe_ens_set_segments.  Every segmentation computes each cell by the same operations (levels that start
a segment to a rounding, test_gpu_segments), so states are compared bit for bit with plain runs of
the segments that the ensemble reports."""
import numpy as np
import pytest

import fe_py
from test_gpu_ensemble import _member, _plain_run

pytestmark = pytest.mark.gpu


def _fill(ens, shapes, tmp_path, **over):
    ps = [dict(fe_py.CFG0, Nx=nx, Ny=ny, Nz=nz, NtBatch=1, **over) for nx, ny, nz in shapes]
    for k, p in enumerate(ps):
        _member(ens, p, tmp_path / "e", seed=200 + k)
    return ps


# members, and the segments on 256 work-groups: one small member spreads as a lone run does; 16 of
# 8 tiles fill the chip in one round of 24 levels; many members take whole columns
@pytest.mark.parametrize("shapes,nseg", [([(64, 64, 48)], 12), ([(64, 64, 48)] * 16, 2), ([(64, 32, 4)] * 3, 1)])
def test_choice(shapes, nseg, tmp_path):
    ens = fe_py.Ensemble()
    ens.clear()
    try:
        _fill(ens, shapes, tmp_path)
        before = [ens.info(k)["nseg"] for k in range(len(shapes))]
        assert before == [nseg] * len(shapes), before
        ens.steps(1)
        assert [ens.info(k)["nseg"] for k in range(len(shapes))] == before
    finally:
        ens.clear()


def test_set_segments_stay_when_members_come(tmp_path):
    ens = fe_py.Ensemble()
    ens.clear()
    try:
        ps = _fill(ens, [(64, 24, 22)], tmp_path, amd_zSegments=3)
        ps += _fill(ens, [(70, 19, 33), (64, 64, 48)], tmp_path)
        ens.set_segments(2, 5)
        ens.steps(1)
        ps += _fill(ens, [(40, 40, 17)], tmp_path)
        zseg = [8, None, 10, None]
        for k, z in enumerate(zseg):
            assert z is None or ens.info(k)["nseg"] == -(-ps[k]["Nz"] // z), (k, ens.info(k))
        ens.steps(1)
        info = [ens.info(k) for k in range(4)]
        for k, (p, seed, n) in enumerate(zip(ps, (200, 200, 201, 200), (2, 2, 2, 1))):
            ref, ust = _plain_run(dict(p, amd_zSegments=0), tmp_path / "p", seed=seed, nsteps=n, nseg=info[k]["nseg"])
            assert np.array_equal(ens.state(k), ref), (k, info[k])
            assert np.array_equal(ens.ustar(k), ust), k
    finally:
        ens.clear()
