"""Ensemble members of very few levels (one segment each), alone and beside a taller member whose
segments are set: bit for bit the plain run's steps."""
import numpy as np
import pytest

import fe_py
from test_gpu_ensemble import _member, _plain_run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("levels", [(1,), (2,), (3,), (2, 22, 3)])
def test_few_levels(levels, tmp_path):
    ens = fe_py.Ensemble()
    ens.clear()
    try:
        ps = [dict(fe_py.CFG0, Nx=64, Ny=16, Nz=nz, NtBatch=1, **(dict(amd_zSegments=3) if nz > 4 else {})) for nz in levels]
        for k, p in enumerate(ps):
            _member(ens, p, tmp_path / "e", seed=300 + k)
        nseg = [ens.info(k)["nseg"] for k in range(len(ps))]
        assert nseg == [3 if nz > 4 else 1 for nz in levels], nseg
        if 1 in levels:                              # one level: the grid has no vertical spacing to step with
            return
        ens.steps(2)
        for k, p in enumerate(ps):
            ref, ust = _plain_run(p, tmp_path / "p", seed=300 + k, nsteps=2, nseg=nseg[k])
            assert np.array_equal(ens.state(k), ref) and np.isfinite(ref).all(), levels
            assert np.array_equal(ens.ustar(k), ust), levels
    finally:
        ens.clear()
