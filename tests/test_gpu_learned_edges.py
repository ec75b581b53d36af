"""The learned closure's network and correction kernels where their tiles and wraps are at an edge:
a grid with fewer 64-cell tiles than work-groups, one that is ragged in every direction and ends in
a partial tile, and one whose work-groups take several tiles each.  The fused inference gives the
unfused path's bits, and the corrected tendency is the numpy restatement's to the rounding of the
tendencies it is the difference of (FP32: 1e-5 of their scale, a hundred units in the last place)."""
import os

import numpy as np
import pytest

import fe_mlp
import fe_py
from test_gpu_learned_sgs import NH, _model

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(64, 8, 16), (67, 11, 19), (150, 61, 33)], ids=lambda s: "x".join(map(str, s)))
def test_network_and_correction_at_edges(tmp_path, shape, repo):
    nx, ny, nz = shape
    m, p = _model(tmp_path, seed=23, Nx=nx, Ny=ny, Nz=nz)
    s = fe_py.LearnedSGS()
    try:
        s.clear()
        s.load(os.path.join(repo, "fasteddy-model_amd", "sgs_cbl20m.npz"))
        ncell = nx * ny * nz
        s.enable(True, gate=-1.0)                # no cell passes: the TKE closure's tendency
        m.build_frhs(2)
        gated = m.array("hydroFldsFrhs").copy()
        s.enable(False)
        out = {}
        for fused in (True, False):
            s.set_fused(fused)
            s.enable(True, gate=6.0)
            m.build_frhs(2)
            tau, mask = s.last(ncell)
            P = (nx + 31) // 32 * 32
            out[fused] = (tau.copy(), mask.copy(), m.array("hydroFldsFrhs").copy())
            emitted = s.emitted(9 * nz * ny * P).reshape(9, nz, ny, P)[..., :nx].copy()
            assert s.stats()[0] == ncell and s.stats()[1] == mask.sum()
            s.enable(False)
        print(f"{nx}x{ny}x{nz}: cells passing {out[True][1].mean():.3f}")
        assert 0.0 < out[True][1].mean() < 1.0
        for a, b in zip(out[True], out[False]):
            assert np.count_nonzero(a != b) == 0
        tau, mask, F = out[True]
        corr = fe_mlp.sgs_correction(tau.reshape(9, nz, ny, nx), mask.reshape(nz, ny, nx), emitted, m.getf("dXi"),
                                     m.getf("dYi"), m.getf("dZi"), np.ones(nz))
        dF = (F - gated)[1:5, NH:-NH, NH:-NH, NH:-NH].astype(np.float64)
        want = corr.transpose(0, 3, 2, 1)
        assert np.abs(dF - want).max() <= 1e-5 * np.abs(gated[1:5]).max()
        assert np.all(dF[:, (want == 0.0).all(axis=0)] == 0.0)
    finally:
        s.set_fused(True)
        s.clear()
        m.close()
