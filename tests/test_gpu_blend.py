"""Blending weights of the hybrid advection schemes (b_hyb, TKEAdvSelector_b_hyb,
moistureAdvSelectorQv_b): kernels compiled for one weight of every field run where the three agree,
kernels for any weights elsewhere.  Stage tendencies of both against the CPU oracle with the
tolerance of test_gpu_parity (1e-5 of the field maximum from FP64, or twice the FP32 oracle's own
deviation), at whole tiles, partial tiles in x and y and a grid narrower than a tile; and an
ensemble that mixes members of both kinds against plain runs, bit for bit.
"""
import numpy as np
import pytest

import fe_py
from test_gpu_parity import check_tendencies, make, make_moist

pytestmark = pytest.mark.gpu

WEIGHTS = [(0.0, 0.0, 0.0), (0.4, 0.4, 0.4), (0.0, 0.7, 0.0), (0.3, 0.3, 0.9), (1.0, 0.0, 0.5)]


@pytest.mark.parametrize("b,be,bq", WEIGHTS)
@pytest.mark.parametrize("shape,moist,sqv", [((64, 8, 12), False, 3), ((70, 19, 13), False, 3), ((20, 13, 9), False, 3),
                                             ((65, 9, 12), True, 3), ((64, 16, 11), True, 2)])
def test_blending_weights(shape, moist, sqv, b, be, bq, tmp_path):
    nx, ny, nz = shape
    over = dict(Nx=nx, Ny=ny, Nz=nz, b_hyb=b, TKEAdvSelector_b_hyb=be)
    if moist:
        p = dict(fe_py.CFG2, d_zeta=60.0, moistureAdvSelectorQv=sqv, moistureAdvSelectorQv_b=bq, **over)
        m, o32, o64 = make_moist(p, tmp_path, seed=nx)
    else:
        p = dict(fe_py.CFG0, **over)
        m, o32, o64 = make(p, tmp_path, seed=nx)
    try:
        for stage in (0, 2):
            check_tendencies(m, o32, o64, stage, f"{shape} b {b} {be} {bq}")
    finally:
        m.close()


@pytest.mark.parametrize("order", [(0.0, 0.6), (0.6, 0.0)])
def test_ensemble_of_equal_and_unequal_weights(order, tmp_path):
    ens = fe_py.Ensemble()
    ens.clear()
    params = [dict(fe_py.CFG0, Nx=64, Ny=16, Nz=16, NtBatch=2, TKEAdvSelector_b_hyb=be) for be in order]
    try:
        ref = []
        for k, p in enumerate(params):
            for run in ("plain", "member"):
                m = fe_py.Model(p, str(tmp_path))
                try:
                    fe_py.turbulent_state((m.array("hydroFlds"), m.array("sgstkeScalars")), seed=70 + k)
                    m.upload()
                    if run == "plain":
                        m.commence()
                        ref.append(np.concatenate([m.interior(m.array("hydroFlds")), m.interior(m.array("sgstkeScalars"))]).copy())
                    else:
                        ens.add(m)
                finally:
                    m.close()
        for k in range(2):                       # a lone run's z segments, whatever the ensemble would choose
            ens.set_segments(k, 4)
        ens.steps(2)
        for k in range(2):
            assert np.array_equal(ens.state(k), ref[k]), order
    finally:
        ens.clear()
