"""Plain stages whose own cell and x fluxes go through LDS (WENO5; moist over terrain: test_topography):
stage tendencies against the oracle with the tolerance of test_gpu_parity, at whole tiles, partial tiles
in x and y and a grid narrower than a tile, in one segment and in segments down to two levels."""
import pytest

import fe_py
from test_gpu_parity import check_tendencies, make

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nseg", [1, 2, 5])
@pytest.mark.parametrize("shape", [(64, 8, 10), (70, 19, 13), (20, 13, 9), (129, 17, 12)])
def test_weno5(shape, nseg, tmp_path):
    nx, ny, nz = shape
    m, o32, o64 = make(dict(fe_py.CFG0, Nx=nx, Ny=ny, Nz=nz, advectionSelector=5, TKEAdvSelector=5, amd_zSegments=nseg),
                       tmp_path, seed=nx + nseg)
    try:
        for stage in (0, 1, 2):
            check_tendencies(m, o32, o64, stage, f"weno5 {shape} {nseg}")
    finally:
        m.close()
