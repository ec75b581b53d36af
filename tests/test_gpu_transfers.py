"""Host arrays through the pinned ring and the tiled layout conversions: upload then download gives
the interior back bit for bit and the halos by the boundary rules, at extents below, at and past a
64-cell tile edge, at fields of less than one piece, of exactly one page more than a piece (4 MB) and
of many pieces; arrays of one model do not end up in the next model's; network rows on both sides
of the 16 MB line.  All bounds are exact: a transfer changes no bit.
"""
import numpy as np
import pytest

import fe_py

pytestmark = pytest.mark.gpu
NH = 3

SHAPES = [(5, 4, 6), (64, 8, 58), (63, 9, 59), (65, 10, 64), (70, 130, 122), (58, 122, 130), (200, 186, 75)]


@pytest.mark.parametrize("shape", SHAPES, ids=["x".join(map(str, s)) for s in SHAPES])
@pytest.mark.parametrize("halo", [0, 1])
def test_round_trip(shape, halo, tmp_path):
    nx, ny, nz = shape
    if halo and (nx % 64 or ny % 8):
        pytest.skip("lateral halo storage holds whole tiles")
    p = dict(fe_py.CFG2, Nx=nx, Ny=ny, Nz=nz, d_zeta=10.0, dampingLayerDepth=20.0, NtBatch=1, amd_haloBuffer=halo)
    m = fe_py.Model(p, str(tmp_path))
    try:
        rng = np.random.default_rng(nx)
        names = ("hydroFlds", "sgstkeScalars", "moistScalars")
        want = {}
        for n in names:
            a = m.array(n)
            a[...] = rng.standard_normal(a.shape, np.float32)
            want[n] = a[:, NH:-NH, NH:-NH, NH:-NH].copy()
        surf = {n: rng.standard_normal(m.shape2, np.float32) for n in ("fricVel", "htFlux", "tskin", "z0m", "z0t")}
        for n, a in surf.items():
            m.array(n)[...] = a
        m.upload()
        for n in names:
            m.array(n)[...] = np.nan
        m.download()
        for n in names:
            a = m.array(n)
            assert np.array_equal(a[:, NH:-NH, NH:-NH, NH:-NH], want[n]), n
            inner = a[:, :, :, NH:-NH]
            for ax, size in ((1, nx), (2, ny)):            # periodic sides
                idx = (np.arange(-NH, size + NH) % size) + NH
                assert np.array_equal(inner, np.take(inner, idx, axis=ax)), (n, ax)
        h, q, e = (m.array(n) for n in ("hydroFlds", "moistScalars", "sgstkeScalars"))
        bs = m.array("hydroBaseStateFlds")
        for f, b in ((0, 0), (4, 1)):
            for k in list(range(NH)) + list(range(nz + NH, nz + 2 * NH)):
                assert np.array_equal(h[f, :, :, k], bs[b, :, :, k]), (f, k)
        for k in range(NH):
            assert np.array_equal(h[1:4, :, :, k], h[1:4, :, :, NH])
            assert np.array_equal(q[..., k], q[..., NH]) and np.array_equal(q[..., nz + NH + k], q[..., nz + NH - 1])
            assert not e[..., nz + NH + k].any() and not h[3, :, :, nz + NH + k].any()
        for n, a in surf.items():
            if n not in ("fricVel", "htFlux"):
                assert np.array_equal(m.array(n)[NH:-NH, NH:-NH], a[NH:-NH, NH:-NH]), n
    finally:
        m.close()


def test_models_in_turn(tmp_path):
    """Slots sized for a small model serve a larger one after it, and the other way round."""
    for k, (nx, ny, nz) in enumerate(((16, 8, 10), (150, 140, 60), (16, 8, 10))):
        m = fe_py.Model(dict(fe_py.CFG0, Nx=nx, Ny=ny, Nz=nz, NtBatch=1), str(tmp_path))
        try:
            a = m.array("hydroFlds")
            a[...] = np.random.default_rng(k).standard_normal(a.shape, np.float32)
            want = m.interior(a).copy()
            m.upload()
            a[...] = 0
            m.download()
            assert np.array_equal(m.interior(a), want), k
        finally:
            m.close()


@pytest.mark.parametrize("rows", [1, 16383, 16384, 16500])
def test_network_rows_on_both_sides_of_the_line(rows, tmp_path):
    m = fe_py.Model(dict(fe_py.CFG0, Nx=64, Ny=8, Nz=16, NtBatch=1), str(tmp_path))
    s = fe_py.LearnedSGS()
    try:
        s.clear()
        s.init_params(3)
        X = np.random.default_rng(rows).standard_normal((rows, 256), np.float32)
        Y = s.forward(X)
        i = np.unique(np.array([0, rows // 2, rows - 1]))
        assert np.array_equal(s.forward(X[i]), Y[i])       # a row's output does not depend on the others
    finally:
        s.clear()
        m.close()
