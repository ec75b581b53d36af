"""A network call that fails on its way (an error left by another call of the program is reported by its
first launch) returns with the caller's arrays no longer in use and the stream idle: they may change at
once, and the next call is right."""
import ctypes
import re

import numpy as np
import pytest

import fe_py

pytestmark = pytest.mark.gpu


def _runtime():
    maps = open("/proc/self/maps").read()
    return ctypes.CDLL(re.search(r"(/\S*libamdhip64\.so\S*)", maps).group(1))


@pytest.mark.parametrize("rows", [7, 12000, 17000])
def test_error_on_the_way(rows, tmp_path):
    m = fe_py.Model(dict(fe_py.CFG0, Nx=64, Ny=8, Nz=16, NtBatch=1), str(tmp_path))
    s = fe_py.LearnedSGS()
    try:
        s.clear()
        s.init_params(3)
        rng = np.random.default_rng(rows)
        X = rng.normal(size=(rows, 256)).astype(np.float32)
        T = rng.normal(size=(rows, 16)).astype(np.float32)
        want, (loss, grad) = s.forward(X), s.gradient(X, T)
        hip = _runtime()
        for call in (lambda a: s.forward(a), lambda a: s.gradient(a, T)):
            a = X.copy()
            assert hip.hipSetDevice(1 << 20) != 0            # no such device: an error for the next check to report
            with pytest.raises(RuntimeError):
                call(a)
            a[:] = np.nan
            del a
            assert np.array_equal(s.forward(X), want)
            l2, g2 = s.gradient(X, T)
            assert abs(l2 - loss) <= 1e-12 * loss and np.array_equal(g2, grad)
    finally:
        s.clear()
        m.close()
