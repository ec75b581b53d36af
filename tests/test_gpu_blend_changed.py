"""Blending weights of the hybrid schemes changed after the set-up: b_hyb, TKEAdvSelector_b_hyb and
moistureAdvSelectorQv_b are the program's variables and every launch takes their current values, so a
model set up with one set and given another computes, bit for bit, what a model set up with the
latter does; likewise a member given its weights between its set-up and fe_ens_add_member.  From
equal to unequal weights and back, by one weight at a time.
"""
import numpy as np
import pytest

import fe_py

pytestmark = pytest.mark.gpu

KEYS = ("b_hyb", "TKEAdvSelector_b_hyb", "moistureAdvSelectorQv_b")


def _model(moist, weights, tmp_path, **over):
    p = dict(fe_py.CFG2, d_zeta=60.0) if moist else dict(fe_py.CFG0)
    p.update(Nx=70, Ny=11, Nz=12, NtBatch=2, **over)
    p.update({k: w for k, w in zip(KEYS, weights) if moist or k != KEYS[2]})
    m = fe_py.Model(p, str(tmp_path))
    fe_py.turbulent_state((m.array("hydroFlds"), m.array("sgstkeScalars")), seed=5)
    if moist:
        fe_py.moist_state(m, seed=6)
    m.upload()
    return m


def _give(m, weights, moist):
    for k, w in zip(KEYS, weights):
        if moist or k != KEYS[2]:
            m.setf(k, w)


def _outputs(m, moist):
    """Tendencies of a plain and of the physics stage, and the state after two steps."""
    names = ["hydroFlds", "sgstkeScalars"] + ["moistScalars"] * moist
    out = []
    for stage in (0, 2):
        m.build_frhs(stage)
        out += [m.interior(m.array(n + "Frhs")).copy() for n in names]
    m.commence()
    return out + [m.interior(m.array(n)).copy() for n in names]


@pytest.mark.parametrize("moist,before,after", [
    (False, (0.0, 0.0), (0.0, 0.7)), (False, (0.2, 0.2), (0.9, 0.2)), (False, (0.0, 0.7), (0.3, 0.3)),
    (True, (0.0, 0.0, 0.0), (0.0, 0.0, 0.6)), (True, (0.1, 0.1, 0.1), (0.8, 0.1, 0.1)), (True, (0.0, 0.5, 0.2), (0.4, 0.4, 0.4))])
def test_weights_changed_after_setup(moist, before, after, tmp_path):
    got = []
    for start in (after, before):
        m = _model(moist, start, tmp_path)
        try:
            _give(m, after, moist)
            got.append(_outputs(m, moist))
        finally:
            m.close()
    for k, (a, b) in enumerate(zip(*got)):
        assert np.array_equal(a, b), (k, before, after)


def test_member_weights_changed_before_it_is_added(tmp_path):
    before, after = (0.0, 0.0), (0.0, 0.7)
    m = _model(False, after, tmp_path, amd_zSegments=1)
    try:
        m.commence()
        ref = np.concatenate([m.interior(m.array("hydroFlds")), m.interior(m.array("sgstkeScalars"))]).copy()
    finally:
        m.close()
    ens = fe_py.Ensemble()
    ens.clear()
    try:
        for w in (before, after):                    # a member of equal weights first
            m = _model(False, before, tmp_path, amd_zSegments=1)
            try:
                _give(m, w, False)
                ens.add(m)
            finally:
                m.close()
        ens.steps(2)
        assert np.array_equal(ens.state(1), ref)
        assert not np.array_equal(ens.state(0), ref)
    finally:
        ens.clear()
