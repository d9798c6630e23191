"""The one-wave kernel and the workgroup's, each in the external forces it runs
them in, where the choice between the two lies; outputs by every kind of read."""
import numpy
import pytest

import wendy_amd
from conftest import rel_inf
from oracle import nbody_oracle as O
from wendy_amd import forces

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('force', [forces.Isothermal(-0.7, 1.2), forces.Harmonic(0.3)],
                         ids=['isothermal', 'harmonic'])
@pytest.mark.parametrize('mass', ['equal', 'lognormal'])
@pytest.mark.parametrize('n', [255, 256, 257, 512])
def test_small_in_a_force(gpu_lib, n, mass, force):
    x, v, m = O.sech2_disk(n, seed=n, mass='equal' if mass == 'equal' else ('lognormal', 0.5))
    st = O.ApproxState(x, v, m, 0.05, 10, ext_force=force)
    sim = wendy_amd.Sim(x, v, m, numpy.sum(m), -1.)
    sim.set_ext_force(force, 0.)
    px, pv = wendy_amd._lib.pinned_empty(n), wendy_amd._lib.pinned_empty(n)
    sim.advance(0.005, 10)
    for _ in range(3):
        wx, wv = [a.copy() for a in st.onestep()[:2]]
        sim.read_and_advance(px, pv, 0.005, 10)
        # (tanh on the device differs from the host's in the last place)
        assert rel_inf(px, wx) <= 1e-10 and rel_inf(pv, wv) <= 1e-10
    sim.set_ext_force(None)  # in one wave from here on
    sim.read(px, pv)
    wx, wv = [a.copy() for a in st.onestep()[:2]]
    assert rel_inf(px, wx) <= 1e-10 and rel_inf(pv, wv) <= 1e-10
    st = O.ApproxState(wx, wv, m, 0.05, 10)
    for _ in range(2):
        sim.advance(0.005, 10)
        wx, wv = [a.copy() for a in st.onestep()[:2]]
        sim.read_and_advance(px, pv, 0.005, 10)
        st.onestep()
        assert rel_inf(px, wx) <= 1e-10 and rel_inf(pv, wv) <= 1e-10
    sim.close()
