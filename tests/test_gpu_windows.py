"""The one-wave kernel (n <= 512) against the oracle, at the sizes where a
lane's block ends.

Equal masses are a power of two here, so that rank * m is the reference's
running sum exactly: those cases are bitwise, and so is the one-wave kernel's
sequential prefix of any masses.
"""
import numpy
import pytest

import wendy_amd
from conftest import bits_equal, rel_inf
from oracle import nbody_oracle as O
from wendy_amd import forces

pytestmark = pytest.mark.gpu

TOL = 1e-10


def disk(n, mass, seed=None):
    x, v, m = O.sech2_disk(n, seed=n if seed is None else seed,
                           mass='equal' if mass == 'equal' else ('lognormal', 0.5))
    if mass == 'equal':
        m = numpy.full(n, 2. ** -numpy.ceil(numpy.log2(max(n, 2))))
    return x, v, m


def check(x, v, m, dt, nleap, nout, omega=None, force=None, exact=True):
    sim = wendy_amd.Sim(x, v, m, numpy.sum(m), -1. if omega is None else omega ** 2.)
    try:
        if force is not None:
            sim.set_ext_force(force, 0.)
        st = O.ApproxState(x, v, m, dt, nleap, omega=omega, ext_force=force)
        gx, gv = numpy.empty(len(x)), numpy.empty(len(x))
        for k in range(nout):
            sim.advance(dt / nleap, nleap)
            sim.read(gx, gv)
            wx, wv = st.onestep()[:2]
            if exact:
                assert bits_equal(gx, wx) and bits_equal(gv, wv), \
                    (k, rel_inf(gx, wx), rel_inf(gv, wv))
            else:
                assert rel_inf(gx, wx) <= TOL and rel_inf(gv, wv) <= TOL, \
                    (k, rel_inf(gx, wx), rel_inf(gv, wv))
        return sim.path_stats(), sim.warm_failures()
    finally:
        sim.close()


@pytest.mark.parametrize('mass', ['equal', 'lognormal'])
@pytest.mark.parametrize('n', [1, 2, 3, 127, 128, 129, 255, 256, 257, 511, 512])
def test_one_wave(gpu_lib, n, mass):
    """Few to many crossings per step (dt = 0.05 and 2): both orders of the
    prefix's restart are met."""
    x, v, m = disk(n, mass)
    for dt, nleap in ((0.05, 20), (2., 7)):
        check(x, v, m, dt, nleap, 2, omega=0.3)
