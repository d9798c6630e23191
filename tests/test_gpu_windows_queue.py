"""Intervals enqueued behind each other in windows: more of them than are kept in
flight, and a failure among them, from which on they are redone in order.  Masses
a power of two: bitwise against the oracle."""
import numpy
import pytest

import wendy_amd
from conftest import bits_equal
from oracle import nbody_oracle as O
from wendy_amd import forces

pytestmark = pytest.mark.gpu


def disk(n):
    x, v, _ = O.sech2_disk(n, seed=n)
    return x, v, numpy.full(n, 2. ** -numpy.ceil(numpy.log2(n)))


@pytest.mark.parametrize('n', [513, 6145, 30001])
@pytest.mark.parametrize('knot', [False, True])
def test_many_intervals(gpu_lib, n, knot):
    """Steps of changing size and number; with a knot of sheets that collapses
    meanwhile, halos fail now and then."""
    x, v, m = disk(n)
    if knot:
        v = numpy.where(numpy.abs(x) < 0.3, -10. * x, 0.)
    force = forces.Harmonic(0.3)
    sim = wendy_amd.Sim(x, v, m, numpy.sum(m), -1.)
    sim.set_ext_force(force, 0.)
    st = O.ApproxState(x, v, m, 1., 1, ext_force=force)
    gx, gv = numpy.empty(n), numpy.empty(n)
    k = 0
    for count in (1, 2, 45, 20):
        for _ in range(count):
            st.h, st.nleap = (1e-3, 1e-3, 5e-4)[k % 3], 1 + k % 4
            k += 1
            sim.advance(st.h, st.nleap)
            wx, wv = st.onestep()[:2]
        sim.read(gx, gv)
        assert bits_equal(gx, wx) and bits_equal(gv, wv), k
        assert sim.time() == st.t
    redos = sim.path_stats()[2]
    sim.close()
    if not knot:
        assert redos == 0


@pytest.mark.parametrize('n', [600, 3000])
def test_overflow_among_them(gpu_lib, n):
    """One sheet's oscillation grows by some orders of magnitude a step, until it
    overflows in an interval in the middle."""
    x, v, m = disk(n)
    x[7] = 1e290
    out = []
    for kw in ({}, {'path': 'large', 'warm': False}):
        sim = wendy_amd.Sim(x, v, m, numpy.sum(m), 1e6, **kw)
        gx, gv = numpy.empty(n), numpy.empty(n)
        for _ in range(12):
            sim.advance(0.1, 2)
        sim.read(gx, gv)
        out.append((gx, gv, sim.path_stats()))
        sim.close()
    assert numpy.isnan(out[0][0]).any() and out[0][2][2] == 1
    for a, b in zip(out[0][:2], out[1][:2]):
        assert numpy.array_equal(a, b, equal_nan=True)
