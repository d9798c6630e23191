"""When the windows hold, when they are given up and when they are tried again.
Masses a power of two: bitwise against the oracle."""
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


@pytest.mark.parametrize('by', ['omega', 'force'])
def test_strong_fields_from_rest(gpu_lib, by):
    """A field that grows with |x| is all that moves the sheets: the halos allow
    for it from the start."""
    n = 20001
    x, v, m = disk(n)
    v[:] = 0.
    omega, force = (30., None) if by == 'omega' else (None, forces.Harmonic(30.))
    sim = wendy_amd.Sim(x, v, m, numpy.sum(m), -1. if omega is None else omega ** 2.)
    sim.set_ext_force(force, 0.)
    st = O.ApproxState(x, v, m, 1e-4, 10, omega=omega, ext_force=force)
    gx, gv = numpy.empty(n), numpy.empty(n)
    for _ in range(3):
        sim.advance(1e-5, 10)
        sim.read(gx, gv)
        wx, wv = st.onestep()[:2]
        assert bits_equal(gx, wx) and bits_equal(gv, wv)
    stats = sim.path_stats()
    sim.close()
    assert stats == (30, 0, 0)  # in windows, nothing redone
    if by == 'omega':
        b = wendy_amd.Batch([x, x], [v, v], [m, m], omegas=[omega, None])
        for _ in range(3):
            b.advance(1e-5, 10)
        bx, bv, _ = b.read()
        b.close()
        assert bits_equal(bx[0], wx) and bits_equal(bv[0], wv)


@pytest.mark.parametrize('n,h', [(10000, 0.1), (32768, 0.03)])
def test_steps_too_large_for_windows(gpu_lib, n, h):
    """About a thousand ranks a step: one step per launch is faster."""
    x, v, m = disk(n)
    sim = wendy_amd.Sim(x, v, m, numpy.sum(m), -1.)
    for _ in range(2):
        sim.advance(h, 20)
    stats = sim.path_stats()
    sim.close()
    assert stats[:2] == (20, 20)  # a radix interval, then the warm-start kernel


def test_steps_of_another_size_try_again(gpu_lib):
    """A knot of sheets falls through one point within an interval, where no
    halos hold; later, shorter steps are taken in windows again."""
    n = 20001
    x, _, m = disk(n)
    v = numpy.where(numpy.abs(x) < 0.3, -10. * x, 0.)
    sim = wendy_amd.Sim(x, v, m, numpy.sum(m), -1.)
    st = O.ApproxState(x, v, m, 0.04, 400)
    gx, gv = numpy.empty(n), numpy.empty(n)

    def both(h, nleap):
        st.h, st.nleap = h, nleap
        sim.advance(h, nleap)
        sim.read(gx, gv)
        wx, wv = st.onestep()[:2]
        assert bits_equal(gx, wx) and bits_equal(gv, wv)
        return sim.path_stats()
    for _ in range(4):
        warm, cold, redo = both(1e-4, 400)
    assert cold > 0 and redo >= 3
    assert both(5e-5, 20) == (warm + 20, cold, redo)
    # (not the ones they were given up for: a radix interval again)
    assert both(1e-4, 400)[1:] == (cold + 400, redo)
    sim.close()
