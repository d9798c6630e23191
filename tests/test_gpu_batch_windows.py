"""A batch in windows of several steps per launch: its simulations against
the oracle, from the first interval (one workgroup per simulation) on.

Equal masses are a power of two, so that rank * m is the reference's running
sum exactly: bitwise.  Unequal masses use the exact fixed-point prefix: 1e-10,
the bar of the approximate path.
"""
import numpy
import pytest

import wendy_amd
from conftest import bits_equal, rel_inf
from oracle import nbody_oracle as O

pytestmark = pytest.mark.gpu

TOL = 1e-10
OMEGA = 0.1


def sims(ns, masses):
    out = []
    for k, (n, mass) in enumerate(zip(ns, masses)):
        x, v, m = O.sech2_disk(n, seed=1000 + k,
                               mass='equal' if mass == 'equal' else ('lognormal', 0.5))
        if mass == 'equal':
            m = numpy.full(n, 2. ** -numpy.ceil(numpy.log2(max(n, 2))))
        out.append((x, v, m))
    return out


def run(states, masses, steps, read_each):
    b = wendy_amd.Batch(*[list(a) for a in zip(*states)], omegas=[OMEGA] * len(states))
    refs = [O.ApproxState(x, v, m, steps[0][0], steps[0][1], omega=OMEGA)
            for x, v, m in states]
    got = None
    try:
        want = [None] * len(states)
        for i, (dt, nleap) in enumerate(steps):
            b.advance(dt / nleap, nleap)
            for k, r in enumerate(refs):
                r.h, r.nleap = dt / nleap, nleap
                want[k] = [a.copy() for a in r.onestep()[:2]]
            if read_each or i == len(steps) - 1:
                got = b.read()
                for k, mass in enumerate(masses):
                    for g, w in zip((got[0][k], got[1][k]), want[k]):
                        if mass == 'equal':
                            assert bits_equal(g, w), (i, k, len(g), rel_inf(g, w))
                        else:
                            assert rel_inf(g, w) <= TOL, (i, k, len(g), rel_inf(g, w))
    finally:
        b.close()


@pytest.mark.parametrize('read_each', [False, True])
@pytest.mark.parametrize('mass', ['equal', 'lognormal', 'mixed'])
@pytest.mark.parametrize('ns', [(1,), (3, 511, 2048, 2049, 4097), (30001,),
                                (700,) * 40 + (16384, 5000)])
def test_batch_windows(gpu_lib, ns, mass, read_each):
    """Odd and even step counts, one step per interval, a change of the step
    between intervals (a new plan from windows)."""
    masses = [mass if mass != 'mixed' else ('equal', 'lognormal')[k % 2]
              for k in range(len(ns))]
    steps = [(0.01, 10)] * 3 + [(0.02, 7)] * 3 + [(0.001, 1)] * 2
    run(sims(ns, masses), masses, steps, read_each)


def test_failed_windows_are_repaired(gpu_lib):
    """The inner sheets of two simulations move together while a plan holds:
    their windows report it and the rest of the interval is done by the
    workgroup-per-simulation kernel, beside others that go on in windows."""
    masses = ['equal', 'equal', 'lognormal', 'equal']
    states = sims((20000, 3000, 12000, 9000), masses)
    for k in (0, 2):
        x, v, m = states[k]
        states[k] = (x, numpy.where(numpy.abs(x) < 0.05, -10. * x, 0.), m)
    run(states, masses, [(0.05, 10)] * 4, True)
