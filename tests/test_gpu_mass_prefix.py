"""The mass below each sheet, in the windows and in a batch, against its exact
value: masses of few values, whose fixed-point rounding errors would add up if
they all leaned the same way.

From rest, one step of h = 2^-12 leaves v = h * a exactly, and
a = (totmass - 2 C) - m: the roundings of C (twice), of the difference and of
the subtraction of m are below 2^-53 of the total mass each, and the n
fixed-point errors, of at most 2^-61 of it and independent, below four times
sqrt(n) / 2 of that: 4 * 2^-53 + 4 sqrt(n) 2^-61.  (To nearest, 1.5e6 sheets of
two values were 1.6e-13 off.)
"""
import numpy
import pytest

import wendy_amd

pytestmark = pytest.mark.gpu

H = 2. ** -12


def state(n, kind):
    rs = numpy.random.default_rng(n)
    x = 2. * numpy.arctanh(numpy.clip(2. * rs.random(n) - 1., -1. + 1e-12, 1. - 1e-12))
    if kind == 'tracers':
        m = numpy.zeros(n)
        m[:(n + 1) // 2] = 1. / ((n + 1) // 2)
    else:
        m = numpy.where(rs.random(n) < 0.3, 1., numpy.where(rs.random(n) < 0.5, 3.3, 0.017))
        m = m / m.sum()
    return x, numpy.zeros(n), m


def exact_acceleration(x, m):
    """In whole numbers of 2^-112: every mass here is one."""
    o = numpy.argsort(x, kind='stable')
    top = numpy.floor(numpy.ldexp(m[o], 60))
    low = numpy.ldexp(numpy.ldexp(m[o], 60) - top, 52).astype(numpy.int64)
    parts = ((top.astype(numpy.int64), -60), (low >> 26, -86), (low & ((1 << 26) - 1), -112))
    c = sum(numpy.ldexp((numpy.cumsum(p) - p).astype(numpy.longdouble), e) for p, e in parts)
    a = numpy.empty(len(x), dtype=numpy.longdouble)
    a[o] = (numpy.longdouble(numpy.sum(m)) - 2 * c) - m[o]
    return a


@pytest.mark.parametrize('kind', ['tracers', 'species'])
@pytest.mark.parametrize('n', [600, 1500, 20001, 1500001])
def test_mass_below(gpu_lib, n, kind):
    x, v, m = state(n, kind)
    tot = numpy.sum(m)
    want = exact_acceleration(x, m)
    tol = (4. * 2. ** -53 + 4. * numpy.sqrt(n) * 2. ** -61) * tot
    sim = wendy_amd.Sim(x, v, m, tot, -1.)
    gx, gv = numpy.empty(n), numpy.empty(n)
    sim.advance(H, 1)
    sim.read(gx, gv)
    st = sim.path_stats()
    sim.close()
    assert st[1:] == (0, 0)  # in windows
    out = [gv]
    if n < 1 << 16:  # (one workgroup puts a batch's simulation in order at first)
        b = wendy_amd.Batch([x], [v], [m])
        b.advance(H, 1)
        out.append(b.read()[1][0])
        b.close()
    for got in out:
        assert numpy.max(numpy.abs(got.astype(numpy.longdouble) / H - want)) <= tol
