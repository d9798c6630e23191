"""Windows that fail beside others of their launch that start later: more of
them than the GPU holds at a time, and halos that a collapsing knot of sheets
outgrows in the middle of the ranks.  Masses a power of two: bitwise as on the
large path.
"""
import ctypes

import numpy
import pytest

import wendy_amd
from conftest import bits_equal
from oracle import nbody_oracle as O
from wendy_amd import _lib

pytestmark = pytest.mark.gpu

N, H, NLEAP, OUT = 900001, 1e-4, 400, 3


def knot(seed):
    x = numpy.sort(O.sech2_disk(N, seed=seed)[0])
    return x, numpy.where(numpy.abs(x) < 0.3, -10. * x, 0.), numpy.full(N, 2. ** -20)


def advanced(sim):
    x, v = numpy.empty(N), numpy.empty(N)
    for _ in range(OUT):
        sim.advance(H, NLEAP)
    sim.read(x, v)
    st = sim.path_stats()
    sim.close()
    return x, v, st


def test_failures_beside_later_windows(gpu_lib):
    states = [knot(k) for k in (1, 2, 3)]
    want = [advanced(wendy_amd.Sim(x, v, m, numpy.sum(m), -1., path='large'))
            for x, v, m in states]
    x, v, m = states[0]
    got = advanced(wendy_amd.Sim(x, v, m, numpy.sum(m), -1.))
    assert got[2][2] >= 1  # a window of the single simulation failed
    assert bits_equal(got[0], want[0][0]) and bits_equal(got[1], want[0][1])
    b = wendy_amd.Batch(*[list(a) for a in zip(*states)])
    for _ in range(OUT):
        b.advance(H, NLEAP)
    gx, gv, _ = b.read()
    b.close()
    for k, w in enumerate(want):
        assert bits_equal(gx[k], w[0]) and bits_equal(gv[k], w[1]), k


@pytest.mark.parametrize('kind', ['overflow', 'collapse'])
@pytest.mark.parametrize('n', [600, 3000, 20000])
def test_outputs_of_an_interval_whose_first_launch_failed(gpu_lib, n, kind):
    """Several launches an interval, the first of which fails, with outputs
    written by the last one: from the first call on a fresh simulation, when
    none of its buffers has held a state yet."""
    x, v, _ = O.sech2_disk(n, seed=n)
    m = numpy.full(n, 2. ** -numpy.ceil(numpy.log2(n)))
    h, nleap, omega2 = 1e-3, 200, 900.
    if kind == 'overflow':
        x[7] = 1.7e308
    else:
        v, omega2 = numpy.where(numpy.abs(x) < 0.3, -10. * x, 0.), 0.01
    a = wendy_amd.Sim(x, v, m, numpy.sum(m), omega2)
    b = wendy_amd.Sim(x, v, m, numpy.sum(m), omega2, path='large', warm=False)
    got = _lib.pinned_empty(n), _lib.pinned_empty(n)
    want = x.copy(), v.copy()
    try:
        for _ in range(4):
            # (no interval has run yet at the first call: no time of one)
            _lib.check(gpu_lib.wdy_read_and_advance(
                a._h, *[g.ctypes.data_as(ctypes.c_void_p) for g in got], h, nleap, None))
            for g, w in zip(got, want):
                assert numpy.array_equal(g, w, equal_nan=True)
            b.advance(h, nleap)
            b.read(*want)
        # (the field at the sheet that overflows leaves no room for several
        # windows, and without several a collapse does no harm)
        if (kind == 'overflow') == (n <= 6144):
            assert a.path_stats()[2] >= 1
    finally:
        a.close()
        b.close()
