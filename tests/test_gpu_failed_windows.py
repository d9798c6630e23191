"""Windows that fail beside others of their launch that start later: more of
them than the GPU holds at a time, and halos that a collapsing knot of sheets
outgrows in the middle of the ranks.  Masses a power of two: bitwise as on the
large path.
"""
import numpy
import pytest

import wendy_amd
from conftest import bits_equal
from oracle import nbody_oracle as O

pytestmark = pytest.mark.gpu

N, H, NLEAP, OUT = 900001, 1e-4, 400, 3


def knot(seed):
    x, _, _ = O.sech2_disk(N, seed=seed)
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
