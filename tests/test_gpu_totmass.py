"""A total mass that is not the masses' sum, as a caller of wdy_create may give
it: F = (totmass - 2 C) - m, whatever totmass is, at every small size."""
import numpy
import pytest

import wendy_amd
from conftest import rel_inf
from oracle import nbody_oracle as O

pytestmark = pytest.mark.gpu

TOL = 1e-10


@pytest.mark.parametrize('factor', [0.125, 0.999, 0., 8.])
@pytest.mark.parametrize('n', [100, 600, 1000, 1536])
def test_any_total_mass(gpu_lib, n, factor):
    x, v, m = O.sech2_disk(n, seed=n, mass=('lognormal', 0.5))
    out = []
    for path in (None, 'small'):
        sim = wendy_amd.Sim(x, v, m, factor * numpy.sum(m), 0.01, path=path)
        gx, gv = numpy.empty(n), numpy.empty(n)
        for _ in range(3):
            sim.advance(0.01, 10)
        sim.read(gx, gv)
        sim.close()
        out.append((gx, gv))
    assert rel_inf(out[0][0], out[1][0]) <= TOL and rel_inf(out[0][1], out[1][1]) <= TOL
