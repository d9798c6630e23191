"""Individual energies and potentials at the sizes where a block of points, a
block of sheets or a stretch of sheets ends, against sums in extended
precision.

All terms are positive and every sum is a tree above chains of at most
n / 256 + 128 additions, 148 here: relative errors stay below
(148 + 20) * 2^-53 = 1.9e-14.
"""
import numpy
import pytest

import wendy_amd

pytestmark = pytest.mark.gpu

RTOL = 1.9e-14


def state(n, seed):
    rs = numpy.random.default_rng(seed)
    return rs.standard_normal(n), rs.standard_normal(n), rs.uniform(0.5, 2., n) / n


def sums(y, x, m):
    x, m = x.astype(numpy.longdouble), m.astype(numpy.longdouble)
    return numpy.array([numpy.sum(m * numpy.abs(x - a)) for a in y], dtype=numpy.longdouble)


@pytest.mark.parametrize('n', [1, 2, 15, 16, 17, 255, 257, 1025, 4095, 4096, 4097, 5001])
def test_individual_energies(gpu_lib, n):
    x, v, m = state(n, n)
    for twopiG, omega in ((1., None), (2., 0.4)):
        w = twopiG * m * sums(x, x, m) + m * v ** 2. / 2.
        if omega is not None:
            w = w + m * omega ** 2. * x ** 2. / 2.
        got = wendy_amd.energy(x, v, m, twopiG=twopiG, individual=True, omega=omega)
        numpy.testing.assert_allclose(got, w.astype(float), rtol=RTOL)


@pytest.mark.parametrize('ny', [1, 3, 4, 5, 63, 4096, 4100])
@pytest.mark.parametrize('n', [1, 2, 257, 2047, 2048, 5000])
def test_potential(gpu_lib, n, ny):
    x, v, m = state(n, n)
    y = numpy.random.default_rng(ny).uniform(-3., 3., ny)
    numpy.testing.assert_allclose(wendy_amd.potential(y, x, v, m),
                                  sums(y, x, m).astype(float), rtol=RTOL)
