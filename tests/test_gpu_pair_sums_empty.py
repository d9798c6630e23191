"""The potential of no sheets is the harmonic term alone."""
import numpy
import pytest

import wendy_amd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('ny', [1, 5, 4096])
@pytest.mark.parametrize('omega', [None, 0.4])
def test_potential_of_no_sheets(gpu_lib, ny, omega):
    y = numpy.linspace(-3., 3., ny)
    none = numpy.empty(0)
    want = numpy.zeros(ny) if omega is None else omega ** 2. * (y * y) / 2.
    assert numpy.array_equal(wendy_amd.potential(y, none, none, none, omega=omega), want)
    assert len(wendy_amd.energy(none, none, none, individual=True, omega=omega)) == 0
