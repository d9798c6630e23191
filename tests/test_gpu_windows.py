"""Several leapfrog steps per launch: the one-wave kernel (n <= 512) and the
windows of sorted sheets with halos (the default path above), against the
oracle, at the sizes where a tile, a lane's block or a window ends.

Equal masses are a power of two here, so that rank * m is the reference's
running sum exactly: those cases are bitwise, and so is the one-wave kernel's
sequential prefix of any masses.  The windows' unequal masses use the exact
fixed-point prefix: 1e-10, the bar of the approximate path.
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


@pytest.mark.parametrize('mass', ['equal', 'lognormal'])
@pytest.mark.parametrize('n', [513, 1024, 1025, 2047, 4096, 4097, 6144, 6145,
                               16385, 50001])
def test_windows(gpu_lib, n, mass):
    """Step sizes from less than a rank to hundreds of ranks per step, one to
    many steps per launch, an uneven number of steps."""
    x, v, m = disk(n, mass)
    for dt, nleap in ((0.0005, 1), (0.0023, 23), (0.02, 13)):
        st, _ = check(x, v, m, dt, nleap, 2, omega=0.1, exact=mass == 'equal')
        if n > 6144:
            assert st == (2 * nleap, 0, 0)  # no radix interval, nothing redone


@pytest.mark.parametrize('force', [forces.Harmonic(0.3), forces.Pulse(0.4, 0.01, 0.02)])
@pytest.mark.parametrize('n', [200, 3000, 20000])
def test_external_force(gpu_lib, n, force):
    x, v, m = disk(n, 'equal')
    # the device's exp differs from the host's in the last place
    check(x, v, m, 0.02, 10, 2, force=force, exact=isinstance(force, forces.Harmonic))


@pytest.mark.parametrize('n', [500, 3000, 20000])
def test_tied_groups(gpu_lib, n):
    """Groups of 40 sheets that start and stay at one position."""
    x, v, m = disk(n, 'equal')
    x = x[(numpy.arange(n) // 40) * 40]
    v = numpy.zeros(n)
    m = numpy.zeros(n)
    m[0] = 1.
    check(x, v, m, 0.1, 8, 2)


def test_halo_too_narrow_is_redone(gpu_lib):
    """The inner sheets move together during the first interval, to half the
    distances the halos were sized for: the windows there report it and the
    interval is redone with wider ones."""
    n = 20000
    x, v, m = disk(n, 'equal')
    v = numpy.where(numpy.abs(x) < 0.05, -10. * x, 0.)
    st, fail = check(x, v, m, 0.05, 10, 3)
    assert st[0] > 0 and st[2] >= 1 and fail[1] >= 1


@pytest.mark.parametrize('kind', ['outliers', 'tails', 'clump'])
@pytest.mark.parametrize('n', [600, 1000, 4000, 6144, 20000])
def test_uneven_density(gpu_lib, n, kind):
    """Bins of one width would hold most of the sheets here: the windows cut
    theirs by rank."""
    x, v, m = disk(n, 'equal')
    if kind == 'outliers':
        x[0], x[1] = 300., -1e4
    elif kind == 'tails':
        x = numpy.clip(numpy.random.default_rng(n).standard_cauchy(n), -1e5, 1e5)
    else:
        x[:n // 3] *= 1e-5
    for dt, nleap in ((0.006, 20), (0.2, 20)):
        check(x, v, m, dt, nleap, 2, omega=0.1)


@pytest.mark.parametrize('n', [200, 3000, 20000])
def test_overflow_as_on_the_other_paths(gpu_lib, n):
    """A sheet that overflows to infinity, then NaN: the others' ranks are as
    the keys' order has them."""
    x, v, m = disk(n, 'equal')
    x[7] = 1.7e308
    out = []
    for kw in ({}, {'path': 'large', 'warm': False}):
        sim = wendy_amd.Sim(x, v, m, numpy.sum(m), 900., **kw)
        gx, gv = numpy.empty(n), numpy.empty(n)
        for _ in range(3):
            sim.advance(0.001, 4)
        sim.read(gx, gv)
        sim.close()
        out.append((gx, gv))
    assert numpy.isnan(out[0][0]).any()
    for a, b in zip(*out):
        assert numpy.array_equal(a, b, equal_nan=True)


@pytest.mark.parametrize('n', [3, 512, 513, 4097, 30000, 65537])
def test_outputs_of_pipelined_reads(gpu_lib, n):
    """read_and_advance: pinned and pageable arrays, one of the two left out,
    reads and an energy in between, a collapse that is redone."""
    x, v, m = disk(n, 'equal')
    if n == 30000:
        v = numpy.where(numpy.abs(x) < 0.05, -10. * x, 0.)
    st = O.ApproxState(x, v, m, 0.05, 10, omega=0.1)
    sim = wendy_amd.Sim(x, v, m, numpy.sum(m), 0.1 ** 2.)
    bufs = [(wendy_amd._lib.pinned_empty(n), wendy_amd._lib.pinned_empty(n)),
            (numpy.empty(n), numpy.empty(n))]
    gx, gv = numpy.empty(n), numpy.empty(n)
    try:
        sim.advance(0.005, 10)
        for k in range(8):
            xo, vo = bufs[(k // 2) % 2]
            if k == 3:
                sim.energy()
            if k == 5:
                sim.read(gx, gv)
            sim.read_and_advance(xo, vo if k != 6 else None, 0.005, 10)
            wx, wv = st.onestep()[:2]
            assert bits_equal(xo, wx), k
            assert k == 6 or bits_equal(vo, wv), k
            assert k != 5 or (bits_equal(gx, wx) and bits_equal(gv, wv))
        sim.read(gx, gv)
        wx, wv = st.onestep()[:2]
        assert bits_equal(gx, wx) and bits_equal(gv, wv)
    finally:
        sim.close()


@pytest.mark.parametrize('mass', ['equal', 'lognormal'])
@pytest.mark.parametrize('n', [150001, 300001, 700001])
def test_large_windows_as_on_another_path(gpu_lib, n, mass):
    """Step sizes up to where the windows no longer pay, so every window shape
    of this range.  Equal masses: the same bits as the large path.  Unequal
    ones: as in a batch, whose mass prefix is exact too (the radix intervals of
    the large path add theirs up in doubles)."""
    x, v, m = disk(n, mass)
    x = numpy.sort(x)
    for h, nleap in ((2.5e-4, 20), (5e-4, 7), (1e-3, 10), (2e-3, 5), (3e-3, 1)):
        out = []
        for path in (None, 'large') if mass == 'equal' else (None,):
            sim = wendy_amd.Sim(x, v, m, numpy.sum(m), 0.1 ** 2., path=path)
            gx, gv = numpy.empty(n), numpy.empty(n)
            for _ in range(2):
                sim.advance(h, nleap)
            sim.read(gx, gv)
            st = sim.path_stats()
            sim.close()
            out.append((gx, gv))
        if mass != 'equal':
            if st[1]:        # not in windows at this step size
                continue
            b = wendy_amd.Batch([x], [v], [m], omegas=[0.1])
            for _ in range(2):
                b.advance(h, nleap)
            got = b.read()
            b.close()
            out.append((got[0][0], got[1][0]))
        assert bits_equal(out[0][0], out[1][0]) and bits_equal(out[0][1], out[1][1]), h
