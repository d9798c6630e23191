"""What the library's host code does when device memory runs out or a kernel
reports back, without a GPU: in a process of its own, on a stand-in for the HIP
runtime (fake_hip.cpp) that writes launches down and fails allocations on demand.
"""
import os
import shutil
import subprocess
import sys

import pytest

from conftest import ROOT

HEAD = r'''
import ctypes, sys
fake = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
fake.fake_log.restype = ctypes.c_char_p
fake.fake_deny.argtypes = [ctypes.c_size_t]
fake.fake_deny_new.argtypes = [ctypes.c_size_t]
fake.fake_spacing.argtypes = [ctypes.c_double]
fake.fake_register.argtypes = [ctypes.c_void_p, ctypes.c_size_t]
NONE = ctypes.c_size_t(-1).value
sys.path.insert(0, sys.argv[2])
import numpy
import wendy_amd


def launched():
    names = fake.fake_log().decode().split('\n')
    fake.fake_clear()
    return names


def sim(n, mass='unequal', **kw):
    rs = numpy.random.default_rng(n)
    m = rs.uniform(0.5, 2., n) / n if mass == 'unequal' else numpy.full(n, 1. / n)
    return wendy_amd.Sim(rs.standard_normal(n), rs.standard_normal(n), m, numpy.sum(m),
                         -1., **kw)


def count(names, what):
    return sum(what in k for k in names)

'''


@pytest.fixture(scope='module')
def fake(tmp_path_factory):
    cxx = os.environ.get('CXX') or shutil.which('g++')
    assert cxx, 'no C++ compiler'
    so = str(tmp_path_factory.mktemp('fake') / 'libfake_hip.so')
    subprocess.run([cxx, '-std=c++17', '-O1', '-fPIC', '-shared',
                    os.path.join(ROOT, 'tests', 'fake_hip.cpp'), '-o', so], check=True)
    return so


def run(fake, body):
    got = subprocess.run([sys.executable, '-c', HEAD + body, fake, ROOT],
                         capture_output=True, text=True, timeout=300)
    assert got.returncode == 0, (got.returncode, got.stdout, got.stderr)


def test_windows_declined_without_memory_for_the_warm_path(fake):
    """Its arrays are allocated when they are first needed: radix steps then,
    and no launch of the warm kernel without them."""
    run(fake, r'''
s = sim(20000)            # the stand-in reports no room for windows
launched()
config = s.warm_config()  # a question allocates nothing
fake.fake_deny(1)
assert s.warm_config() == config and config[0] >= 0
for _ in range(2):
    s.advance(0.01, 3)
    k = launched()
    assert count(k, 'k_scatter') > 0 and count(k, 'k_warm_step') == 0, k
fake.fake_deny(NONE)
s.advance(0.01, 3)        # and back to it
assert count(launched(), 'k_warm_step') > 0
s.close()
''')


@pytest.mark.parametrize('mass', ['equal', 'unequal'])
def test_warm_path_that_cannot_grow(fake, mass):
    run(fake, r'''
s = sim(20000, '%s', path='large')
fake.fake_deny(1)         # this step size calls for more buckets either side
for _ in range(2):
    launched()
    s.advance(10., 3)
    k = launched()
    assert count(k, 'k_scatter') > 0 and count(k, 'k_warm_step') == 0, k
try:
    s.tune(0, 8, 0)
    raise AssertionError('tuned without memory')
except MemoryError:
    pass
s.advance(0.01, 3)
assert count(launched(), 'k_warm_step') == 0
s.close()
''' % mass)


@pytest.mark.parametrize('granted', [0, 1, 2, 3])
def test_batch_without_memory_for_windows(fake, granted):
    """The interval runs in the workgroup-per-simulation kernel, wherever among
    the windows' allocations the memory runs out, and a later plan may have it."""
    run(fake, r'''
b = [numpy.random.default_rng(k) for k in range(40)]
x = [r.standard_normal(700) for r in b]
b = wendy_amd.Batch(x, x, [r.uniform(0.5, 2., 700) / 700. for r in b])
b.advance(1e-3, 10)
fake.fake_deny([1, 4 * 40 + 1, 40 * 100 + 1, 40 * 700 * 8 + 1][%d])
for _ in range(2):
    launched()
    b.advance(1e-3, 10)
    k = launched()
    assert count(k, 'k_batch_advance') == 1
    assert (count(k, 'k_span_many') > 0) == (%d == 3), k
fake.fake_deny(NONE)
for _ in range(2):
    b.advance(2e-3, 10)
assert count(launched(), 'k_span_many') > 0
b.close()
''' % (granted, granted))


@pytest.mark.parametrize('n', [300, 1000, 20000])
def test_outputs_without_memory_for_staging(fake, n):
    """They are de-sorted by a launch of their own."""
    run(fake, r'''
fake.fake_spacing(1e-4)   # room for windows
s = sim(%d)
x, v = numpy.empty(s.n), numpy.empty(s.n)
s.advance(1e-6, 2)
fake.fake_deny(1)
for _ in range(3):
    launched()
    s.read_and_advance(x, v, 1e-6, 2)
    assert count(launched(), 'k_desort') == 1
fake.fake_deny(NONE)
s.read_and_advance(x, v, 1e-6, 2)
launched()
s.read_and_advance(x, v, 1e-6, 2)
assert count(launched(), 'k_desort') == 0
s.close()
''' % n)


@pytest.mark.parametrize('bad', ['numpy.inf', 'numpy.nan'])
@pytest.mark.parametrize('n', [2000, 9000])
def test_one_simulation_not_finite(fake, n, bad):
    """The others of its batch stay in windows."""
    run(fake, r'''
@ctypes.CFUNCTYPE(None, ctypes.c_char_p, ctypes.POINTER(ctypes.c_void_p))
def report(name, args):
    # what k_batch_form(descs, arrays, many, err) says of every simulation: ten
    # widths of 4, 8, ... ranks, the largest |v| and |x|; `many` ends with their
    # address
    if b'k_batch_form' in name:
        many = ctypes.cast(args[2], ctypes.POINTER(ctypes.c_void_p))
        info = numpy.ctypeslib.as_array(
            ctypes.cast(many[5], ctypes.POINTER(ctypes.c_double)), shape=(40, 12))
        info[:, :10] = 1e-3 * 2. ** numpy.arange(2, 12)
        info[:, 10:] = 1.
        info[39, 10] = %s  # the smallest


fake.fake_hook(report)
r = [numpy.random.default_rng(k) for k in range(40)]
x = [q.standard_normal(%d if k < 39 else 100) for k, q in enumerate(r)]
b = wendy_amd.Batch(x, x, [numpy.full(len(q), 1. / len(q)) for q in x])
for _ in range(2):
    b.advance(1e-3, 10)
assert count(launched(), 'k_span_many') > 0
b.close()
''' % (bad, n))


def test_batch_of_changing_steps(fake):
    """A plan sorts every simulation: only for steps that have come twice."""
    run(fake, r'''
x = [numpy.random.default_rng(k).standard_normal(700) for k in range(40)]
b = wendy_amd.Batch(x, x, [numpy.full(700, 1. / 700.)] * 40)
for k in range(6):
    b.advance((1e-3, 2e-3)[k % 2], 10)
for k in range(6):
    b.advance(1e-3, 10 + k)
assert count(launched(), 'k_batch_form') == 0
b.advance(1e-3, 15)
k = launched()
assert count(k, 'k_batch_form') > 0 and count(k, 'k_span_many') > 0
b.close()
''')


def test_outputs_written_by_a_kernel(fake):
    """Only into memory that is page-locked from end to end."""
    run(fake, r'''
fake.fake_spacing(1e-4)
s = sim(1000)
s.advance(1e-6, 2)


def copied(x, v):
    launched()
    s.read_and_advance(x, v, 1e-6, 2)
    return count(launched(), 'k_copy_out') > 0


pinned = wendy_amd._lib.pinned_empty
assert copied(pinned(1000), pinned(1000))
big = pinned(3000)
assert copied(big[:1000], big[2000:])
plain = numpy.empty(1000)
assert not copied(plain, pinned(1000)) and not copied(pinned(1000), plain)
fake.fake_register(plain.ctypes.data, 800)           # its ends, by themselves
fake.fake_register(plain.ctypes.data + 7200, 800)
assert not copied(plain, pinned(1000)) and not copied(pinned(1000), plain)
s.close()
''')


def test_inputs_are_looked_over(fake):
    """A bad value is found wherever it stands; a negative mass, or a total mass
    that is not the sum, leaves a simulation without windows."""
    run(fake, r'''
for n in list(range(1, 20)) + [1000]:
    good = [numpy.linspace(-1., 1., n), numpy.linspace(2., -2., n), numpy.full(n, 1. / n)]
    for i in sorted({0, n // 3, n - 1}):
        for a in range(3):
            for bad in (numpy.nan, numpy.inf, -numpy.inf):
                xvm = [q.copy() for q in good]
                xvm[a][i] = bad
                try:
                    wendy_amd.Sim(*xvm, 1., -1.)
                    raise AssertionError((n, i, a, bad))
                except ValueError as e:
                    assert 'sheet %d' % i in str(e), e
        m = good[2].copy()
        m[i] *= 2.
        if n > 1:
            try:
                wendy_amd.Sim(good[0], good[1], m, 1., -1., equal_mass=True)
                raise AssertionError((n, i))
            except ValueError as e:
                assert 'm[%d]' % (i or 1) in str(e), e
        for m, total, windows in ((good[2], 1., True), (m, m.sum(), True), (m, 3., False),
                                  (numpy.where(m == m[i], -m, m), m.sum(), False)):
            launched()
            wendy_amd.Sim(good[0], good[1], m, total, -1., equal_mass=False).close()
            assert (count(launched(), 'k_span_widths') == 1) == (windows and n > 512), n
''')


def test_every_set_holds_indices(fake):
    """Those of a simulation with windows and of a batch, before any launch reads
    them."""
    run(fake, r'''
@ctypes.CFUNCTYPE(None, ctypes.c_char_p, ctypes.POINTER(ctypes.c_void_p))
def look(name, args):
    at = [int(ctypes.cast(args[k], ctypes.POINTER(ctypes.c_uint64))[0]) for k in sets.get(name, ())]
    seen.extend(at)


seen = []
sets = {}
sim(1000).close()
assert count(launched(), 'k_iota') == 2  # the staged set, and the one not sorted into
sim(1000, path='large').close()
assert count(launched(), 'k_iota') == 1
x = numpy.linspace(-1., 1., 700)
wendy_amd.Batch([x], [x], [x * 0. + 1.]).close()
init = [q for q in launched() if 'k_batch_init' in q][0].encode()
sets[init] = (3, 4)               # (n, x, key, idx, idx2)
fake.fake_hook(look)
wendy_amd.Batch([x], [x], [x * 0. + 1.]).close()
assert len(seen) == 2 and len(set(seen)) == 2 and 0 not in seen
''')


@pytest.mark.parametrize('n', [1 << 20, (1 << 20) + 1])
def test_warm_path_of_large_simulations(fake, n):
    """Set up with the simulation above 2^20 sheets, whatever windows it has."""
    run(fake, r'''
s = sim(%d, 'equal')      # no room for windows here
launched()
fake.fake_deny(1)
s.advance(1e-9, 3)
assert (count(launched(), 'k_warm_step') > 0) == (s.n > 1 << 20)
s.close()
''' % n)


@pytest.mark.parametrize('n', [3, 1000, 20000])
def test_read_before_the_first_interval(fake, n):
    """There is no time of an interval to ask for yet, and no error of that left
    for the next call."""
    run(fake, r'''
fake.fake_spacing(1e-4)
s = sim(%d)
x, v = numpy.empty(s.n), numpy.empty(s.n)
assert s.read(x, v) == 0.
s.advance(1e-6, 2)
assert s.read(x, v) > 0.
s.close()
s = sim(%d)
assert s.read_and_advance(x, v, 1e-6, 2) == 0.
assert s.read(x, v) > 0.
s.close()
b = wendy_amd.Batch([x], [x], [numpy.full(s.n, 1.)])
assert b.read()[2] == 0.
b.advance(1e-6, 2)
assert b.read()[2] > 0.
b.close()
''' % (n, n))


def test_batch_without_host_memory_for_windows(fake):
    """Their list: no exception leaves the library, the interval runs without them."""
    run(fake, r'''
x = [numpy.random.default_rng(k).standard_normal(700) for k in range(1100)]
b = wendy_amd.Batch(x, x, [numpy.full(700, 1. / 700.)] * 1100)
b.advance(1e-3, 10)
launched()
fake.fake_deny_new(4096)
for _ in range(2):
    b.advance(1e-3, 10)
fake.fake_deny_new(NONE)
k = launched()
assert count(k, 'k_batch_advance') == 2 and count(k, 'k_span_many') == 0, k
for _ in range(2):
    b.advance(2e-3, 10)
assert count(launched(), 'k_span_many') > 0
b.close()
''')
