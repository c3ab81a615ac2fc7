"""States between host arrays and the device: complex arrays and split planes,
through one pinned block (up to 3 MB of host arrays) and through the staged
copies above it, for every precision.  Odd counts put an unequal split on the
two staging areas."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

from conftest import bits_equal

pytestmark = pytest.mark.gpu

# points whose put (24 B each) or get (16 B) ends below, at and above 3 MB
SIZES = [3, 401, 131071, 131072, 131073, 196608, 196609, 400001]


@pytest.fixture(scope="module")
def hip():
    import nlsemagic_amd as nm
    if nm.device_count() < 1:
        pytest.fail("no HIP device visible")
    return nm


def _stored(U, prec):
    """What a state of this precision holds of U, widened to double."""
    if prec == 2:
        return U
    hi = U.astype(np.complex64)
    lo = (U - hi.astype(np.complex128)).astype(np.complex64)
    return hi.astype(np.complex128) + (lo.astype(np.complex128) if prec == 3 else 0)


@pytest.mark.parametrize("prec", [2, 1, 3])
@pytest.mark.parametrize("n", SIZES)
def test_state_round_trip(hip, n, prec):
    print("CASE", n, prec, flush=True)
    rng = np.random.default_rng(n + prec)
    U = rng.standard_normal(n) + 1j * rng.standard_normal(n)
    V = rng.standard_normal(n)
    exp = _stored(U, prec)
    sol = hip.Solver((n,), 1, prec, 1, -1.0, 1.0, 0.01, 0.001)
    sol.set_state(U, V)
    assert bits_equal(sol.state(), exp)
    dp = C.POINTER(C.c_double)
    r, i = np.empty(n), np.empty(n)
    L = hip.lib()
    assert L.nlse_get_state(sol._h, r.ctypes.data_as(dp), i.ctypes.data_as(dp)) == 0
    assert bits_equal(r + 1j * i, exp)
    sol.set_state(np.zeros(n))
    r[:], i[:] = U.real, U.imag
    assert L.nlse_set_state(sol._h, r.ctypes.data_as(dp), i.ctypes.data_as(dp), None) == 0
    assert bits_equal(sol.state(), exp)
    assert L.nlse_set_state(sol._h, r.ctypes.data_as(dp), None, None) == 0  # no imaginary part: zero
    assert bits_equal(sol.state(), _stored(U.real + 0j, prec))
    # V went with the first upload: the energy of a constant state is its sum
    sol.fill(1.0)
    v = V.astype(np.float32).astype(float) if prec != 2 else V
    assert abs(sol.energy()[2] / 0.1 - (v.sum() + 0.5 * n)) < 1e-9 * n
    sol.close()


@pytest.mark.parametrize("prec", [2, 3])
def test_batch_state_round_trip(hip, prec):
    shapes = [(3, 5), (301, 437), (37, 64)]
    rng = np.random.default_rng(prec)
    B = hip.Batch(shapes, -1.0, 1.0, 0.01, 0.001, method=1, precision=prec)
    Us = [rng.standard_normal(s) + 1j * rng.standard_normal(s) for s in shapes]
    for p, U in enumerate(Us):
        B.set_state(p, U, np.zeros(U.shape))
    for p, U in enumerate(Us):
        assert bits_equal(B.state(p), _stored(U, prec))
    B.close()


@pytest.mark.parametrize("prec", [2, 3])
@pytest.mark.parametrize("shape", [(3, 3), (363, 363), (513, 513), (600, 437)])
def test_one_problem_batch_round_trip(hip, shape, prec):
    """A batch whose only problem has an odd count (363^2: put above 3 MB, get
    below; 513^2: both above): the longer half of the staged state has the
    batch's buffers to itself, with no other problem's points behind it."""
    print("CASE", shape, prec, flush=True)
    rng = np.random.default_rng(shape[0] + prec)
    U = rng.standard_normal(shape) + 1j * rng.standard_normal(shape)
    V = rng.standard_normal(shape)
    exp = _stored(U, prec)
    B = hip.Batch([shape], -1.0, 1.0, 0.01, 0.001, method=1, precision=prec)
    B.set_state(0, U, V)
    assert bits_equal(B.state(0), exp)
    dp = C.POINTER(C.c_double)
    r, i = np.empty(shape), np.empty(shape)
    L = hip.lib()
    assert L.nlse_batch_get_state(B._h, 0, r.ctypes.data_as(dp), i.ctypes.data_as(dp)) == 0
    assert bits_equal(r + 1j * i, exp)
    B.set_state(0, np.zeros(shape), V)
    r[:], i[:] = U.real, U.imag
    assert L.nlse_batch_set_state(B._h, 0, r.ctypes.data_as(dp), i.ctypes.data_as(dp), V.ctypes.data_as(dp)) == 0
    assert bits_equal(B.state(0), exp)
    B.close()


# points whose put (24 B each) or get (16 B) lies below or at 256 KB, from where
# a single-precision state passes the pinned block as floats, and whose floats
# (12 B, 8 B) fill a block or just do not
@pytest.mark.parametrize("n", [10922, 10923, 16383, 16384, 262144, 262145, 393216, 393217])
def test_single_precision_through_the_block(hip, n):
    print("CASE", n, flush=True)
    rng = np.random.default_rng(n)
    U = rng.standard_normal(n) + 1j * rng.standard_normal(n)
    U[:6] = [np.inf, -np.inf, 1e-50, 1e50, 3e-42 + 1e39j, -0.0]  # kept, underflowing, overflowing, subnormal
    U[-1] = complex(1 + 2.0 ** -24, np.nan)                      # a tie
    V = rng.standard_normal(n)
    with np.errstate(over="ignore", invalid="ignore"):
        exp = U.astype(np.complex64).astype(np.complex128)
    sol = hip.Solver((n,), 1, 1, 1, -1.0, 1.0, 0.01, 0.001)
    dp = C.POINTER(C.c_double)
    L = hip.lib()
    r, i, v = np.ascontiguousarray(U.real), np.ascontiguousarray(U.imag), V
    gr, gi = np.empty(n), np.empty(n)
    for put in (lambda: sol.set_state(U, V), lambda: sol.set_state(U),
                lambda: L.nlse_set_state(sol._h, *(x.ctypes.data_as(dp) for x in (r, i, v)))):
        sol.set_state(np.zeros(n))
        put()
        assert bits_equal(sol.state(), exp)
        assert L.nlse_get_state(sol._h, gr.ctypes.data_as(dp), gi.ctypes.data_as(dp)) == 0
        assert bits_equal(gr, exp.real.copy()) and bits_equal(gi, exp.imag.copy())
    sol.fill(1.0)
    assert abs(sol.energy()[2] / 0.1 - (V.astype(np.float32).astype(float).sum() + 0.5 * n)) < 1e-9 * n
    sol.close()


@pytest.mark.parametrize("prec", [2, 1, 3])
@pytest.mark.parametrize("n", [401, 400001])
def test_real_states_go_without_a_complex_copy(hip, n, prec):
    """A real array is a state with no imaginary part, whatever the state held
    before, and is handed over as it is."""
    import tracemalloc
    print("CASE", n, prec, flush=True)
    rng = np.random.default_rng(n + prec)
    U = rng.standard_normal(n)
    sol = hip.Solver((n,), 1, prec, 1, -1.0, 1.0, 0.01, 0.001)
    for real in (U, U.astype(np.float32), np.arange(n) % 7, np.arange(n) % 2 == 0, U[::-1]):
        sol.set_state(rng.standard_normal(n) + 1j)
        tracemalloc.start()
        sol.set_state(real)
        peak = tracemalloc.get_traced_memory()[1]
        tracemalloc.stop()
        assert bits_equal(sol.state(), _stored(real.astype(np.float64) + 0j, prec))
        as_is = real.dtype == np.float64 and real.flags.c_contiguous
        assert peak < 20000 + (0 if as_is else 8 * n)
    sol.close()


@pytest.mark.parametrize("prec", [2, 3])
def test_real_batch_states(hip, prec):
    shapes = [(301, 437), (37, 64)]
    rng = np.random.default_rng(prec)
    B = hip.Batch(shapes, -1.0, 1.0, 0.01, 0.001, method=1, precision=prec)
    for p, sh in enumerate(shapes):
        B.set_state(p, rng.standard_normal(sh) + 1j, np.zeros(sh))
    Us = [rng.standard_normal(sh) for sh in shapes]
    for p, U in enumerate(Us):
        B.set_state(p, U, np.zeros(U.shape))
    for p, U in enumerate(Us):
        assert bits_equal(B.state(p), _stored(U + 0j, prec))
    B.close()
