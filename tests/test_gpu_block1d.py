"""1D time-blocked windows: every position of the grid's end in a wave's core.

A wave owns 56 (CD) or 48 (2SHOC) points of its window; grids whose length
leaves one to three points to the last wave need its boundary rule's inward
reach to stay exact through the four stages of a step.
"""
from __future__ import annotations

import numpy as np
import pytest

from conftest import bits_equal

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hip():
    import nlsemagic_amd as nm
    if nm.device_count() < 1:
        pytest.fail("no HIP device visible")
    return nm


# one segment of 64 points and less, several windows, 256-point segments
SIZES = [3, 5, 47, 48, 49, 50, 51, 55, 56, 57, 58, 59, 97, 98, 113, 114, 193, 209, 233, 234, 273, 297, 298, 2049,
         2051, 32801, 50021]


@pytest.mark.parametrize("method", [1, 2])
@pytest.mark.parametrize("n", SIZES)
def test_block1d_every_tail_matches_oracle(hip, oracle, n, method):
    rng = np.random.default_rng(n + method)
    U = (0.9 + 0.3 * rng.uniform(-1, 1, n)) + 1j * (0.3 * rng.uniform(-1, 1, n))
    V = 0.5 * rng.uniform(-1, 1, n)
    for BC in (1, 2, 3, 4, 0):
        if BC == 4 and n < 4:
            continue
        for prec in (2, 1):
            for steps in (3, 37):
                print("CASE", n, method, BC, prec, steps, flush=True)
                got = hip.take_steps(U, V, -1.0, 0.9, 0.04, BC, steps, 0.004, precision=prec, method=method)
                exp = oracle.take_steps(U, V, -1.0, 0.9, 0.04, BC, steps, 0.004, method, precision=prec)
                assert bits_equal(got, exp), (BC, prec, steps)


@pytest.mark.parametrize("method", [1, 2])
@pytest.mark.parametrize("n", SIZES)
def test_block1d_compensated_matches_unblocked(hip, n, method):
    """Compensated states: the bits of the kernels without windows (the whole
    chunk in one workgroup, or a launch per stage above 4096 points), for a
    chunk of several launches and an odd one after it."""
    rng = np.random.default_rng(n + method)
    U = (0.9 + 0.3 * rng.uniform(-1, 1, n)) + 1j * (0.3 * rng.uniform(-1, 1, n))
    V = 0.5 * rng.uniform(-1, 1, n)
    for BC in (1, 2, 3, 4, 0):
        if BC == 4 and n < 4:
            continue
        print("CASE", n, method, BC, flush=True)
        got = []
        for kind in (None, 0):
            sol = hip.Solver((n,), method, 3, BC, -1.0, 0.9, 0.04, 0.004)
            if kind is not None:
                sol.set_kernel(kind, 8)
            sol.set_state(U, V)
            sol.step(37)
            sol.step(3)
            got.append(sol.state())
            sol.close()
        assert bits_equal(*got), BC
