"""Tiling of the 3D two-stage launches: chunk lengths chosen by grid size.

The chunk length along the first axis depends on the number of tiles per
plane, so grids are picked whose last chunk, row tile or column tile holds one
point, or whose chunks are the shortest and longest the rule gives.  Results
must not depend on the tiling: they equal one stage per launch bit for bit.
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


def _run(hip, shape, method, prec, BC, fusion, U, V, steps):
    sol = hip.Solver(shape, method, prec, BC, -1.0, 0.9, 0.04, 0.004)
    sol.set_fusion(fusion)
    sol.set_state(U, V)
    sol.step(steps)
    got = sol.state()
    sol.close()
    return got


def _field(shape, seed):
    rng = np.random.default_rng(seed)
    U = (0.9 + 0.3 * rng.uniform(-1, 1, shape)) + 1j * (0.3 * rng.uniform(-1, 1, shape))
    return U, 0.5 * rng.uniform(-1, 1, shape)


@pytest.mark.parametrize("prec", [2, 1, 3])
@pytest.mark.parametrize("method", [1, 2])
@pytest.mark.parametrize("shape,BC", [((41, 25, 121), 1), ((13, 300, 57), 3), ((200, 100, 61), 1), ((7, 5, 113), 3)])
def test_pair3d_chunk_lengths(hip, shape, BC, method, prec):
    print("CASE", shape, BC, method, prec, flush=True)
    U, V = _field(shape, sum(shape) + method)
    assert bits_equal(_run(hip, shape, method, prec, BC, 2, U, V, 3), _run(hip, shape, method, prec, BC, 1, U, V, 3))


def _msd_cases():
    """MSD pairs: thin grids along each axis, last tiles of one row, column
    or plane (the tiles then shift by one), several tiles per axis; double
    2SHOC runs pairs on larger grids only."""
    small = [(3, 400, 400), (401, 3, 400), (400, 401, 3), (65, 97, 121), (97, 61, 113), (41, 97, 169), (81, 85, 61)]
    large = [(3, 1001, 900), (1001, 3, 900), (900, 1001, 3), (129, 137, 169), (98, 229, 113)]
    return [(sh, m, pr) for m in (1, 2) for pr in (2, 1, 3) for sh in (large if (m, pr) == (2, 2) else small)]


@pytest.mark.parametrize("shape,method,prec", _msd_cases())
def test_pair3d_msd_matches_one_stage(hip, shape, method, prec):
    """Two MSD stages per launch give the bits of one stage per launch, NaN
    and infinities included where a partner point is zero."""
    print("CASE", shape, method, prec, flush=True)
    U, V = _field(shape, sum(shape) + method)
    sol = hip.Solver(shape, method, prec, 2, -1.0, 0.9, 0.04, 0.004)
    assert sol.config()[0] == 2
    sol.close()
    assert bits_equal(_run(hip, shape, method, prec, 2, 2, U, V, 3), _run(hip, shape, method, prec, 2, 1, U, V, 3))
    U[1, 1, 1] = U[-2, shape[1] // 2, -2] = U[shape[0] // 2, -2, shape[2] // 2] = 0
    a = _run(hip, shape, method, prec, 2, 2, U, V, 1)
    assert bits_equal(a, _run(hip, shape, method, prec, 2, 1, U, V, 1)) and np.isnan(a.real).any()


@pytest.mark.parametrize("shape,method", [((65, 97, 121), 1), ((98, 229, 113), 2)])
def test_pair3d_msd_matches_oracle(hip, oracle, shape, method):
    U, V = _field(shape, sum(shape))
    exp = oracle.take_steps(U, V, -1.0, 0.9, 0.04, 2, 2, 0.004, method)
    assert bits_equal(_run(hip, shape, method, 2, 2, 2, U, V, 2), exp)
