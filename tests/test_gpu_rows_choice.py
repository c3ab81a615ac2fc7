"""2D row-sweep tiles by grid size: the default rows and waves per tile, and the
results of every choice against the oracle.

Grids are picked on both sides of the lines between the choices (8 rows on 16
or 8 waves, 12 rows, 16 rows on 16 or 8 waves), with last tiles of one row or
column.
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


SHAPES = [(9, 57), (41, 49), (129, 145), (341, 253), (489, 337), (515, 389), (1001, 97), (521, 513), (601, 609),
          (737, 673)]


@pytest.mark.parametrize("method,prec", [(1, 2), (1, 1), (2, 2), (2, 1)])
@pytest.mark.parametrize("shape", SHAPES)
def test_default_tiles_match_oracle(hip, oracle, shape, method, prec):
    rng = np.random.default_rng(sum(shape))
    U = (0.9 + 0.3 * rng.uniform(-1, 1, shape)) + 1j * (0.3 * rng.uniform(-1, 1, shape))
    V = 0.5 * rng.uniform(-1, 1, shape)
    for BC in (1, 2, 3):
        print("CASE", shape, method, prec, BC, flush=True)
        exp = oracle.take_steps(U, V, -1.0, 0.9, 0.04, BC, 2, 0.004, method, precision=prec)
        assert bits_equal(hip.take_steps(U, V, -1.0, 0.9, 0.04, BC, 2, 0.004, precision=prec, method=method), exp), BC


@pytest.mark.parametrize("shape", [(64, 64), (512, 512), (1024, 1024)])
def test_rows_asked_for_are_kept(hip, shape):
    for rows in (8, 12, 16):
        sol = hip.Solver(shape, 2, 2, 1, -1.0, 1.0, 0.01, 0.001)
        sol.set_kernel(1, rows)
        assert sol.config() == (4, 1, rows)
        sol.close()
    sol = hip.Solver((1024, 1024), 2, 2, 1, -1.0, 1.0, 0.01, 0.001)
    assert sol.config() == (4, 1, 16)
    sol.close()


@pytest.mark.parametrize("method,prec", [(1, 2), (1, 1), (2, 2), (2, 1)])
@pytest.mark.parametrize("shape", [(3, 20000), (12, 12000), (17, 5000), (32, 2000), (33, 2000), (600, 600), (1024, 200),
                                   (2000, 200), (640, 641)])
def test_skewed_grids_match_oracle(hip, oracle, shape, method, prec):
    """Few rows or columns, and grids at the lines of the choice."""
    rng = np.random.default_rng(sum(shape))
    U = (0.9 + 0.3 * rng.uniform(-1, 1, shape)) + 1j * (0.3 * rng.uniform(-1, 1, shape))
    V = 0.5 * rng.uniform(-1, 1, shape)
    for BC in (1, 2):
        print("CASE", shape, method, prec, BC, flush=True)
        exp = oracle.take_steps(U, V, -1.0, 0.9, 0.04, BC, 2, 0.004, method, precision=prec)
        assert bits_equal(hip.take_steps(U, V, -1.0, 0.9, 0.04, BC, 2, 0.004, precision=prec, method=method), exp), BC


@pytest.mark.parametrize("shape,rows", [((3, 20000), {1: 8, 2: 8}), ((12, 12000), {1: 8, 2: 16}), ((17, 5000), {1: 8, 2: 16}),
                                        ((600, 600), {1: 8, 2: 12}), ((2000, 200), {1: 8, 2: 16}), ((1024, 1024), {1: 16, 2: 16})])
def test_rows_by_shape(hip, shape, rows):
    """The rows of single-precision solvers (256 compute units)."""
    for method, r in rows.items():
        sol = hip.Solver(shape, method, 1, 1, -1.0, 1.0, 0.01, 0.001)
        assert sol.config() == (4, 1, r), (shape, method)
        sol.close()


@pytest.mark.parametrize("method,BC", [(1, 1), (1, 2), (2, 1), (2, 2), (1, 3), (2, 3)])
@pytest.mark.parametrize("shape", [(9, 57), (129, 145), (341, 253), (17, 5000), (521, 513), (601, 609), (1001, 97)])
def test_default_tiles_compensated(hip, shape, method, BC):
    """Compensated single precision on the chosen tiles: the bits of the
    LDS-tile kernels."""
    print("CASE", shape, method, BC, flush=True)
    rng = np.random.default_rng(sum(shape))
    U = (0.9 + 0.3 * rng.uniform(-1, 1, shape)) + 1j * (0.3 * rng.uniform(-1, 1, shape))
    V = 0.5 * rng.uniform(-1, 1, shape)
    got = []
    for kind in (None, 0):
        sol = hip.Solver(shape, method, 3, BC, -1.0, 0.9, 0.04, 0.004)
        if kind is not None:
            sol.set_kernel(kind, 8)
        sol.set_state(U, V)
        sol.step(3)
        got.append(sol.state())
        sol.close()
    assert bits_equal(*got)
