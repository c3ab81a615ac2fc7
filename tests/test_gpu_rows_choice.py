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
