"""Batches on the GPU with a workgroup per tile and with fewer, over sizes on
either side of the row-sweep tile's edges (16 rows; 48 columns for 2SHOC, 56
for CD), so that tiles inside the grid, on its edge columns only and on its
first or last rows all occur: every problem equals the same problem stepped
alone by the LDS-tile kernels, bit for bit (double also against the oracle)."""
from __future__ import annotations

import numpy as np
import pytest

from conftest import bits_equal

pytestmark = pytest.mark.gpu

SHAPES = [(15, 47), (16, 48), (17, 49), (33, 97), (49, 56), (50, 57), (81, 113), (97, 145), (161, 168), (65, 170)]


@pytest.mark.parametrize("BC", [1, 2, 3])
@pytest.mark.parametrize("method,precision", [(1, 2), (2, 2), (1, 3), (2, 3)])
@pytest.mark.parametrize("grid", [None, 8])
def test_batch_tiles(oracle, method, precision, BC, grid):
    import nlsemagic_amd as nm
    print("CASE batch tiles", method, precision, BC, grid, flush=True)
    rng = np.random.default_rng(7)
    n = len(SHAPES)
    s, a = [(-1.0) ** i for i in range(n)], [0.5 + 0.05 * i for i in range(n)]
    h2, k = [0.04] * n, [0.003] * n
    U = [1 + 0.2 * rng.uniform(-1, 1, sh) + 0.2j * rng.uniform(-1, 1, sh) for sh in SHAPES]
    V = [0.3 * rng.uniform(-1, 1, sh) for sh in SHAPES]
    B = nm.Batch(SHAPES, s, a, h2, k, method=method, precision=precision, BC=BC)
    if grid:
        B.configure(4, 16, grid, 0)
    for i in range(n):
        B.set_state(i, U[i], V[i])
    B.step(3)
    for i in range(n):
        S = nm.Solver(SHAPES[i], method, precision, BC, s[i], a[i], h2[i], k[i])
        S.set_kernel(0, 8)
        S.set_state(U[i], V[i])
        S.step(3)
        assert bits_equal(B.state(i), S.state()), SHAPES[i]
        S.close()
        if precision == 2:
            assert bits_equal(B.state(i), oracle.take_steps(U[i], V[i], s[i], a[i], h2[i], BC, 3, k[i], method)), SHAPES[i]
    B.close()


@pytest.mark.parametrize("kind,rows,fusion", [(0, 8, 2), (0, 16, 2), (0, 32, 2), (2, 16, 2), (1, 8, 2), (1, 12, 4),
                                              (1, 16, 4)])
def test_launch_follows_kernel_until_configured(kind, rows, fusion):
    """Choosing a kernel family takes that family's stages and workgroups per
    launch; what configure() set stays."""
    import nlsemagic_amd as nm
    print("CASE batch launch", kind, rows, flush=True)
    B = nm.Batch([(40, 50), (33, 97)], -1.0, 1.0, 0.04, 0.003, method=2, precision=2)
    assert B.config()[:3] == (4, 1, 16)
    every = B.config()[3]  # a workgroup for every tile
    B.set_kernel(kind, rows)
    assert B.config()[:3] == (fusion, kind, rows)
    assert (B.config()[3] == every) == (kind == 1)
    B.set_kernel(1, 16)
    assert B.config() == (4, 1, 16, every)
    B.configure(1, 16, 64, 0)
    B.set_kernel(kind, rows)
    assert B.config() == (1, kind, rows, 64)
    B.close()


def test_single_precision_keeps_whole_steps_on_8_rows():
    import nlsemagic_amd as nm
    for method, precision in ((1, 2), (1, 3), (2, 3)):
        B = nm.Batch([(40, 50)], -1.0, 1.0, 0.04, 0.003, method=method, precision=precision)
        B.set_kernel(1, 8)
        assert B.config()[0] == 4, (method, precision)
        B.close()


@pytest.mark.parametrize("precision", [2, 3])
def test_diagnostics_of_more_problems_than_a_grid_axis(precision):
    """70,000 problems of 3 x 3 and one larger one: more than the 65,535 that
    one launch of the batch reductions takes."""
    import nlsemagic_amd as nm
    print("CASE batch diagnostics", precision, flush=True)
    n, big = 70_000, 65_540
    shapes = [(3, 3)] * n
    shapes[big] = (40, 33)
    B = nm.Batch(shapes, -1.0, 1.0, 0.04, 0.003, method=1, precision=precision)
    exp = np.zeros((n, 3))
    rng = np.random.default_rng(precision)
    for p in (0, 1, 65_533, 65_534, 65_535, 65_536, big, n - 1):
        U = rng.integers(-8, 9, shapes[p]) + 1j * rng.integers(-8, 9, shapes[p])  # sums of squares: exact
        B.set_state(p, U, np.zeros(shapes[p]))
        exp[p] = (U.real ** 2 + U.imag ** 2).sum(), U.real.max(), 0
    assert np.array_equal(B.diagnostics(), exp)
    B.close()
