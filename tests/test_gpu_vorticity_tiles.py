"""The vorticity kernel's tiles on the GPU: 7 rows x 56 or 60 columns, chunks of 4
to 16 planes by grid size, neighbours across rows from the previous step's
planes.  Sizes lie on either side of each tile edge, with enough tiles for
every chunk length; the kernel keeps the oracle's operand order in double, so
the results agree bit for bit."""
from __future__ import annotations

import numpy as np
import pytest

from conftest import bits_equal

pytestmark = pytest.mark.gpu


# planes either side of one chunk of 4, rows of 7, columns of 60; (70, 150, 130)
# takes chunks between 4 and 16 planes, (65, 222, 182) chunks of 16
@pytest.mark.parametrize("shape", [(4, 7, 60), (5, 8, 61), (6, 6, 59), (7, 13, 62), (8, 14, 63), (9, 15, 122), (4, 6, 56),
                                   (5, 9, 112), (6, 10, 168), (4, 15, 240), (5, 7, 248),
                                   (17, 21, 64), (70, 150, 130), (65, 222, 182)])
@pytest.mark.parametrize("precision", [2, 1, 3])
def test_tile_edges(oracle, shape, precision):
    import nlsemagic_amd as nm
    print("CASE vorticity tiles", shape, precision, flush=True)
    rng = np.random.default_rng(sum(shape))
    U = 1 + 0.3 * rng.standard_normal(shape) + 0.3j * rng.standard_normal(shape)
    S = nm.Solver(shape, 1, precision, 1, -1.0, 1.0, 0.04, 0.004)
    S.set_state(U)
    got = S.vorticity(1 / (2 * 0.2), 1e-3)
    state = S.state()  # as held, widened to double
    S.close()
    assert all(bits_equal(g, e) for g, e in zip(got, oracle.vorticity3d(state, 1 / (2 * 0.2), 1e-3)))
