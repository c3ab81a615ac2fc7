"""Reductions (diagnostics, energy, kfull) allocate neither device nor pinned
host memory: their results go to a slot the solver got when it was created."""
from __future__ import annotations

import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_reductions_allocate_nothing_in_a_fresh_process():
    code = """
import nlsemagic_amd as nm
S = nm.Solver((64, 65), 2, 2, 2, -1.0, 1.0, 0.01, 0.001)
S.fill(0.5)
before = nm.device_allocations(), nm.pinned_allocations()
for _ in range(2):
    S.step(2)
    S.diagnostics(), S.energy(), S.kfull()
print("new:", nm.device_allocations() - before[0], nm.pinned_allocations() - before[1])
S.close()
"""
    r = subprocess.run([sys.executable, "-c", code], cwd=ROOT, capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stderr
    assert r.stdout.split() == ["new:", "0", "0"]


def test_solvers_beyond_the_slots_reduce_alike():
    """130 solvers at once, 128 slots: the last ones copy their results; slots
    given back are taken again."""
    import nlsemagic_amd as nm
    print("CASE 130 solvers", flush=True)
    for turn in range(2):
        S = [nm.Solver((40 + i,), 1, 2, 1, -1.0, 1.0, 0.01, 0.001) for i in range(130)]
        before = nm.device_allocations(), nm.pinned_allocations()
        for i, s in enumerate(S):
            s.fill(1.0 + i)
        for i, s in enumerate(S):
            assert s.diagnostics() == ((40 + i) * (1.0 + i) ** 2, 1.0 + i, 0)
        assert (nm.device_allocations(), nm.pinned_allocations()) == before
        for s in S:
            s.close()
