"""Planning time of deep circuits in one tile grows with their ops, not with
their square: 16 times the layers take at most 64 times as long (linear 16,
quadratic 256)."""
import time

import pytest

import pyramaterised_amd as pyqc
from pyramaterised_amd import engine as E
from pyramaterised_amd import templates as T


def _seconds(n, layers, make):
    qc = pyqc.PQC(n)
    qc.add_layers(make(layers, n))
    ops = qc.ops()
    best = 1e9
    for _ in range(3):
        t = time.perf_counter()
        E.Plan(n, ops)
        best = min(best, time.perf_counter() - t)
    return best


@pytest.mark.parametrize("make", [T.clifford_HE_layers, T.qg_circuit_layers])
def test_small_tile_plans_take_linear_time(make):
    n = 5
    assert _seconds(n, 3200, make) < 64 * _seconds(n, 200, make)
