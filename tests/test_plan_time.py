"""Planning time of deep circuits in one tile grows with their ops, not with
their square: 16 times the layers may take 128 times the processor time
(linear 16, three times that where the op records outgrow the caches,
quadratic 256 and as much more)."""
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
        t = time.process_time()
        E.Plan(n, ops)
        best = min(best, time.process_time() - t)
    return best


@pytest.mark.parametrize("make", [T.clifford_HE_layers, T.qg_circuit_layers])
def test_small_tile_plans_take_linear_time(make):
    n = 5
    assert _seconds(n, 6400, make) < 128 * _seconds(n, 400, make)
