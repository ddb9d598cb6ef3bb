"""Specialised complex128 sweeps trade real and imaginary parts through LDS
one after the other.  Every transition (wave-local, block-wide, after a
cross-lane exchange), staged and direct loads and stores, rolling and standard
write layouts give the same bits as the persistent form, which trades whole
amplitudes."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,tile,low,rolling", [(10, 10, 3, False), (12, 12, 3, False), (13, 13, 3, False),
                                                (13, 10, 3, True), (14, 11, 4, True), (14, 12, 3, False)])
@pytest.mark.parametrize("extra", ["none", "no_direct", "no_wave_local", "no_exchange"])
def test_halves_match_whole_tiles(n, tile, low, rolling, extra):
    import pyramaterised_amd as pyqc
    from pyramaterised_amd import _lib as L
    from pyramaterised_amd import engine as E
    from pyramaterised_amd import templates as T
    flag = {"none": 0, "no_direct": L.PQS_PLAN_NO_DIRECT, "no_wave_local": L.PQS_PLAN_NO_WAVE_LOCAL,
            "no_exchange": L.PQS_PLAN_NO_EXCHANGE}[extra]
    rng = np.random.default_rng(n + tile)
    qc = pyqc.PQC(n, jit=False)
    for layer in T.clifford_HE_layers(2, n):
        qc.add_layer(layer)
    qc.add_layer([pyqc.R_zz([0, n - 1], n), pyqc.R_xx([1, n // 2], n), pyqc.CZ([2, n - 2], n), pyqc.R_x(n // 2, n)])
    ops = qc.ops()
    flags = flag | (L.PQS_PLAN_ROLLING if rolling else 0)
    a = E.Plan(n, ops, tile_bits=tile, low_bits=low, flags=flags).jit()
    b = E.Plan(n, ops, tile_bits=tile, low_bits=low, flags=flags | L.PQS_PLAN_JIT_PERSISTENT).jit()
    th = rng.random((3, qc.n_true_params)) * 2 * np.pi
    vec = rng.normal(size=1 << n) + 1j * rng.normal(size=1 << n)
    for init in (E.Init.zero(), E.Init.from_vector(vec / np.linalg.norm(vec))):
        assert torch.equal(E.run(a, th, init), E.run(b, th, init)), init.kind
