"""The executor of complex128 states below 10 qubits at the edges of its
ranges: every width, batches that do not fill a wave, tiles smaller than the
state, circuits deeper than one angle refill, every op kind, vector and
product starts, tangents.  States against the oracle: each gate rounds every
amplitude by a few eps, so a normalised state of G gates is off by at most
about 4 G eps < 1e-12 at the depths used."""
import numpy as np
import pytest

from helpers import build_oracle, build_pkg, random_spec
from oracle import sim as OS

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def pyqc():
    import pyramaterised_amd
    return pyramaterised_amd


@pytest.mark.parametrize("n", [2, 3, 4, 5, 6, 7, 8, 9])
@pytest.mark.parametrize("batch", [1, 67])
def test_every_op_kind_and_width(pyqc, n, batch):
    from pyramaterised_amd import engine as E
    spec = random_spec(n, 6 if n < 6 else 3, np.random.default_rng(10 * n))
    qc = pyqc.PQC(n)
    qc.add_layer(build_pkg(spec, n, pyqc))
    og = build_oracle(spec, n)
    P = qc.n_true_params
    prm = np.random.default_rng(n).random((batch, P)) * 2 * np.pi
    plan = E.Plan(n, qc.ops())
    got = E.run(plan, prm, qc.init()).cpu().numpy()
    for b in sorted({0, batch // 2, batch - 1}):
        ref = OS.run(og, prm[b], n)
        assert np.linalg.norm(got[b] - ref) / np.linalg.norm(ref) < 1e-12
    # the same rows alone: a result does not depend on its place in a wave
    alone = E.run(plan, prm[batch - 1], qc.init()).cpu().numpy()[0]
    assert np.array_equal(alone, got[batch - 1])


@pytest.mark.parametrize("n,tile", [(7, 2), (7, 4), (11, 5), (12, 9), (10, 9)])
def test_tiles_smaller_than_the_state(pyqc, n, tile):
    """Several tiles per state: control and phase bits outside the tile."""
    from pyramaterised_amd import engine as E
    spec = random_spec(n, 2, np.random.default_rng(n + tile))
    spec = [x for x in spec if x[0] != "shared_Rx"]  # a generator, not a tile matter
    qc = pyqc.PQC(n)
    qc.add_layer(build_pkg(spec, n, pyqc))
    prm = np.random.default_rng(3).random((3, qc.n_true_params)) * 2 * np.pi
    got = E.run(E.Plan(n, qc.ops(), tile_bits=tile, low_bits=1), prm, qc.init()).cpu().numpy()
    og = build_oracle(spec, n)
    for b in range(3):
        ref = OS.run(og, prm[b], n)
        assert np.linalg.norm(got[b] - ref) / np.linalg.norm(ref) < 1e-12


@pytest.mark.parametrize("n", [2, 4, 6, 9])
def test_deep_layers_and_angles_at_pi(pyqc, n):
    """More layers than one angle refill and one growth check cover, half of
    the angles at and next to pi."""
    from pyramaterised_amd import engine as E
    from pyramaterised_amd import templates as T
    from oracle import circuits as OC
    layers = 30
    qc = pyqc.PQC(n)
    qc.add_layers(T.qg_circuit_layers(layers, n))
    th = np.random.default_rng(n).random(qc.n_true_params) * 2 * np.pi
    th[::2] = np.pi + np.array([0.0, 1e-9, -1e-14])[np.arange(len(th[::2])) % 3]
    og = OC.qg_circuit(layers, n)
    ref = OS.run(og, th, n)
    got = E.run(E.Plan(n, qc.ops()), th, qc.init()).cpu().numpy()[0]
    assert np.linalg.norm(got - ref) < 1e-11  # 2700 gates at 4 eps
    # from a state vector, and in place over it
    from_vec = E.run(E.Plan(n, qc.ops()), th, E.Init.from_vector(ref)).cpu().numpy()[0]
    rows = E.Init.from_vector(ref).device_args(0, E.device())[1].reshape(1, -1).clone()
    E.run_rows(E.Plan(n, qc.ops()), th, rows)
    assert np.array_equal(rows.cpu().numpy()[0], from_vec)
