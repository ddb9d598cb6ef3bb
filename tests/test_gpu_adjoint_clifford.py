"""Energy gradients of small complex128 circuits at angles where rotations are
Clifford gates or flips: cosines of half the angle down to 6e-17, whole layers
of them and one after the other.  Every amplitude is rounded by a few eps per
gate as at any angle, so gradients of size <= 4 agree with the oracle's
2 Re <H psi|d_p psi> to 1e-12."""
import numpy as np
import pytest

from oracle import circuits as OC
from oracle import sim as OS

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def pyqc():
    import pyramaterised_amd
    return pyramaterised_amd


@pytest.mark.parametrize("angles", ["pi", "multiples", "most_then_all"])
@pytest.mark.parametrize("layers", [3, 10])
@pytest.mark.parametrize("n", [3, 4, 5, 6, 7, 8])
def test_gradient_at_clifford_angles(pyqc, n, layers, angles):
    from pyramaterised_amd import adjoint
    from pyramaterised_amd import templates as T
    qc = pyqc.PQC(n)
    for layer in T.clifford_HE_layers(layers, n):
        qc.add_layer(layer)
    H = pyqc.PauliSum(n, {(1,) * 2 + (0,) * (n - 2): 0.5, (0,) * (n - 2) + (3,) * 2: -1.0, (2,) + (0,) * (n - 1): 0.3})
    Hd = H.full()
    og = OC.clifford_he(layers, n)
    P = qc.n_true_params
    rng = np.random.default_rng(100 * n + layers)
    for draw in range(1 if angles == "pi" else 4):
        if angles == "pi":
            th = np.full(P, np.pi)
        elif angles == "multiples":
            th = rng.integers(0, 4, P) * (np.pi / 2)
        else:  # most rotations of a layer, then all of the next one
            th = np.full(P, np.pi)
            th[rng.integers(0, P, P // 8)] = 0.3
        e, g = adjoint.energy_and_gradient(qc, th, H)
        assert adjoint.program(qc).fused_plan() is not None
        psi, d = OS.run(og, th, n), OS.derivative_states(og, th, n)
        hpsi = Hd @ psi
        want = np.array([2 * np.real(np.vdot(hpsi, di)) for di in d])
        assert np.isfinite(g).all(), (draw, np.flatnonzero(~np.isfinite(g)))
        assert abs(e - np.real(np.vdot(psi, hpsi))) < 1e-12
        assert np.max(np.abs(g - want)) < 1e-12, draw


@pytest.mark.parametrize("angles", ["pi", "multiples"])
@pytest.mark.parametrize("n", [9, 11])
def test_specialised_gradient_at_clifford_angles(pyqc, n, angles):
    """The same with specialised sweeps (tiles of 10 bits and more)."""
    from pyramaterised_amd import adjoint
    from pyramaterised_amd import templates as T
    layers = 10
    qc = pyqc.PQC(n)
    for layer in T.clifford_HE_layers(layers, n):
        qc.add_layer(layer)
    H = pyqc.PauliSum(n, {(1,) * 2 + (0,) * (n - 2): 0.5, (0,) * (n - 2) + (3,) * 2: -1.0, (2,) + (0,) * (n - 1): 0.3})
    P = qc.n_true_params
    prog = adjoint.program(qc)
    rng = np.random.default_rng(n)
    for _ in range(1 if angles == "pi" else 4):
        th = np.full(P, np.pi) if angles == "pi" else rng.integers(0, 4, P) * (np.pi / 2)
        prog._fused = False  # point by point
        e0, g0 = adjoint.energy_and_gradient(qc, th, H)
        prog._fused, prog._want_jit = None, True
        e1, g1 = adjoint.energy_and_gradient(qc, th, H)
        assert prog.fused_plan() is not None
        assert np.isfinite(g1).all() and abs(e0 - e1) < 1e-12
        assert np.max(np.abs(g0 - g1)) < 1e-12
