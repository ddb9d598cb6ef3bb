"""Specialised sweeps with two-qubit gates and Pauli-sum generators against
the interpreted ones: states and Jacobians of the templates that use them, at
the smallest specialised width and with one or more sweeps, and c-number
angles at pi.  Both routes round each amplitude by a few eps per gate (at most
500 gates here), so they differ by less than 1e-12."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _circuit(pyqc, name, n):
    from pyramaterised_amd import templates as T
    layers = {"xxz": lambda: T.XXZ_layers(3, n), "fsim": lambda: T.fSim_circuit_layers(3, n),
              "fixed_fsim": lambda: T.fSim_circuit_layers(3, n, rotator="z", fixed=True),
              "fermionic": lambda: T.fermionic_circuit_layers(1, n), "tfim": lambda: T.TFIM_layers(3, n),
              "rpp": lambda: [[pyqc.R_xx([0, n - 1], n), pyqc.R_y(0, n), pyqc.CNOT([1, 0], n), pyqc.R_yy([0, 2], n),
                               pyqc.R_xx([2, 1], n), pyqc.CNOT([3, 2], n), pyqc.R_yy([n - 1, 2], n)] * 3]}[name]()
    qc = pyqc.PQC(n)
    qc.initial_state = pyqc.tensor([pyqc.basis(2, 1)] * (n // 2) + [pyqc.basis(2, 0)] * (n - n // 2))
    for l in layers:
        qc.add_layer(l)
    return qc


@pytest.mark.parametrize("name", ["xxz", "fsim", "fixed_fsim", "fermionic", "tfim", "rpp"])
@pytest.mark.parametrize("n,tile", [(10, 10), (12, 12), (14, 11)])
def test_specialised_two_qubit_sweeps_match_interpreted(name, n, tile):
    import pyramaterised_amd as pyqc
    from pyramaterised_amd import _lib as L
    from pyramaterised_amd import engine as E
    print(f"two-qubit specialised {name} n={n} tile={tile}", flush=True)
    qc = _circuit(pyqc, name, n)
    P = qc.n_true_params
    th = np.random.default_rng(n).random(P) * 2 * np.pi
    th[::3] = np.pi
    kw = dict(tile_bits=tile, low_bits=3, flags=L.PQS_PLAN_ROLLING)
    for gen in (False, True):
        ops = qc.ops(gen)
        a, b = E.Plan(n, ops, **kw), E.Plan(n, ops, **kw).jit()
        assert len(b.jit_sweep_sources()) == b.n_sweeps  # nothing left to the interpreter
        if gen:
            (p0, j0), (p1, j1) = (E.jacobian(p, th, qc.init()) for p in (a, b))
            assert (j0 - j1).abs().max().item() < 1e-12
        else:
            p0, p1 = (E.run(p, th, qc.init()) for p in (a, b))
        assert (p0 - p1).abs().max().item() < 1e-12
