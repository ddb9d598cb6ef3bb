"""Host side of the energy gradient: which circuits take the one-plan pass."""
import pytest

import pyramaterised_amd as pyqc
from pyramaterised_amd import adjoint
from pyramaterised_amd import engine as E


@pytest.mark.parametrize("n,fused", [(16, True), (29, True), (30, False), (32, False)])
def test_one_plan_pass_only_where_its_workspace_fits(n, fused, monkeypatch):
    """The pass needs two buffers of 2^(n+1) amplitudes beside the pair: 32
    GiB at 29 qubits, and 256 GiB next to the pair's 128 at 32, where the
    point-by-point pass needs none."""
    monkeypatch.setattr(E.Plan, "jit", lambda self: self)  # planning only: no device here
    qc = pyqc.PQC(n)
    qc.add_layer([pyqc.R_y(q, n) for q in range(n)])
    prog = adjoint.AdjointProgram(qc)
    prog._want_jit = True
    assert (prog.fused_plan() is not None) == fused
