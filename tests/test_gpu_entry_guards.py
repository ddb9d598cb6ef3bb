"""Entry points refuse what they cannot run: measurement plans outside
pqs_adjoint, also once the plan is on the device, and host parameter rows
shorter than the plan's slots; the energy gradient without room for the
one-plan pass."""
import ctypes as C

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def pyqc():
    import pyramaterised_amd
    return pyramaterised_amd


def _hea(pyqc, n, layers=2):
    from pyramaterised_amd import templates as T
    qc = pyqc.PQC(n)
    qc.add_layers(T.clifford_HE_layers(layers, n))
    return qc


@pytest.mark.parametrize("n", [5, 10])
def test_measurement_plans_run_with_pqs_adjoint_alone(pyqc, n):
    from pyramaterised_amd import _lib as L
    from pyramaterised_amd import adjoint
    from pyramaterised_amd import engine as E
    lib, ctx = L.lib(), E.context()
    qc = _hea(pyqc, n)
    th = np.random.default_rng(n).random(qc.n_true_params)
    prog = adjoint.program(qc)
    prog._want_jit = True
    adjoint.energy_and_gradient(qc, th)  # the plan is on the device now
    plan, dim = prog.fused_plan(), 1 << (n + 1)
    out = torch.full((2, dim), 7.0, dtype=torch.complex128, device="cuda")
    alt = torch.empty_like(out)
    p = E.to_device(th)
    table = torch.zeros(lib.pqs_batch_table_bytes(2), dtype=torch.uint8, device="cuda")
    st = E.stream_ptr()
    tail = (1, None, E.ptr(alt))
    for rc in (lib.pqs_run_batch_noalloc(ctx.handle, plan.handle, E.ptr(out), dim, 2, E.ptr(p), 0, *tail, None, st),
               lib.pqs_run_table(ctx.handle, plan.handle, E.ptr(table), 2, None, st),
               lib.pqs_batch_table(ctx.handle, plan.handle, E.ptr(out), dim, 2, E.ptr(p), 0, *tail, E.ptr(table), st),
               lib.pqs_run_batch(ctx.handle, plan.handle, E.ptr(out), dim, 2, E.ptr(p), 0, None, 1, None, None, st),
               lib.pqs_jacobian(ctx.handle, plan.handle, E.ptr(p), 1, None, None, E.ptr(out), None, st)):
        assert rc == L.PQS_ERR_UNSUPPORTED
    assert bool((out == 7.0).all())


@pytest.mark.parametrize("kind", ["rotations", "fsim"])
def test_host_rows_cover_the_plan_slots(pyqc, kind):
    from pyramaterised_amd import engine as E
    n = 4
    if kind == "rotations":
        qc = _hea(pyqc, n)
    else:  # the largest slot is fSim's phi
        qc = pyqc.PQC(n)
        qc.add_layer([pyqc.R_y(0, n), pyqc.fSim([1, 2], n)])
    P = qc.n_true_params
    plan, full = E.Plan(n, qc.ops()), E.Plan(n, qc.ops(True))
    th = np.random.default_rng(1).random((2, P))
    assert bool(torch.isfinite(torch.view_as_real(E.run(plan, th, qc.init()))).all())
    for short in (th[:, :P - 1], th[0, :P - 1], np.zeros(0)):
        with pytest.raises(E.EngineError):
            E.run(plan, short, qc.init())
    E.jacobian(full, th[0], qc.init())
    with pytest.raises(E.EngineError):
        E.jacobian(full, th[0, :P - 1], qc.init())
    # a longer vector is fine: the plan reads its slots
    longer = np.concatenate([th, np.full((2, 3), 9.0)], axis=1)
    assert torch.equal(E.run(plan, longer, qc.init()), E.run(plan, th, qc.init()))


def test_gradient_without_room_for_the_one_plan_pass(pyqc, monkeypatch):
    """A failed workspace reservation takes the point-by-point pass: both
    round each amplitude by a few eps per gate, gradients of size <= 4."""
    from pyramaterised_amd import _lib as L
    from pyramaterised_amd import adjoint
    n = 6
    qc = _hea(pyqc, n)
    th = np.random.default_rng(3).random(qc.n_true_params)
    e0, g0 = adjoint.energy_and_gradient(qc, th)
    real = L.lib()

    class NoRoom:
        calls = 0

        def __getattr__(self, name):
            return getattr(real, name)

        def pqs_adjoint(self, *args):
            NoRoom.calls += 1
            return L.PQS_ERR_NOMEM

    monkeypatch.setattr(adjoint.L, "lib", lambda: NoRoom())
    e1, g1 = adjoint.energy_and_gradient(qc, th)
    assert NoRoom.calls == 1
    assert e1 == e0 and np.max(np.abs(g0 - g1)) < 1e-12
