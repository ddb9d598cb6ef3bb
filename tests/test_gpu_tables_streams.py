"""Device-written instance tables of plans with rolling layouts (each row with
a second buffer of its own), and the entry points that take host inputs or
evolve a pair, on a second context and stream behind busy work."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def pyqc():
    import pyramaterised_amd
    return pyramaterised_amd


def _hea(pyqc, n, layers):
    from pyramaterised_amd import templates as T
    qc = pyqc.PQC(n, jit=n >= 10)  # one form of its plan from the first call on
    qc.add_layers(T.clifford_HE_layers(layers, n))
    return qc


def _busy(x, k=12):
    for _ in range(k):
        x.mul_(1.0000001)


@pytest.mark.parametrize("jit", [False, True])
@pytest.mark.parametrize("dtype", ["complex128", "complex64"])
def test_rolling_batches_with_a_device_written_table(pyqc, dtype, jit):
    """Beyond 42 rows a kernel writes the table: rows packed and padded (the
    second buffers stay packed), every start, in place, and pairs, bit for bit
    the same rows run alone."""
    from pyramaterised_amd import _lib as L
    from pyramaterised_amd import engine as E
    lib = L.lib()
    n, B = 12, 60
    rng = np.random.default_rng(23)
    qc = _hea(pyqc, n, 3)
    plan = E.Plan(n, qc.ops(), dtype=dtype, tile_bits=10, low_bits=2, flags=L.PQS_PLAN_ROLLING)
    assert plan.rolling and plan.n_sweeps > 1
    if jit:
        plan.jit()
    P, dim, cdt = qc.n_true_params, 1 << n, E.CDTYPE[plan.dtype]
    th = rng.random((B, P)) * 2 * np.pi
    vec = rng.normal(size=dim) + 1j * rng.normal(size=dim)
    prod = [v / np.linalg.norm(v) for v in rng.normal(size=(n, 2)) + 1j * rng.normal(size=(n, 2))]
    some = (0, 1, 41, 42, B - 1)
    for init in (E.Init.zero(), E.Init.product(prod), E.Init.from_vector(vec / np.linalg.norm(vec))):
        got = E.run(plan, th, init)
        for b in some:
            assert torch.equal(got[b], E.run(plan, th[b], init)[0]), (init.kind, b)
    rows = torch.as_tensor(rng.normal(size=(B, dim)) + 1j * rng.normal(size=(B, dim))).to(cdt).cuda()
    got = E.run_rows(plan, th, rows.clone())
    for b in some:
        assert torch.equal(got[b], E.run_rows(plan, th[b], rows[b:b + 1].clone())[0]), b
    pad = torch.full((B, dim + 5), 7.0, dtype=cdt, device="cuda")
    pt = E.to_device(th)
    ov = torch.zeros(B // 2, dtype=torch.complex128, device="cuda")
    E.check(lib.pqs_run_batch(E.context().handle, plan.handle, E.ptr(pad), dim + 5, B, E.ptr(pt), P, None, 1, None,
                              None, E.stream_ptr()))
    want = E.run(plan, th, E.Init.zero())
    assert torch.equal(pad[:, :dim].contiguous(), want) and bool((pad[:, dim:] == 7.0).all())
    pad.fill_(7.0)
    E.check(lib.pqs_run_batch_pairs(E.context().handle, plan.handle, E.ptr(pad), dim + 5, B, E.ptr(pt), P, 1, None,
                                    None, E.ptr(ov), E.stream_ptr()))
    st = want.to(torch.complex128).cpu()
    ref = (st[0:B:2].conj() * st[1:B:2]).sum(1)
    # 2^12 products of unit vectors, one rounding of at most 2^-53 each
    assert float((ov.cpu() - ref).abs().max()) < dim * 2.0 ** -53
    assert bool((pad[:, dim:] == 7.0).all())


@pytest.mark.parametrize("n", [6, 11])
def test_host_inputs_and_gradients_on_a_second_stream(pyqc, n):
    """Same bits as on the default context, with the caller's arrays reused at
    once and other work on the default stream meanwhile."""
    from pyramaterised_amd import adjoint
    from pyramaterised_amd import engine as E
    rng = np.random.default_rng(n)
    qc = _hea(pyqc, n, 2)
    P = qc.n_true_params
    plan, full = E.Plan(n, qc.ops()), E.Plan(n, qc.ops(True))
    prog = adjoint.program(qc)
    prog._want_jit = True
    th = rng.random((3, P)) * 2 * np.pi
    init = qc.init()
    want = [E.run(plan, t, init) for t in th]
    want_j = [E.jacobian(full, t, init) for t in th]
    want_g = [adjoint.energy_and_gradient(qc, t) for t in th]
    other, side = E.Context(torch.cuda.current_device()), torch.cuda.Stream()
    x, y = (torch.ones(1 << 26, dtype=torch.float64, device="cuda") for _ in range(2))
    torch.cuda.synchronize()
    _busy(x)
    for i in range(3):
        with E.using(other, side):
            _busy(y, 2)
            buf = th[i].copy()
            got, (psi, J) = E.run(plan, buf, init), E.jacobian(full, buf, init)
            buf[:] = 0.25
            e, g = adjoint.energy_and_gradient(qc, th[i])
        here = E.run(plan, th[i], init)  # the default context's workspace meanwhile
        torch.cuda.synchronize()
        assert torch.equal(got, want[i]) and torch.equal(here, want[i])
        assert torch.equal(psi, want_j[i][0]) and torch.equal(J, want_j[i][1])
        assert e == want_g[i][0] and np.array_equal(g, want_g[i][1])
