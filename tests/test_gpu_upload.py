"""Host-to-device uploads (pqs_upload, engine.to_device): the bytes land
exactly for every dtype, size and alignment, in stream order behind a busy
stream, beyond the staging ring's buffer count and with the caller reusing
its array at once; a plan first launched on one stream runs correctly on
another stream while its arrays are still being copied on the first."""
import ctypes as C

import numpy as np
import pytest
import torch

from oracle import circuits as OC
from oracle import sim as OS
from tests.helpers import infidelity

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def E():
    from pyramaterised_amd import engine
    return engine


def _busy(x, k=12):
    """Queue about k passes over x (hundreds of MB) on the current stream."""
    for _ in range(k):
        x.mul_(1.0000001)


def test_to_device_dtypes_and_sizes(E):
    rng = np.random.default_rng(3)
    for dt in (np.float64, np.float32, np.complex128, np.complex64, np.int64, np.int32):
        for n in (0, 1, 3, 4, 1000, 1 << 20):
            if np.issubdtype(dt, np.complexfloating):
                a = (rng.random(n) + 1j * rng.random(n)).astype(dt)
            elif np.issubdtype(dt, np.integer):
                a = rng.integers(-2 ** 30, 2 ** 30, n).astype(dt)
            else:
                a = (rng.random(n) * 1e6).astype(dt)
            t = E.to_device(a)
            assert t.is_cuda and tuple(t.shape) == a.shape
            assert np.array_equal(t.cpu().numpy(), a), (dt, n)
    m = rng.random((7, 13))
    assert np.array_equal(E.to_device(m).cpu().numpy(), m)
    assert np.array_equal(E.to_device(m[:, ::2]).cpu().numpy(), m[:, ::2])  # strided input
    with pytest.raises(TypeError):
        E.to_device(np.zeros(3, dtype=np.uint16))


def test_upload_unaligned_destinations_and_errors(E):
    from pyramaterised_amd import _lib as L
    lib = L.lib()
    rng = np.random.default_rng(5)
    buf = torch.zeros(8192, dtype=torch.uint8, device="cuda")
    ctx = E.context().handle
    for off, nb in ((0, 16), (1, 1), (3, 17), (8, 40), (16, 4096), (5, 4000), (0, 4095)):
        src = rng.integers(1, 256, nb, dtype=np.uint8)
        buf.zero_()
        E.check(lib.pqs_upload(ctx, C.c_void_p(buf.data_ptr() + off), C.c_void_p(src.ctypes.data), nb,
                               E.stream_ptr()))
        got = buf.cpu().numpy()
        assert np.array_equal(got[off:off + nb], src), (off, nb)
        assert not got[:off].any() and not got[off + nb:].any(), (off, nb)
    src = np.ones(8, dtype=np.uint8)
    E.check(lib.pqs_upload(ctx, C.c_void_p(buf.data_ptr()), C.c_void_p(src.ctypes.data), 0, E.stream_ptr()))
    for args in ((None, C.c_void_p(buf.data_ptr()), C.c_void_p(src.ctypes.data), 8),
                 (ctx, C.c_void_p(0), C.c_void_p(src.ctypes.data), 8),
                 (ctx, C.c_void_p(buf.data_ptr()), C.c_void_p(0), 8),
                 (ctx, C.c_void_p(buf.data_ptr()), C.c_void_p(src.ctypes.data), -1)):
        with pytest.raises(L.EngineError):
            E.check(lib.pqs_upload(*args, E.stream_ptr()))


def test_uploads_behind_a_busy_stream_beyond_the_ring(E):
    s = torch.cuda.Stream()  # default priority
    x = torch.ones(1 << 27, dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    outs = []
    with torch.cuda.stream(s):
        _busy(x)
        for i in range(80):  # more uploads than staging buffers, all queued behind the busy work
            a = np.full(1000 + 7 * i, float(i))
            outs.append(E.to_device(a))
            a[:] = -1.0  # the caller reuses its array at once
        big = np.arange(1 << 22, dtype=np.float64)  # larger than any staging buffer so far
        t_big = E.to_device(big)
        big[:] = 0.0
        _busy(x, 2)
    torch.cuda.synchronize()
    for i, t in enumerate(outs):
        assert t.numel() == 1000 + 7 * i and bool((t == float(i)).all()), i
    assert np.array_equal(t_big.cpu().numpy(), np.arange(1 << 22, dtype=np.float64))


def test_plan_first_launched_on_another_stream(E):
    import pyramaterised_amd as pyqc
    from pyramaterised_amd import templates as T
    n, p = 10, 5
    rng = np.random.default_rng(9)
    sa, sb = torch.cuda.Stream(), torch.cuda.Stream()
    ca, cb = E.Context(torch.cuda.current_device()), E.Context(torch.cuda.current_device())
    x = torch.ones(1 << 27, dtype=torch.float64, device="cuda")
    og = OC.clifford_he(p, n)
    for jit in (False, True):
        qc = pyqc.PQC(n, jit=jit)
        for layer in T.clifford_HE_layers(p, n):
            qc.add_layer(layer)
        th = rng.random(qc.n_true_params) * 2 * np.pi
        plan, init = qc.plan(), qc.init()
        torch.cuda.synchronize()
        with E.using(ca, sa):
            _busy(x)  # the plan's arrays are copied behind this work on sa
            out_a = E.run(plan, th, init)
        with E.using(cb, sb):  # sb must wait for those copies
            out_b = E.run(plan, th, init)
            out_b2 = E.run(plan, th, init)
        torch.cuda.synchronize()
        want = OS.run(og, th, n)
        for out in (out_a, out_b, out_b2):
            assert infidelity(out.cpu().numpy().ravel(), want) < 1e-12, jit


@pytest.mark.parametrize("off", [0, 8, 3])
def test_upload_sizes_at_the_path_edges(E, off):
    """Largest argument upload (2048 bytes), the smallest staged one, and the
    edges of the staged pieces (512 KB): every byte, and none beyond."""
    from pyramaterised_amd import _lib as L
    lib = L.lib()
    rng = np.random.default_rng(7)
    piece = 512 << 10
    buf = torch.zeros(3 * piece, dtype=torch.uint8, device="cuda")
    ctx = E.context().handle
    for nb in (15, 16, 2032, 2047, 2048, 2049, 2064, piece - 16, piece, piece + 1, piece + 16, 2 * piece + 48):
        src = rng.integers(1, 256, nb, dtype=np.uint8)
        buf.zero_()
        E.check(lib.pqs_upload(ctx, C.c_void_p(buf.data_ptr() + off), C.c_void_p(src.ctypes.data), nb,
                               E.stream_ptr()))
        want = src.copy()
        src.fill(0)  # the caller reuses its array at once
        got = buf.cpu().numpy()
        assert np.array_equal(got[off:off + nb], want), (off, nb)
        assert not got[:off].any() and not got[off + nb:].any(), (off, nb)


@pytest.mark.parametrize("rolling", [False, True])
@pytest.mark.parametrize("dtype", ["complex128", "complex64"])
def test_device_written_batch_tables(E, dtype, rolling):
    """Batches whose instance table a kernel writes (beyond 2048 bytes: 43
    instances) equal the same rows run alone, bit for bit: every initial
    state, shared parameters, padded rows, rows evolved in place
    (their input inside the batch's own rows), and pairs."""
    import pyramaterised_amd as pyqc
    from pyramaterised_amd import templates as T
    from pyramaterised_amd import _lib as L
    lib = L.lib()
    n, B = 7, 60
    rng = np.random.default_rng(11)
    qc = pyqc.PQC(n)
    for layer in T.clifford_HE_layers(3, n):
        qc.add_layer(layer)
    plan = E.Plan(n, qc.ops(), dtype=dtype, tile_bits=5, low_bits=2, flags=L.PQS_PLAN_ROLLING if rolling else 0)
    P, dim, cdt = qc.n_true_params, 1 << n, E.CDTYPE[plan.dtype]
    th = rng.random((B, P)) * 2 * np.pi
    vec = rng.normal(size=dim) + 1j * rng.normal(size=dim)
    vec /= np.linalg.norm(vec)
    prod = [v / np.linalg.norm(v) for v in rng.normal(size=(n, 2)) + 1j * rng.normal(size=(n, 2))]
    for init in (E.Init.zero(), E.Init.product(prod), E.Init.from_vector(vec)):
        got = E.run(plan, th, init)
        for b in (0, 1, 41, 42, B - 1):
            assert torch.equal(got[b], E.run(plan, th[b], init)[0]), (init.kind, b)
    rows = torch.as_tensor(rng.normal(size=(B, dim)) + 1j * rng.normal(size=(B, dim))).to(cdt).cuda()
    want = [E.run_rows(plan, th[b], rows[b:b + 1].clone())[0] for b in range(B)]
    got = E.run_rows(plan, th, rows.clone())
    assert all(torch.equal(got[b], want[b]) for b in range(B))
    # one shared parameter vector, rows 2^n + 5 amplitudes apart, from |0..0>
    p = E.to_device(th[3])
    pad = torch.full((B, dim + 5), 7.0, dtype=cdt, device="cuda")
    E.check(lib.pqs_run_batch(E.context().handle, plan.handle, E.ptr(pad), dim + 5, B, E.ptr(p), 0, None, 1, None,
                              None, E.stream_ptr()))
    one = E.run(plan, th[3], E.Init.zero())[0]
    assert all(torch.equal(pad[b, :dim], one) for b in range(B)) and bool((pad[:, dim:] == 7.0).all())
    # pairs of the padded rows
    ov = torch.zeros(B // 2, dtype=torch.complex128, device="cuda")
    pt = E.to_device(th)
    E.check(lib.pqs_run_batch_pairs(E.context().handle, plan.handle, E.ptr(pad), dim + 5, B, E.ptr(pt), P, 1,
                                    None, None, E.ptr(ov), E.stream_ptr()))
    st = E.run(plan, th, E.Init.zero()).to(torch.complex128).cpu()
    ref = (st[0:B:2].conj() * st[1:B:2]).sum(1)
    # 2^7 products of unit vectors: 128 roundings of at most 2^-53 each
    assert float((ov.cpu() - ref).abs().max()) < 128 * 2.0 ** -53


@pytest.mark.parametrize("dtype", ["complex128", "complex64"])
def test_host_inputs_match_device_inputs(E, dtype):
    """Runs and Jacobians whose inputs travel with the instance table give the
    bits of the same calls with inputs on the GPU: every initial state, row
    counts around the size limit, tangents, and the caller's arrays reused at
    once behind a busy stream."""
    import pyramaterised_amd as pyqc
    from pyramaterised_amd import templates as T
    n = 5
    rng = np.random.default_rng(17)
    qc = pyqc.PQC(n)
    for layer in T.clifford_HE_layers(1, n):
        qc.add_layer(layer)
    P = qc.n_true_params
    plain, full = E.Plan(n, qc.ops(), dtype=dtype), E.Plan(n, qc.ops(True), dtype=dtype)
    vec = rng.normal(size=1 << n) + 1j * rng.normal(size=1 << n)
    prod = [v / np.linalg.norm(v) for v in rng.normal(size=(n, 2)) + 1j * rng.normal(size=(n, 2))]
    x = torch.ones(1 << 26, dtype=torch.float64, device="cuda")
    edge = E.HOST_INPUT_BYTES // (8 * P + 48)
    for init in (E.Init.zero(), E.Init.product(prod), E.Init.from_vector(vec / np.linalg.norm(vec))):
        for B in (1, 2, edge - 1, edge, edge + 1):
            th = rng.random((B, P)) * 2 * np.pi
            dev = torch.as_tensor(th, device="cuda")
            tg = [-1] * (B - 1) + [P - 1]
            _busy(x, 2)
            got, got_t = E.run(plain, th, init), E.run(full, th, init, tangents=tg)
            psi, J = E.jacobian(full, th[0], init)
            want = th[0].copy()
            th[:] = 0.5  # the caller reuses its array at once
            assert torch.equal(got, E.run(plain, dev, init)), (init.kind, B)
            assert torch.equal(got_t, E.run(full, dev, init, tangents=tg)), (init.kind, B)
            pd, Jd = E.jacobian(full, torch.as_tensor(want, device="cuda"), init)
            assert torch.equal(psi, pd) and torch.equal(J, Jd), (init.kind, B)
    with pytest.raises(E.EngineError):
        E.run(full, want, E.Init.zero(), tangents=[P])
    bare = E.Plan(n, [], dtype=dtype)  # no parameters at all
    assert torch.equal(E.run(bare, np.zeros(0), E.Init.zero()), E.run(bare, torch.zeros(1, device="cuda"), E.Init.zero()))
