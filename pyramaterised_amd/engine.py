"""Device layer: contexts, plans and the calls into libpqs on torch tensors.

PyTorch provides device memory and the current HIP stream; all arithmetic of
the hot path runs in libpqs's HIP kernels.  Every function here requires a
gfx950 GPU and raises ``EngineError`` otherwise.
"""
import contextlib
import ctypes as C
import hashlib
import json
import os
import subprocess
import sys
import tempfile
import threading

import numpy as np
import torch

from . import _lib as L
from ._lib import EngineError, check

_tls = threading.local()

CDTYPE = {L.PQS_C128: torch.complex128, L.PQS_C64: torch.complex64}
DTYPES = {"complex128": L.PQS_C128, "c128": L.PQS_C128, "complex64": L.PQS_C64, "c64": L.PQS_C64}


def dtype_code(dtype):
    if isinstance(dtype, int):
        return dtype
    if dtype in (torch.complex128, np.complex128):
        return L.PQS_C128
    if dtype in (torch.complex64, np.complex64):
        return L.PQS_C64
    try:
        return DTYPES[str(dtype)]
    except KeyError:
        raise ValueError(f"unsupported state dtype {dtype!r}") from None


def device():
    """The torch device the engine runs on (current CUDA/HIP device)."""
    # (an initialised runtime has a device; asking again costs 2 us)
    if not torch.cuda.is_initialized() and not torch.cuda.is_available():
        raise EngineError("no GPU visible: the statevector engine runs only on gfx950 (MI355X)")
    return torch.device("cuda", torch.cuda.current_device())


class Context:
    """libpqs context on one device (one per device per host thread)."""

    def __init__(self, dev_index):
        self.handle = C.c_void_p()
        self.device_index = dev_index
        check(L.lib().pqs_ctx_create(dev_index, C.byref(self.handle)))
        n_cu, lds = C.c_int32(), C.c_int32()
        arch = C.create_string_buffer(64)
        check(L.lib().pqs_device_info(self.handle, C.byref(n_cu), C.byref(lds), arch, 64))
        self.n_cu, self.max_lds, self.arch = n_cu.value, lds.value, arch.value.decode()

    def set_max_blocks(self, max_blocks):
        """Cap the blocks of one sweep launch (0: no cap); a larger batched
        sweep is split over instance ranges, with the same results.  Short
        kernels of other streams then wait at most one such launch."""
        check(L.lib().pqs_ctx_set_max_blocks(self.handle, int(max_blocks)))

    def __del__(self):
        h = getattr(self, "handle", None)
        if h and h.value:
            try:
                L.lib().pqs_ctx_destroy(h)
            except Exception:
                pass


def context():
    o = getattr(_tls, "override", None)
    if o is not None:
        return o
    dev = device()
    ctxs = getattr(_tls, "ctxs", None)
    if ctxs is None:
        ctxs = _tls.ctxs = {}
    c = ctxs.get(dev.index)
    if c is None:
        c = ctxs[dev.index] = Context(dev.index)
    return c


@contextlib.contextmanager
def using(ctx, stream):
    """Issue engine calls on ``stream`` with context ``ctx``.  A context's
    workspace serves one stream at a time, so work spread over several
    streams needs one context per stream."""
    prev = getattr(_tls, "override", None)
    _tls.override = ctx
    try:
        with torch.cuda.stream(stream):
            yield
    finally:
        _tls.override = prev


@contextlib.contextmanager
def marked(name):
    """A named profiler range (roctx, seen by rocprofv3 --marker-trace when
    PQS_ROCTX=1) around the block; nothing otherwise."""
    lib = L.lib()
    check(lib.pqs_range_push(str(name).encode()))
    try:
        yield
    finally:
        lib.pqs_range_pop()


_CHILD = r"""
import ctypes, sys
lib = ctypes.CDLL(sys.argv[1])
lib.pqs_jit_prepare.argtypes = [ctypes.c_char_p, ctypes.c_int64]
for path in sys.argv[2:]:
    src = open(path, "rb").read()
    if lib.pqs_jit_prepare(src, len(src)) != 0:
        sys.exit(1)
"""


def _compile_in_children(srcs, workers):
    """Compile kernel sources into the code-object cache with child
    processes that load only libpqs (never the GPU)."""
    with tempfile.TemporaryDirectory() as d:
        paths = []
        for i, s in enumerate(srcs):
            p = os.path.join(d, f"s{i}.hip")
            with open(p, "wb") as f:
                f.write(s)
            paths.append(p)
        groups = [paths[i::workers] for i in range(min(workers, len(paths)))]
        procs = [subprocess.Popen([sys.executable, "-c", _CHILD, L.LIB_PATH] + g) for g in groups]
        for pr in procs:
            pr.wait()
        # failures are reported by the in-process compile that follows


def max_tile_bits(dtype_c):
    """Largest tile (qubits) whose amplitudes fit in one workgroup's LDS."""
    lds = context().max_lds
    amp = 16 if dtype_c == L.PQS_C128 else 8
    k = 1
    while (2 ** (k + 1)) * amp <= lds and k + 1 <= (13 if dtype_c == L.PQS_C128 else 14):
        k += 1
    return k


def jit_cache_dir():
    """Directory of the code-object cache (PQS_JIT_CACHE, default
    $TMPDIR/pqs_jit_cache); tuning decisions are kept beside the code."""
    env = os.environ.get("PQS_JIT_CACHE")
    return env if env else os.path.join(os.environ.get("TMPDIR", "/tmp"), "pqs_jit_cache")


def tile_candidates(n, dtype_c):
    """Tile shapes (tile bits, forced low bits, flags) the tuner times.

    c128: 12-bit tiles (64 KiB of LDS, two resident blocks per CU, so one
    block's LDS phases overlap the other's HBM traffic) and 11-bit tiles
    (five blocks per CU) with rolling layouts (the tile moves freely over
    the qubits; out of place) and 128 B or 256 B write runs, or fixed low
    qubits (in place); 12-bit rolling tiles with and without exchange
    transitions.  c64: 11- to 13-bit tiles (16-64 KiB).  Which wins
    depends on the circuit and the batch: deep sweeps favour more resident
    blocks, shallow HBM-bound ones larger tiles.
    """
    R = L.PQS_PLAN_ROLLING
    if dtype_c == L.PQS_C128:
        # register-phase transitions by cross-lane swaps save LDS round trips
        # but keep flips and scales materialised across them: timed both ways
        c = [(11, 3, R), (12, 4, R), (12, 4, R | L.PQS_PLAN_NO_EXCHANGE), (12, 3, R), (12, 4, 0)]
    else:
        c = [(12, 4, R), (13, 4, R), (11, 4, R), (13, 4, 0)]
    out = []
    for k, low, fl in c:
        k = min(k, n)
        cand = (k, min(low, k), fl)
        if cand not in out:
            out.append(cand)
    return out


def _n_params(ops):
    return 1 + max([-1] + [max(o.slot, o.slot2) for o in ops])


def tuned_plan(n_qubits, ops, dtype_c, batch, init, workers=None, pairs=False):
    """Build the plan for each tile shape of ``tile_candidates``, specialise
    all of them, time evolutions of each on this GPU (random angles, up to
    2^28 amplitudes of the batch; the median of five interleaved rounds) and
    return the first candidate within TUNE_TOLERANCE of the fastest.  With
    ``pairs`` the timed call is the pair run (``run_pairs``: the last sweep
    as the pair kernel), which the caller will make.  The choice is cached
    in memory and in the code-object cache directory, keyed by the op list,
    the dtype, the timed batch size and the call."""
    cands = tile_candidates(n_qubits, dtype_c)
    arr = (L.Op * max(1, len(ops)))(*ops)
    B = 1 if n_qubits >= 26 else max(1, min(int(batch), (1 << 28) >> n_qubits))
    pairs = bool(pairs) and B >= 2
    if pairs:
        B -= B % 2
    key = hashlib.sha1(bytes(arr) + repr((n_qubits, dtype_c, B, cands, pairs)).encode() +
                       L.library_fingerprint().encode()).hexdigest()[:24]
    choice = _tune_memo.get(key)
    path = os.path.join(jit_cache_dir(), f"tune_{key}.json")
    if choice is None and os.path.exists(path):
        try:
            with open(path) as f:
                choice = tuple(json.load(f)["shape"])
        except (OSError, ValueError, KeyError):
            choice = None
    if choice is not None and tuple(choice) in cands:
        return Plan(n_qubits, ops, dtype_c, tile_bits=choice[0], low_bits=choice[1], flags=choice[2]).jit(workers=workers)
    plans = [Plan(n_qubits, ops, dtype_c, tile_bits=k, low_bits=lo, flags=fl) for k, lo, fl in cands]
    if workers is None:
        workers = min(16, os.cpu_count() or 1)
    srcs = [s for p in plans for s in p.jit_sweep_sources()]
    if workers > 1 and len(srcs) > 1:
        _compile_in_children(srcs, workers)
    for p in plans:
        p.jit(workers=1)
    dev = device()
    g = torch.Generator(device="cpu").manual_seed(1)
    th = (torch.rand((B, max(1, _n_params(ops))), generator=g, dtype=torch.float64) * 2 * np.pi).to(dev)
    out = torch.empty((B, 1 << n_qubits), dtype=CDTYPE[dtype_c], device=dev)
    ov = torch.empty(max(1, B // 2), dtype=torch.complex128, device=dev)

    def call(p):
        if pairs:
            run_pairs(p, th, init, out=out, overlaps=ov)
        else:
            run(p, th, init, out=out)

    # five interleaved rounds, the median of each candidate: a single pass
    # in candidate order favours the later ones (the first timings of a
    # process run while the clocks ramp up), and the fastest of a few
    # rounds follows outliers (16 qubits, 2048 states: the 12-bit plan's
    # best round 2% under the 11-bit plan's, which is 4% faster at 10,000)
    rounds = [[] for _ in plans]
    for _ in range(5):
        for i, p in enumerate(plans):
            call(p)
            s, e = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            s.record()
            for _ in range(2):
                call(p)
            e.record()
            e.synchronize()
            rounds[i].append(s.elapsed_time(e))
    times = [float(np.median(r)) for r in rounds]
    del out, ov
    best = pick_candidate(times)
    _tune_memo[key] = cands[best]
    try:
        os.makedirs(jit_cache_dir(), exist_ok=True)
        with open(path, "w") as f:
            json.dump({"shape": list(cands[best]), "candidates": [list(c) for c in cands],
                       "ms_per_run": [t / 2 for t in times], "batch": B, "pairs": pairs}, f)
    except OSError:
        pass
    return plans[best]


_tune_memo = {}
TUNE_TOLERANCE = 0.015


def pick_candidate(times, tolerance=None):
    """Index of the first candidate (in list order) whose time is within
    ``tolerance`` (default TUNE_TOLERANCE) of the fastest: near-ties do not
    flip the choice from box to box."""
    tol = TUNE_TOLERANCE if tolerance is None else tolerance
    fastest = min(times)
    return next(i for i, t in enumerate(times) if t <= fastest * (1 + tol))


def stream_ptr():
    return C.c_void_p(torch.cuda.current_stream().cuda_stream)


def ptr(t):
    return C.c_void_p(t.data_ptr()) if t is not None else C.c_void_p(0)


class Plan:
    """A compiled op list (pqs_plan).  Host-only to build; runs on the GPU."""

    def __init__(self, n_qubits, ops, dtype=L.PQS_C128, tile_bits=0, low_bits=0, block=0, flags=0):
        self.n = int(n_qubits)
        self.dtype = dtype_code(dtype)
        if tile_bits == 0 and torch.cuda.is_available():
            tile_bits = max_tile_bits(self.dtype)
        self.n_ops = len(ops)
        self.flags = int(flags)
        arr = (L.Op * max(1, len(ops)))(*ops)
        opts = L.PlanOpts(tile_bits, low_bits, block, self.dtype, flags)
        self.handle = C.c_void_p()
        check(L.lib().pqs_plan_create(self.n, arr, len(ops), C.byref(opts), C.byref(self.handle)))
        ns, tb, ne, nt = C.c_int32(), C.c_int32(), C.c_int32(), C.c_int32()
        check(L.lib().pqs_plan_info(self.handle, C.byref(ns), C.byref(tb), C.byref(ne), C.byref(nt)))
        self.n_sweeps, self.tile_bits, self.n_exec, self.n_tangents = ns.value, tb.value, ne.value, nt.value
        self.jitted = False

    def __del__(self):
        h = getattr(self, "handle", None)
        if h and h.value:
            try:
                L.lib().pqs_plan_destroy(h)
            except Exception:
                pass

    def sweeps(self):
        """[(tile_qubits, op_indices)] for every sweep (host-side description)."""
        out = []
        for s in range(self.n_sweeps):
            tq = (C.c_int32 * 64)()
            oi = (C.c_int32 * max(1, self.n_ops))()
            nt, no = C.c_int32(), C.c_int32()
            check(L.lib().pqs_plan_sweep(self.handle, s, tq, C.byref(nt), oi, C.byref(no)))
            out.append((list(tq[:nt.value]), list(oi[:no.value])))
        return out

    def layouts(self):
        """[(read_pos, write_pos)] per sweep: bit position of every qubit in
        the layout the sweep reads and the one it writes."""
        out = []
        for s in range(self.n_sweeps):
            r, w = (C.c_int32 * self.n)(), (C.c_int32 * self.n)()
            check(L.lib().pqs_plan_sweep_layout(self.handle, s, r, w))
            out.append((list(r), list(w)))
        return out

    @property
    def rolling(self):
        return any(r != w for r, w in self.layouts())

    def jit(self, load=True, workers=None):
        """Specialise the plan's sweeps into straight-line kernels (hiprtc);
        with load, later runs on this device use them.  hiprtc serialises
        compiles within a process, so the sweeps are compiled by ``workers``
        child processes (no GPU use) into the shared code-object cache
        first."""
        srcs = self.jit_sweep_sources()
        if workers is None:
            workers = min(16, os.cpu_count() or 1)
        if workers > 1 and len(srcs) > 1:
            _compile_in_children(srcs, workers)
        ctx = context() if load else None
        check(L.lib().pqs_plan_jit(ctx.handle if ctx else None, self.handle, 1 if load else 0))
        self.jitted = bool(load)
        return self

    def jit_sweep_sources(self):
        out = []
        for s in range(self.n_sweeps):
            n = C.c_int64()
            check(L.lib().pqs_plan_jit_sweep_source(self.handle, s, None, 0, C.byref(n)))
            if n.value == 0:
                continue
            buf = C.create_string_buffer(n.value + 1)
            check(L.lib().pqs_plan_jit_sweep_source(self.handle, s, buf, n.value + 1, C.byref(n)))
            out.append(buf.value)
        return out

    def jit_source(self):
        n = C.c_int64()
        ns = C.c_int32()
        check(L.lib().pqs_plan_jit_source(self.handle, None, 0, C.byref(n), C.byref(ns)))
        buf = C.create_string_buffer(n.value + 1)
        check(L.lib().pqs_plan_jit_source(self.handle, buf, n.value + 1, C.byref(n), C.byref(ns)))
        return buf.value.decode(), ns.value

    def tangent_sweep(self, t):
        s = C.c_int32()
        check(L.lib().pqs_plan_tangent_sweep(self.handle, t, C.byref(s)))
        return s.value

    def tangent_parts(self, t):
        """Parts the generator of tangent t was split into (1: unsplit)."""
        n = C.c_int32()
        check(L.lib().pqs_plan_tangent_parts(self.handle, t, C.byref(n)))
        return n.value


# ------------------------------------------------------------------- init state

_ZERO_KET = np.array([1.0, 0.0])
_ZERO_KET_TOL = 1e-8 + 1e-5 * _ZERO_KET


class Init:
    """Initial state of a run: |0..0>, a product state (per-qubit 2-vectors),
    or a full state vector."""

    def __init__(self, kind, table=None, vector=None):
        self.kind = kind  # "zero" | "product" | "vector"
        self.table = table
        self.vector = vector

    @staticmethod
    def zero():
        return Init("zero")

    @staticmethod
    def product(factors):
        t = np.asarray([np.asarray(f, dtype=np.complex128).ravel() for f in factors])
        if t.ndim != 2 or t.shape[1] != 2:
            raise ValueError("product initial state needs one 2-vector per qubit")
        # np.allclose(t, [1, 0]) at its default tolerances, spelled out: 2 us
        # against 20 us, which a 4-qubit call notices
        if (np.abs(t - _ZERO_KET) <= _ZERO_KET_TOL).all():
            return Init("zero")
        return Init("product", table=t)

    @staticmethod
    def from_vector(v):
        return Init("vector", vector=v)

    def device_args(self, dtype_c, dev):
        """(init code, src tensor or None, table tensor or None)."""
        if self.kind == "zero":
            return 1, None, None
        npdt = np.complex128 if CDTYPE[dtype_c] == torch.complex128 else np.complex64
        if self.kind == "product":
            if dev == device():
                return 2, None, to_device(np.asarray(self.table).reshape(-1), npdt)
            return 2, None, torch.as_tensor(self.table.reshape(-1), dtype=CDTYPE[dtype_c], device=dev)
        v = self.vector
        if not torch.is_tensor(v) and dev == device():
            return 0, to_device(np.asarray(v).reshape(-1), npdt), None
        if not torch.is_tensor(v):
            v = torch.as_tensor(np.asarray(v).reshape(-1))
        v = v.to(device=dev, dtype=CDTYPE[dtype_c]).contiguous()
        return 0, v, None


# ------------------------------------------------------------------ entry points

_NP_TO_TORCH = {np.dtype(np.float64): torch.float64, np.dtype(np.float32): torch.float32,
                np.dtype(np.complex128): torch.complex128, np.dtype(np.complex64): torch.complex64,
                np.dtype(np.int64): torch.int64, np.dtype(np.int32): torch.int32}


def to_device(a, dtype=None):
    """Host array -> device tensor on the current device, in the current
    stream's order.  The bytes are staged in the context's pinned buffers
    before this returns and a kernel on the stream copies them (pqs_upload),
    so the host does not wait for the stream's earlier work and the copy
    does not queue behind other streams' DMA copies."""
    a = np.ascontiguousarray(a, dtype=dtype)
    if a.dtype not in _NP_TO_TORCH:
        raise TypeError(f"to_device: unsupported dtype {a.dtype}")
    t = torch.empty(a.shape, dtype=_NP_TO_TORCH[a.dtype], device=device())
    if a.nbytes:
        check(L.lib().pqs_upload(context().handle, ptr(t), C.c_void_p(a.ctypes.data), a.nbytes, stream_ptr()))
    return t


def _params_tensor(params, dev, rows=None):
    if torch.is_tensor(params) and (params.is_cuda or params.requires_grad):
        p = params.to(device=dev, dtype=torch.float64).contiguous()
    else:
        host = params.to(torch.float64).numpy() if torch.is_tensor(params) else params
        if dev != device():
            raise ValueError("parameters on the host go to the current device only")
        p = to_device(np.asarray(host, dtype=np.float64))
    if rows is not None and p.dim() == 1:
        p = p.unsqueeze(0)
    return p


# run(): inputs up to this many bytes (48 a row for the instance table) go to
# the GPU as one launch's argument (2048 bytes with the table's padding): one
# 4-qubit state 43 -> 27 us.  Larger batches keep their own upload, whose rows
# need no workspace.
HOST_INPUT_BYTES = 1536


def _host_rows(params):
    """Host parameters as float64 rows (B, P), at least one column; None for
    device or differentiable tensors and other shapes."""
    if torch.is_tensor(params):
        if params.is_cuda or params.requires_grad:
            return None
        params = params.to(torch.float64).numpy()
    a = np.asarray(params, dtype=np.float64)
    if a.ndim not in (1, 2):
        return None
    a = np.ascontiguousarray(a.reshape(1, -1) if a.ndim == 1 else a)
    return a if a.size else np.zeros((max(1, a.shape[0]), 1))


def _host_init(init, dtype_c, dev):
    """(init code, source tensor or None, host table or None)."""
    if init.kind != "product":
        code, src, _ = init.device_args(dtype_c, dev)
        return code, src, None
    npdt = np.complex128 if CDTYPE[dtype_c] == torch.complex128 else np.complex64
    return 2, None, np.ascontiguousarray(np.asarray(init.table).reshape(-1), dtype=npdt)


def _np_ptr(a):
    return C.c_void_p(a.ctypes.data) if a is not None else C.c_void_p(0)


def run(plan, params, init, tangents=None, out=None):
    """Evolve a batch: params (B, P) or (P,) -> states (B, 2^N).

    tangents: None or a length-B sequence of tangent indices (-1 = plain).
    """
    ctx = context()
    dev = device()
    rows = _host_rows(params)
    small = rows is not None and rows.nbytes + 48 * rows.shape[0] + (
        32 * plan.n if init.kind == "product" else 0) <= HOST_INPUT_BYTES
    if small:
        p = rows
    else:
        p = _params_tensor(params, dev, rows=True)
        if p.numel() == 0:
            p = torch.zeros((max(1, p.shape[0]) if p.dim() == 2 else 1, 1), dtype=torch.float64, device=dev)
    B = p.shape[0]
    dim = 1 << plan.n
    cdt = CDTYPE[plan.dtype]
    if out is None:
        out = torch.empty((B, dim), dtype=cdt, device=dev)
    elif out.shape != (B, dim) or out.dtype != cdt or not out.is_contiguous():
        raise ValueError("out has the wrong shape, dtype or layout")
    tg = None
    if tangents is not None:
        tg = (C.c_int32 * B)(*[int(t) for t in tangents])
    if small:
        code, src, tab = _host_init(init, plan.dtype, dev)
        check(L.lib().pqs_run_batch_host(ctx.handle, plan.handle, ptr(out), dim, B, _np_ptr(p), p.shape[1], tg, code,
                                         ptr(src), _np_ptr(tab), stream_ptr()))
        if src is not None:
            _keepalive(src)
        return out
    code, src, tab = init.device_args(plan.dtype, dev)
    pstride = p.stride(0) if p.shape[0] > 1 else 0
    check(L.lib().pqs_run_batch(ctx.handle, plan.handle, ptr(out), dim, B, ptr(p), pstride, tg, code, ptr(src),
                                ptr(tab), stream_ptr()))
    # keep temporaries alive until the stream has consumed them
    _keepalive(src, tab, p)
    return out


def run_pairs(plan, params, init, out=None, overlaps=None):
    """Evolve an even batch (params (B, P)) and return (states (B, 2^N),
    overlaps (B/2,) complex128) with overlaps[i] = <state_2i|state_2i+1>
    (pqs_run_batch_pairs: a plan with specialised sweeps forms the overlaps
    in its last sweep, without reading the states back)."""
    ctx = context()
    dev = device()
    p = _params_tensor(params, dev, rows=True)
    if p.numel() == 0:
        p = torch.zeros((max(1, p.shape[0]) if p.dim() == 2 else 1, 1), dtype=torch.float64, device=dev)
    B = p.shape[0]
    if B % 2:
        raise ValueError("run_pairs needs an even batch")
    dim = 1 << plan.n
    cdt = CDTYPE[plan.dtype]
    if out is None:
        out = torch.empty((B, dim), dtype=cdt, device=dev)
    elif out.shape != (B, dim) or out.dtype != cdt or not out.is_contiguous():
        raise ValueError("out has the wrong shape, dtype or layout")
    if overlaps is None:
        overlaps = torch.empty(B // 2, dtype=torch.complex128, device=dev)
    elif overlaps.shape != (B // 2,) or overlaps.dtype != torch.complex128 or not overlaps.is_contiguous():
        raise ValueError("overlaps has the wrong shape, dtype or layout")
    code, src, tab = init.device_args(plan.dtype, dev)
    pstride = p.stride(0) if p.shape[0] > 1 else 0
    check(L.lib().pqs_run_batch_pairs(ctx.handle, plan.handle, ptr(out), dim, B, ptr(p), pstride, code, ptr(src),
                                      ptr(tab), ptr(overlaps), stream_ptr()))
    _keepalive(src, tab, p)
    return out, overlaps


def run_multi(jobs):
    """Evolve batches of several plans in one multi-plan run (pqs_run_multi):
    jobs = [(plan, params (B, P) or (P,), Init)] -> list of (B, 2^N_plan)
    state tensors.  The plans may differ in width and depth (one launch per
    sweep round and tile size covers all of them)."""
    ctx = context()
    dev = device()
    plans, outs, keep = [], [], []
    insts, inst_plan, tabs = [], [], []
    for plan, params, init in jobs:
        if plan.dtype != jobs[0][0].dtype:
            raise ValueError("multi-plan runs take plans of one dtype")
        k = len(plans)
        plans.append(plan)
        p = _params_tensor(params, dev, rows=True)
        if p.numel() == 0:
            p = torch.zeros((max(1, p.shape[0]), 1), dtype=torch.float64, device=dev)
        B = p.shape[0]
        out = torch.empty((B, 1 << plan.n), dtype=CDTYPE[plan.dtype], device=dev)
        code, src, tab = init.device_args(plan.dtype, dev)
        keep += [p, src, tab]
        for b in range(B):
            inst = L.Instance()
            inst.state_dev = out[b].data_ptr()
            inst.src_dev = src.data_ptr() if src is not None else None
            inst.params_dev = p[b].data_ptr()
            inst.tangent = -1
            inst.init = code
            insts.append(inst)
            inst_plan.append(k)
            tabs.append(tab.data_ptr() if tab is not None else None)
        outs.append(out)
    n = len(insts)
    if n == 0:
        return outs
    parr = (C.c_void_p * len(plans))(*[pl.handle.value for pl in plans])
    iarr = (L.Instance * n)(*insts)
    ipl = (C.c_int32 * n)(*inst_plan)
    tarr = (C.c_void_p * n)(*tabs)
    check(L.lib().pqs_run_multi(ctx.handle, parr, len(plans), iarr, ipl, tarr, n, stream_ptr()))
    _keepalive(*keep)
    return outs


def run_rows(plan, params, states):
    """Evolve every row of a (B, 2^N) state tensor in place through the plan
    (row b with params[b], or one shared (P,) vector) -> states."""
    ctx = context()
    dev = states.device
    p = _params_tensor(params, dev, rows=True)
    if p.numel() == 0:
        p = torch.zeros((1, 1), dtype=torch.float64, device=dev)
    B, dim = states.shape
    if not states.is_contiguous() or dim != 1 << plan.n or states.dtype != CDTYPE[plan.dtype]:
        raise ValueError("states must be a contiguous (B, 2^N) tensor of the plan's dtype")
    pstride = p.stride(0) if p.shape[0] > 1 else 0
    if p.shape[0] not in (1, B):
        raise ValueError("params must have one row or one row per state")
    check(L.lib().pqs_run_batch(ctx.handle, plan.handle, ptr(states), dim, B, ptr(p), pstride, None, 0, None,
                                None, stream_ptr()))
    _keepalive(p)
    return states


class BatchGraph:
    """All sweep launches of one batched run captured in a HIP graph.

    The instance table is written once into a device buffer owned by this
    object (``pqs_batch_table``); the capture holds only kernel launches
    (``pqs_run_table``).  ``replay()`` re-runs the evolution on the same
    buffers: update ``self.params`` (and the source state, if any) in place
    between replays.  Rolling-layout plans get their second buffer here."""

    def __init__(self, plan, params, init, out=None):
        ctx = context()
        dev = device()
        self.plan = plan
        self.params = _params_tensor(params, dev, rows=True).clone()
        B = self.params.shape[0]
        dim = 1 << plan.n
        cdt = CDTYPE[plan.dtype]
        self.out = out if out is not None else torch.empty((B, dim), dtype=cdt, device=dev)
        if self.out.shape != (B, dim) or self.out.dtype != cdt or not self.out.is_contiguous():
            raise ValueError("out has the wrong shape, dtype or layout")
        code, src, tab = init.device_args(plan.dtype, dev)
        self._src, self._tab = src, tab
        # the second buffer of rolling layouts; a plan asked for them with more
        # than one sweep may use them even where every layout it reports is
        # standard, and a plan that does not ignores the buffer
        need_alt = plan.rolling or (plan.flags & L.PQS_PLAN_ROLLING and plan.n_sweeps > 1)
        self.alt = torch.empty_like(self.out) if need_alt else None
        nb = L.lib().pqs_batch_table_bytes(B)
        self.table = torch.empty(nb, dtype=torch.uint8, device=dev)
        check(L.lib().pqs_batch_table(ctx.handle, plan.handle, ptr(self.out), dim, B, ptr(self.params),
                                      self.params.shape[1], code, ptr(src), ptr(self.alt), ptr(self.table),
                                      stream_ptr()))
        self._launch()  # eager once: device image, kernel attributes
        torch.cuda.synchronize()
        self.graph = torch.cuda.CUDAGraph()
        side = torch.cuda.Stream()  # default priority
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            with torch.cuda.graph(self.graph, stream=side):
                self._launch()
        torch.cuda.current_stream().wait_stream(side)

    def _launch(self):
        check(L.lib().pqs_run_table(context().handle, self.plan.handle, ptr(self.table), self.params.shape[0],
                                    ptr(self._tab), stream_ptr()))

    def replay(self):
        self.graph.replay()
        return self.out


def jacobian(plan, params, init, psi_out=None, jac_out=None):
    """psi (2^N,), J (n_tangents, 2^N) in one forward pass."""
    ctx = context()
    dev = device()
    dim = 1 << plan.n
    cdt = CDTYPE[plan.dtype]
    psi = psi_out if psi_out is not None else torch.empty(dim, dtype=cdt, device=dev)
    J = jac_out if jac_out is not None else torch.empty((max(plan.n_tangents, 0), dim), dtype=cdt, device=dev)
    rows = _host_rows(params)
    if rows is not None:
        code, src, tab = _host_init(init, plan.dtype, dev)
        check(L.lib().pqs_jacobian_host(ctx.handle, plan.handle, _np_ptr(rows), rows.size, code, ptr(src), _np_ptr(tab),
                                        ptr(psi), ptr(J) if plan.n_tangents > 0 else C.c_void_p(0), stream_ptr()))
        if src is not None:
            _keepalive(src)
        return psi, J
    p = _params_tensor(params, dev)
    if p.numel() == 0:
        p = torch.zeros(1, dtype=torch.float64, device=dev)
    code, src, tab = init.device_args(plan.dtype, dev)
    check(L.lib().pqs_jacobian(ctx.handle, plan.handle, ptr(p), code, ptr(src), ptr(tab), ptr(psi),
                               ptr(J) if plan.n_tangents > 0 else C.c_void_p(0), stream_ptr()))
    _keepalive(src, tab, p)
    return psi, J


def inner_pairs(states, a_idx, b_idx):
    """<s_a|s_b> for rows of a (B, dim) tensor -> complex128 (n_pairs,)."""
    ctx = context()
    dev = states.device
    if states.dim() == 1:
        states = states.unsqueeze(0)
    B, dim = states.shape
    if not states.is_contiguous():
        states = states.contiguous()
    a = torch.as_tensor(np.asarray(a_idx, dtype=np.int64) * dim, device=dev)
    b = torch.as_tensor(np.asarray(b_idx, dtype=np.int64) * dim, device=dev)
    n = a.numel()
    out = torch.empty(n, dtype=torch.complex128, device=dev)
    if n:
        check(L.lib().pqs_inner(ctx.handle, dtype_code(states.dtype), ptr(states), dim, ptr(a), ptr(b), n,
                                ptr(out), stream_ptr()))
    _keepalive(a, b)
    return out


def inner(x, y):
    """<x|y> of two state tensors (same length) -> complex."""
    ctx = context()
    dev = x.device
    x = x.reshape(-1).contiguous()
    y = y.reshape(-1).to(dtype=x.dtype).contiguous()
    dim = x.numel()
    # express both as offsets from x's storage
    esz = x.element_size()
    off_b = (y.data_ptr() - x.data_ptr())
    if off_b % esz:
        stacked = torch.stack([x, y])
        return inner_pairs(stacked, [0], [1])[0]
    a = torch.zeros(1, dtype=torch.int64, device=dev)
    b = torch.full((1,), off_b // esz, dtype=torch.int64, device=dev)
    out = torch.empty(1, dtype=torch.complex128, device=dev)
    check(L.lib().pqs_inner(ctx.handle, dtype_code(x.dtype), ptr(x), dim, ptr(a), ptr(b), 1, ptr(out),
                            stream_ptr()))
    _keepalive(a, b, y)
    return out[0]


def mw(states, n_qubits):
    """Reduced 1-qubit density matrices and Meyer-Wallach Q for a batch.
    Returns (rho (B, N, 4) float64 [r00, r11, Re r01, Im r01], Q (B,))."""
    ctx = context()
    if states.dim() == 1:
        states = states.unsqueeze(0)
    states = states.contiguous()
    B = states.shape[0]
    rho = torch.empty((B, n_qubits, 4), dtype=torch.float64, device=states.device)
    q = torch.empty(B, dtype=torch.float64, device=states.device)
    check(L.lib().pqs_mw(ctx.handle, dtype_code(states.dtype), ptr(states), n_qubits, B, ptr(rho), ptr(q),
                         stream_ptr()))
    return rho, q


def gram(a, b):
    """out[i, j] = <a_i|b_j> for (m, dim) and (n, dim) tensors -> complex128 (m, n)."""
    ctx = context()
    a = a.contiguous() if a.dim() == 2 else a.reshape(1, -1).contiguous()
    b = b.contiguous() if b.dim() == 2 else b.reshape(1, -1).contiguous()
    if a.dtype != b.dtype:
        b = b.to(a.dtype)
    m, dim = a.shape
    n = b.shape[0]
    out = torch.empty((m, n), dtype=torch.complex128, device=a.device)
    check(L.lib().pqs_gram(ctx.handle, dtype_code(a.dtype), ptr(a), dim, m, ptr(b), dim, n, dim, ptr(out),
                           stream_ptr()))
    return out


def pair_fidelities(states):
    """|<s_a|s_b>|^2 over combinations(range(S), 2) of the rows of an (S, dim)
    tensor (S >= 2) -> float64 (S (S - 1) / 2,)."""
    ctx = context()
    states = states.contiguous()
    S, dim = states.shape
    out = torch.empty(S * (S - 1) // 2, dtype=torch.float64, device=states.device)
    check(L.lib().pqs_pair_fidelities(ctx.handle, dtype_code(states.dtype), ptr(states), dim, S, dim, ptr(out),
                                      stream_ptr()))
    return out


def qfim(J, psi):
    """F = 4 Re(J J^dag - (J psi^*)(psi J^dag)) -> float64 (P, P)."""
    ctx = context()
    J = J.contiguous()
    P, dim = J.shape
    psi = psi.reshape(-1).to(J.dtype).contiguous()
    F = torch.empty((P, P), dtype=torch.float64, device=J.device)
    if P:
        check(L.lib().pqs_qfim(ctx.handle, dtype_code(J.dtype), ptr(J), P, ptr(psi), dim, ptr(F), stream_ptr()))
    return F


def expect_pauli(states, n_qubits, terms):
    """sum_t c_t <psi|P_t|psi> per row; terms = [(coef, xmask, zmask)] with
    qubit masks (bit q = qubit q).  Returns complex128 (B,)."""
    ctx = context()
    if states.dim() == 1:
        states = states.unsqueeze(0)
    states = states.contiguous()
    B = states.shape[0]
    nt = len(terms)
    xm = (C.c_uint64 * max(1, nt))(*[int(t[1]) for t in terms])
    zm = (C.c_uint64 * max(1, nt))(*[int(t[2]) for t in terms])
    cf = (C.c_double * max(2, 2 * nt))(*[v for t in terms for v in (complex(t[0]).real, complex(t[0]).imag)])
    out = torch.empty(B, dtype=torch.complex128, device=states.device)
    check(L.lib().pqs_expect_pauli(ctx.handle, dtype_code(states.dtype), ptr(states), n_qubits, B, xm, zm, cf, nt,
                                   ptr(out), stream_ptr()))
    return out


def histogram(values, edges):
    """Counts of float64 device values over numpy-style edges -> int64 (nb,)."""
    ctx = context()
    values = values.to(torch.float64).contiguous()
    e = torch.as_tensor(np.asarray(edges, dtype=np.float64), device=values.device)
    nb = e.numel() - 1
    counts = torch.empty(nb, dtype=torch.int64, device=values.device)
    check(L.lib().pqs_histogram(ctx.handle, ptr(values), values.numel(), ptr(e), nb, ptr(counts), stream_ptr()))
    _keepalive(e)
    return counts


def magic_sum(states, n_qubits, alpha):
    """sum_P (<P>^2 / 2^n)^alpha per row -> float64 (B,)."""
    ctx = context()
    if states.dim() == 1:
        states = states.unsqueeze(0)
    states = states.contiguous()
    out = torch.empty(states.shape[0], dtype=torch.float64, device=states.device)
    check(L.lib().pqs_magic(ctx.handle, dtype_code(states.dtype), ptr(states), n_qubits, states.shape[0],
                            float(alpha), ptr(out), stream_ptr()))
    return out


def apply_dense(U, states):
    """out_b = U x_b for a dense dim x dim operator (host or device array,
    complex128) on a (B, dim) or (dim,) state tensor -> new tensor."""
    ctx = context()
    squeeze = states.dim() == 1
    x = states.reshape(1, -1) if squeeze else states
    x = x.contiguous()
    B, dim = x.shape
    u = U if torch.is_tensor(U) else torch.as_tensor(np.ascontiguousarray(U, dtype=np.complex128))
    u = u.to(device=x.device, dtype=torch.complex128).contiguous()
    if u.shape != (dim, dim):
        raise ValueError(f"operator of shape {tuple(u.shape)} on states of dimension {dim}")
    out = torch.empty_like(x)
    check(L.lib().pqs_apply_dense(ctx.handle, dtype_code(x.dtype), ptr(u), dim, ptr(x), dim, B, ptr(out),
                                  stream_ptr()))
    _keepalive(u, x)
    return out.reshape(-1) if squeeze else out


def abs2(z):
    ctx = context()
    z = z.to(torch.complex128).contiguous()
    out = torch.empty(z.shape, dtype=torch.float64, device=z.device)
    check(L.lib().pqs_abs2(ctx.handle, ptr(z), z.numel(), ptr(out), stream_ptr()))
    return out


# Temporaries handed to asynchronous kernels must outlive them: the caching
# allocator may hand their memory to the next tensor as soon as Python drops
# them.  record_stream marks them as used by the current stream.
def _keepalive(*ts):
    s = torch.cuda.current_stream()
    for t in ts:
        if t is not None and torch.is_tensor(t) and t.is_cuda:
            t.record_stream(s)
