"""complex64 tiles run op by op in LDS: lists whose length is at the edges of
a run of 64 ops, every op kind, one wide and several narrow tiles, derivative
ops in and out of a run, against the same list in complex128."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _ops(n, count, rng):
    from pyramaterised_amd import _lib as L
    from pyramaterised_amd.gates import _gen, _op, fsim_gate
    out, slot, tg = [], 0, 0
    u = np.linalg.qr(rng.normal(size=(2, 2)) + 1j * rng.normal(size=(2, 2)))[0]
    while len(out) < count:
        q = int(rng.integers(n))
        q2 = int((q + 1 + rng.integers(max(1, n - 1))) % n)
        kinds = ["RX", "RY", "RZ", "MAT1", "Z"] + (["CX", "CZ", "RXX", "RYY", "RZZ", "FSIM", "MAT2"] if n > 1 else [])
        k = kinds[rng.integers(len(kinds))]
        if k == "MAT1":
            out.append(_op(L.OP_MAT1, q, m=u))
        elif k == "Z":
            out.append(_op(L.OP_MAT1, q, m=np.diag([1.0, 1j])))
        elif k in ("CX", "CZ"):
            out.append(_op(getattr(L, "OP_" + k), q, q2))
        elif k == "MAT2":
            out.append(_op(L.OP_MAT2, q, q2, m=fsim_gate(0.3, 0.9)))
        elif k == "FSIM":
            out.append(_op(L.OP_FSIM, q, q2, slot=slot, slot2=slot + 1))
            slot += 2
        elif k in ("RXX", "RYY", "RZZ"):
            out.append(_op(getattr(L, "OP_" + k), q, q2, slot=slot))
            slot += 1
        else:
            out.append(_op(getattr(L, "OP_" + k), q, slot=slot))
            slot += 1
            if len(out) < count:
                out.append(_gen(tg, "XYZ".index(k[1]) + 1, [q], -0.5j))
                tg += 1
    return out, rng.random(max(1, slot)) * 2 * np.pi, tg


@pytest.mark.parametrize("n,tile,low", [(1, 0, 0), (2, 0, 0), (6, 0, 0), (9, 0, 0), (9, 5, 2), (11, 7, 2)])
@pytest.mark.parametrize("count", [1, 63, 64, 65, 130])
def test_runs_of_ops_match_complex128(n, tile, low, count):
    from pyramaterised_amd import engine as E
    rng = np.random.default_rng(1000 * n + count)
    ops, th, tg = _ops(n, count, rng)
    init = E.Init.product([v / np.linalg.norm(v) for v in rng.normal(size=(n, 2)) + 1j * rng.normal(size=(n, 2))])
    kw = dict(tile_bits=tile, low_bits=low)
    a, b = E.Plan(n, ops, dtype="complex64", **kw), E.Plan(n, ops, dtype="complex128", **kw)
    # every op rounds an amplitude at most 8 times; n for the product state
    tol = 8 * (count + n) * 2.0 ** -24
    tgs = [-1] + sorted({0, tg // 2, tg - 1}) if tg else [-1]
    params = np.tile(th, (len(tgs), 1))
    got, want = E.run(a, params, init, tangents=tgs), E.run(b, params, init, tangents=tgs)
    assert float((got - want).abs().max()) < tol
