"""Derivatives carried by their rotation's angle (a generator right after the
rotation it differentiates, complex128) against the generator op itself: the
same op list with every generator written as two equal terms, which stays a
Pauli sum.  All six rotations, scales and offsets, one parameter on several
rotations, lists that only look like a derivative, angles at 0 and pi."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

ROT = ["RX", "RY", "RZ", "RXX", "RYY", "RZZ"]


def _lists(n, depth, rng):
    """(ops with plain generators, the same with split ones, params)"""
    from pyramaterised_amd import _lib as L
    from pyramaterised_amd.gates import _gen, _op
    one, two, slot = [], [], 0
    shared = None
    for d in range(depth):
        for q in range(n):
            name = ROT[rng.integers(6)]
            q2 = int((q + 1 + rng.integers(n - 1)) % n)
            qs = [q, q2] if len(name) == 3 else [q]
            scale, offset = [(1.0, 0.0), (-1.0, 0.0), (1.0, 0.4), (0.7, -1.1)][rng.integers(4)]
            pauli = "XYZ".index(name[-1]) + 1
            use = slot
            if shared is not None and rng.random() < 0.1:
                use = shared  # one parameter on several rotations
            rot = _op(getattr(L, "OP_" + name), *qs, slot=use, scale=scale, offset=offset)
            coef = -0.5j * scale
            gq, gp = (qs[::-1] if rng.random() < 0.5 else qs), pauli
            odd = rng.integers(8)
            if odd == 0:
                coef *= 1.5 + 0.5j  # not the rotation's derivative
            elif odd == 1:
                gp = pauli % 3 + 1
            elif odd == 2 and len(qs) == 2:
                gq = [qs[0]]
            one += [rot, _gen(use, gp, gq, coef)]
            two += [rot, _gen(use, gp, gq, 0.5 * coef), _gen(use, gp, gq, 0.5 * coef)]
            if use == slot:
                shared = slot if rng.random() < 0.3 else shared
                slot += 1
        for q in range(d % 2, n - 1, 2):
            cx = _op(L.OP_CX, q, q + 1)
            one.append(cx)
            two.append(cx)
    th = rng.random(slot) * 2 * np.pi
    th[::5] = 0.0
    th[1::7] = np.pi
    return one, two, th


@pytest.mark.parametrize("n,depth,tile,low,rolling", [
    (3, 4, 0, 0, False), (8, 3, 0, 0, False), (9, 2, 6, 2, False), (11, 3, 10, 3, False), (12, 3, 12, 3, False),
    (13, 2, 10, 3, True)])
def test_turned_rotations_match_generators(n, depth, tile, low, rolling):
    from pyramaterised_amd import _lib as L
    from pyramaterised_amd import engine as E
    rng = np.random.default_rng(100 + n)
    one, two, th = _lists(n, depth, rng)
    flags = L.PQS_PLAN_ROLLING if rolling else 0
    kw = dict(dtype="complex128", tile_bits=tile, low_bits=low, flags=flags)
    a, b = E.Plan(n, one, **kw), E.Plan(n, two, **kw)
    assert a.n_exec < b.n_exec  # rotations and generators are one op each
    assert sorted(i for _, idx in a.sweeps() for i in idx) == list(range(len(one)))
    vec = rng.normal(size=1 << n) + 1j * rng.normal(size=1 << n)
    vec /= np.linalg.norm(vec)
    # each op rounds every amplitude at most 8 times on either side
    tol = 2 * 8 * len(two) * 2.0 ** -53
    for jit in (False, True):
        if jit and n >= 10:
            a.jit()
        for init in (E.Init.zero(), E.Init.from_vector(vec)):
            pa, ja = E.jacobian(a, th, init)
            pb, jb = E.jacobian(b, th, init)
            assert float((pa - pb).abs().max()) < tol and float((ja - jb).abs().max()) < tol, (jit, init.kind)
            # the same rows as tangent instances of a batch, with plain ones between
            tg = [-1, 0, len(th) - 1, -1, len(th) // 2]
            rows = E.run(a, np.tile(th, (5, 1)), init, tangents=tg)
            for r, t in zip(rows, tg):
                want = pa if t < 0 else ja[t]
                assert float((r - want).abs().max()) < tol, (jit, init.kind, t)


def test_complex64_plans_keep_their_generators():
    from pyramaterised_amd import engine as E
    one, two, _ = _lists(10, 1, np.random.default_rng(3))
    a, b = E.Plan(10, one, dtype="complex64"), E.Plan(10, two, dtype="complex64")
    assert a.n_exec == b.n_exec
