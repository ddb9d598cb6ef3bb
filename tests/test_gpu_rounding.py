"""Rounding of complex128 states against an 80-bit evolution, on a circuit
whose gates share their angles, so that the errors of one (cos, sin) add up
over every gate that uses it instead of averaging out.

With u = 2^-53, a rounded number is off by 0.41 u rms (relative).  A rotation
whose cos and sin are off by d_c and d_s changes the state's norm by c^2 d_c +
s^2 d_s and its angle by c s (d_s - d_c): mean squares 3/4 and 1/4 of
(0.41 u)^2.  m gates of one angle act together (m^2), different angles
independently; rounding the product with c and the sum adds (1 + c^2)
(0.41 u)^2 per gate, independently.  A layer of the XXZ ansatz on n qubits has
two angles on n/2 gates each and two on n gates each.  The states of a batch
have independent angles: their rms error is held to that sum (an upper bound,
since a change of angle moves a state by its generator's spread only)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

U = 2.0 ** -53


def _program(n, layers):
    out, k = [], 0
    for _ in range(layers):
        for first in (1, 0):
            prs = [(q, (q + 1) % n) for q in range(first, n, 2)]
            out += [("zz", p, k) for p in prs] + [("yy", p, k + 1) for p in prs] + [("xx", p, k + 1) for p in prs]
            k += 2
    return out, k


def _evolve(n, prog, th):
    """States of every row of th in long double."""
    s = np.zeros((th.shape[0], 1 << n), dtype=np.clongdouble)
    s[:, ((1 << (n // 2)) - 1) << (n - n // 2)] = 1
    half = th.astype(np.longdouble) / 2
    cos, sin = np.cos(half), np.sin(half)
    j = np.arange(1 << n)
    for kind, (a, b), k in prog:
        c, q = cos[:, k, None], sin[:, k, None]
        za, zb = (j >> (n - 1 - a)) & 1, (j >> (n - 1 - b)) & 1
        sign = np.where(za == zb, 1, -1)[None, :].astype(np.longdouble)
        if kind == "zz":
            s = (c - 1j * q * sign) * s
        else:  # X(x)X, and Y(x)Y = -X(x)X on 00, 11
            p = s[:, j ^ (1 << (n - 1 - a)) ^ (1 << (n - 1 - b))]
            s = c * s - 1j * q * (p if kind == "xx" else -sign * p)
    return s


@pytest.mark.parametrize("n,jit,batch", [(8, False, 192), (10, False, 96), (10, True, 96), (12, True, 32)])
def test_shared_angle_rounding(n, jit, batch):
    """Specialised sweeps take the scale from groups of up to ten cosines,
    multiplied in higher precision and corrected to the rounded tangent: an
    angle's error is that of t = fl(sin / cos) alone, c s d_t with three
    roundings in d_t (mean square 3/8 of (0.41 u)^2), each group rounds the
    scale twice, and an amplitude rounds once per gate."""
    import pyramaterised_amd as pyqc
    from pyramaterised_amd import engine as E
    from pyramaterised_amd import templates as T
    layers = 10
    qc = pyqc.PQC(n)
    qc.initial_state = pyqc.tensor([pyqc.basis(2, 1)] * (n // 2) + [pyqc.basis(2, 0)] * (n - n // 2))
    qc.add_layers(T.XXZ_layers(layers, n))
    prog, P = _program(n, layers)
    assert P == qc.n_true_params
    th = np.random.default_rng(n).random((batch, P)) * 2 * np.pi
    plan = E.Plan(n, qc.ops())
    if jit:
        plan.jit()
    got = E.run(plan, th, qc.init()).cpu().numpy().astype(np.clongdouble)
    err = np.sqrt(float(np.mean(np.sum(np.abs(got - _evolve(n, prog, th)) ** 2, axis=1))))
    together = layers * 2 * ((n // 2) ** 2 + n ** 2)
    if jit:
        bound = 3 / 8 * together + (1 + 2 / 10) * len(prog)
    else:
        bound = together + 1.5 * len(prog)
    assert err < 0.41 * U * np.sqrt(bound), err / U
