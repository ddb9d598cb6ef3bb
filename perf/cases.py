"""Timed workloads of the engine, through its public entry points.

Every case is one call (or the short sequence of calls) that a program using
the package makes over and over: a state at new angles, a batch of sample
states, state pairs for expressibility, the QFIM, an energy gradient, and the
reductions over states that are already on the GPU.  Sizes follow the
benchmark's workloads (16-qubit HEA with 20 layers, 28-qubit brickwork,
12-qubit TFIM, 20-qubit gradients, 2000-state Gram), the circuit templates at
the widths that the tests use (4-12 qubits), and the serving mix (6-20 qubits,
depth 2-40).

``exact`` restates each result with plain torch operations in complex128.
"""
import functools
import math

import numpy as np
import torch

import pyramaterised_amd as pyqc
from pyramaterised_amd import templates as T
from pyramaterised_amd.magic import renyi_entropy_batch


def listed():
    return [
        # one evaluation of a small circuit in an optimisation loop: launches
        # and host work are all there is
        {"name": "state_4q", "kind": "state", "circuit": "hea", "n": 4, "layers": 3, "dtype": "complex128"},
        # the largest single state of the benchmark, in single precision
        {"name": "state_28q_c64", "kind": "state", "circuit": "brickwork", "n": 28, "layers": 30,
         "dtype": "complex64"},
        # sample states of a small ansatz (expressibility, entanglement and
        # magic all start from such a batch)
        {"name": "sample_8q", "kind": "sample", "circuit": "hea", "n": 8, "layers": 10, "batch": 2000,
         "dtype": "complex128"},
        # sample states of a Hamiltonian-variational ansatz (XX, YY and ZZ rotations)
        {"name": "sample_xxz_12q", "kind": "sample", "circuit": "xxz", "n": 12, "layers": 10, "batch": 1000,
         "dtype": "complex128"},
        # the benchmark's headline step: 5000 pairs of 16-qubit states
        {"name": "pairs_16q", "kind": "pairs", "circuit": "hea", "n": 16, "layers": 20, "batch": 10000,
         "dtype": "complex128"},
        # the QFIM at a width where whole rank studies are run
        {"name": "qfim_8q", "kind": "qfim", "circuit": "hea", "n": 8, "layers": 10, "dtype": "complex128"},
        # the benchmark's QFIM of the 12-qubit TFIM ansatz (shared parameters)
        {"name": "qfim_tfim_12q", "kind": "qfim", "circuit": "tfim", "n": 12, "layers": 10, "dtype": "complex128"},
        # the benchmark's QFIM of the 16-qubit HEA (640 parameters)
        {"name": "qfim_16q", "kind": "qfim", "circuit": "hea", "n": 16, "layers": 20, "dtype": "complex128"},
        # the benchmark's energy gradient: 20 qubits, 1600 parameters, one training step
        {"name": "gradient_20q", "kind": "gradient", "circuit": "hea", "n": 20, "layers": 40, "dtype": "complex128"},
        # Meyer-Wallach entanglement of a batch of sample states
        {"name": "entangle_16q", "kind": "entangle", "n": 16, "batch": 1000, "dtype": "complex128"},
        # stabiliser entropy of a batch of sample states
        {"name": "magic_10q", "kind": "magic", "n": 10, "batch": 200, "alpha": 2.0, "dtype": "complex128"},
        # fidelities of all pairs of sample states
        {"name": "allpairs_12q", "kind": "allpairs", "n": 12, "batch": 1000, "dtype": "complex128"},
    ]


def draw(rng):
    def between(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["state", "sample", "sample", "pairs", "qfim", "qfim", "gradient", "entangle", "magic",
                       "allpairs"])
    c = {"kind": kind, "dtype": rng.choice(["complex128", "complex128", "complex64"])}
    if kind == "state":
        c.update(circuit=rng.choice(["hea", "brickwork", "xxz", "fsim"]), n=rng.randint(3, 26),
                 layers=between(2, 30))
    elif kind == "sample":
        n = rng.randint(4, 14)
        layers = between(2, 20)
        c.update(circuit=rng.choice(["hea", "tfim", "xxz", "fsim"]), n=n, layers=layers,
                 batch=between(16, max(17, min(10000, (1 << 25) >> n))))
    elif kind == "pairs":
        n = rng.randint(5, 16)
        c.update(circuit=rng.choice(["hea", "brickwork"]), n=n, layers=between(2, 20),
                 batch=2 * between(16, min(5000, (1 << 28) >> n)))
    elif kind == "qfim":
        n = rng.randint(4, 16)
        c.update(circuit=rng.choice(["hea", "tfim", "xxz"]), n=n, layers=between(2, 20))
    elif kind == "gradient":
        c.update(circuit=rng.choice(["hea", "brickwork", "tfim"]), n=rng.randint(4, 20), layers=between(2, 40))
    elif kind == "entangle":
        n = rng.randint(4, 20)
        c.update(n=n, batch=between(1, max(2, min(10000, (1 << 26) >> n))))
    elif kind == "magic":
        n = rng.randint(3, 12)
        c.update(n=n, batch=between(1, max(2, min(5000, (1 << 27) >> (2 * n)))),
                 alpha=rng.choice([2.0, 2.0, 0.5]))
    else:
        n = rng.randint(4, 16)
        c.update(n=n, batch=between(10, max(11, min(2000, (1 << 27) >> n))))
    if c.get("circuit") == "xxz":  # the template couples pairs: an even width
        c["n"] += c["n"] % 2
    return c


# ------------------------------------------------------------------ the calls

def _layers(c):
    n, p = c["n"], c["layers"]
    return {"hea": T.clifford_HE_layers, "brickwork": T.ry_cz_brickwork_layers, "tfim": T.tfim_open_layers,
            "xxz": T.XXZ_layers, "fsim": T.fSim_circuit_layers}[c["circuit"]](p, n)


@functools.lru_cache(maxsize=None)
def _circuit(circuit, n, layers, dtype):
    """The circuit that a program builds once and evaluates at many angles."""
    c = {"circuit": circuit, "n": n, "layers": layers}
    qc = pyqc.PQC(n, dtype=dtype)
    if circuit == "tfim":
        qc.set_initial_state(T.plus_state())
    elif circuit in ("xxz", "fsim"):
        qc.initial_state = pyqc.tensor([pyqc.basis(2, 1)] * (n // 2) + [pyqc.basis(2, 0)] * (n - n // 2))
    qc.add_layers(_layers(c))
    return qc


def _qc(c):
    return _circuit(c["circuit"], c["n"], c["layers"], c["dtype"])


def _angles(c, seed):
    P = _slots(_program(c))
    shape = (c["batch"], P) if "batch" in c else (P,)
    return np.random.default_rng(seed).random(shape) * 2 * np.pi


def _states(c, seed):
    """Random normalised states (what deep random circuits give)."""
    g = torch.Generator(device="cuda").manual_seed(int(seed))
    s = torch.randn((c["batch"], 1 << c["n"], 2), generator=g, device="cuda", dtype=torch.float64)
    s = torch.view_as_complex(s)
    s /= torch.linalg.vector_norm(s, dim=1, keepdim=True)
    return s.to(torch.complex64) if c["dtype"] == "complex64" else s


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("entangle", "magic", "allpairs"):
        return {"case": case, "states": _states(case, seed), "qc": pyqc.PQC(case["n"], dtype=case["dtype"])}
    ang = _angles(case, seed)
    if kind == "pairs":  # the benchmark's parameters are resident on the GPU
        ang = torch.as_tensor(ang, device="cuda")
    elif kind in ("state", "qfim", "gradient"):
        ang = ang.tolist()
    return {"case": case, "qc": _qc(case), "angles": ang}


def run(state):
    case, qc = state["case"], state["qc"]
    kind = case["kind"]
    if kind == "state":
        return qc.run(state["angles"]).t
    if kind == "sample":
        return qc.run_batch(state["angles"])
    if kind == "pairs":
        return list(qc.run_batch_pairs(state["angles"]))
    m = pyqc.measure.Measurements(qc)
    if kind == "qfim":
        psi = qc.update_state(state["angles"])
        return [psi.t, m.get_QFI()]
    if kind == "gradient":
        g = m.get_gradient_vector(state["angles"])
        return [qc.state.t, np.array(g)]
    if kind == "entangle":
        return m.entanglement_batch(state["states"])
    if kind == "magic":
        return renyi_entropy_batch(state["states"], case["n"], case["alpha"])
    return m.fidelities_all_pairs(state["states"])


# ----------------------------------------------------------- what it has to do

def _program(c):
    """The circuit as [(gate, qubits, slots)], in the order of application."""
    n, out, k = c["n"], [], 0
    for layer in range(c["layers"]):
        if c["circuit"] == "hea":
            out += [("ry", (q,), (k + q,)) for q in range(n)] + [("rz", (q,), (k + n + q,)) for q in range(n)]
            out += [("cx", (q, q + 1), ()) for q in range(0, n - 1, 2)]
            out += [("cx", (q, q + 1), ()) for q in range(1, n - 1, 2)]
            k += 2 * n
        elif c["circuit"] == "brickwork":
            out += [("ry", (q,), (k + q,)) for q in range(n)]
            out += [("cz", (q, q + 1), ()) for q in range(layer % 2, n - 1, 2)]
            k += n
        elif c["circuit"] == "tfim":
            out += [("rzz", (q, q + 1), (k,)) for q in range(n - 1)] + [("rx", (q,), (k + 1,)) for q in range(n)]
            k += 2
        elif c["circuit"] == "xxz":
            for first in (1, 0):
                prs = [(q, (q + 1) % n) for q in range(first, n, 2)]
                out += [("rzz", p, (k,)) for p in prs]
                out += [("ryy", p, (k + 1,)) for p in prs] + [("rxx", p, (k + 1,)) for p in prs]
                k += 2
        else:  # fsim: rotations and fSim on alternating pairs
            out += [("ry", (q,), (k + q,)) for q in range(n)]
            k += n
            if n % 2 == 0:
                prs, left = [(q, (q + 1) % n) for q in range(layer % 2, n, 2)], None
            else:
                left = layer % n
                idx = [q for q in range(n) if q != left]
                prs = []
                if left % 2 == 1:
                    prs.append((idx.pop(0), idx.pop(-1)))
                prs += list(zip(idx[::2], idx[1::2]))
            for p in prs:
                out.append(("fsim", p, (k, k + 1)))
                k += 2
            if left is not None:
                out.append(("ry", (left,), (k,)))
                k += 1
    return out


def _slots(prog):
    return 1 + max(s for _, _, sl in prog for s in sl)


_FLOPS = {"ry": 6, "rx": 6, "rz": 6, "rzz": 6, "rxx": 6, "ryy": 6, "fsim": 14, "cx": 0, "cz": 0}


def work(case):
    """Inputs read once, outputs written once; rotations at 6 flops per
    amplitude, Gram products over the upper triangle."""
    n, kind = case["n"], case["kind"]
    dim, amp = 1 << n, 8 if case["dtype"] == "complex64" else 16
    if kind in ("entangle", "magic", "allpairs"):
        B = case["batch"]
        rd = B * dim * amp
        if kind == "entangle":  # per qubit half the pairs of a complex product, and the norm
            return {"bytes": rd + 8 * B, "flops": B * dim * (4 * n + 4)}
        if kind == "magic":  # per X part a product and a real Walsh-Hadamard transform
            return {"bytes": rd + 8 * B, "flops": B * dim * dim * (7 + n + 3)}
        return {"bytes": rd + 4 * B * (B - 1), "flops": 4 * B * (B - 1) * dim}
    prog = _program(case)
    P = _slots(prog)
    gate = [_FLOPS[g] for g, _, _ in prog]
    evolve = sum(gate) * dim
    if kind in ("state", "sample", "pairs"):
        B = case.get("batch", 1)
        return {"bytes": B * (8 * P + dim * amp), "flops": B * evolve + (4 * B * dim if kind == "pairs" else 0)}
    if kind == "gradient":  # the state, then the state and its partner backwards
        return {"bytes": 16 * P + dim * amp, "flops": 3 * evolve + 8 * P * dim // 2}
    # every derivative state is carried from its gate to the end; then their
    # Gram, upper triangle
    first, after = {}, [0]
    for f in reversed(gate):
        after.append(after[-1] + f)
    after.reverse()
    for i, (_, _, sl) in enumerate(prog):
        for s in sl:
            first.setdefault(s, after[i + 1])
    return {"bytes": 8 * P + dim * amp + 8 * P * P,
            "flops": (sum(gate) + sum(first.values())) * dim + 2 * P * (P + 1) * dim}


# ------------------------------------------------- the results in plain torch

def _rows(s, n, qs):
    """Views of s (B, 2^n): the amplitudes with each setting of the qubits
    (first one most significant)."""
    a = sorted(qs)
    if len(a) == 1:
        v = s.view(-1, 1 << a[0], 2, 1 << (n - 1 - a[0]))
        return [v[:, :, 0], v[:, :, 1]]
    v = s.view(-1, 1 << a[0], 2, 1 << (a[1] - a[0] - 1), 2, 1 << (n - 1 - a[1]))
    flip = qs[0] > qs[1]
    return [v[:, :, y if flip else x, :, x if flip else y] for x in (0, 1) for y in (0, 1)]


def _apply(s, n, gate, qs, th, inverse=False):
    """The gate on every row of s, in place; th: per slot a number or one
    value per row."""
    r = _rows(s, n, qs)
    if gate in ("cx", "cz"):
        if gate == "cz":
            r[3].neg_()
        else:
            t = r[2].clone()
            r[2].copy_(r[3])
            r[3].copy_(t)
        return
    th = [torch.as_tensor(t, dtype=torch.float64, device=s.device) for t in th]
    sg = -1.0 if inverse else 1.0
    wide = [t.reshape([-1] + [1] * (r[0].dim() - 1)) if t.dim() else t for t in th]
    if gate == "fsim":
        c, q = torch.cos(wide[0]), -1j * sg * torch.sin(wide[0])
        x, y = c * r[1] + q * r[2], q * r[1] + c * r[2]
        r[1].copy_(x)
        r[2].copy_(y)
        r[3].mul_(torch.exp(-1j * sg * wide[1]))
        return
    c, q = torch.cos(wide[0] / 2), sg * torch.sin(wide[0] / 2)
    if gate in ("rz", "rzz"):
        lo, hi = c - 1j * q, c + 1j * q
        for i, v in enumerate(r):
            v.mul_(hi if bin(i).count("1") % 2 else lo)
        return
    for a, b, f in {"ry": [(0, 1, -1)], "rx": [(0, 1, -1j)], "rxx": [(0, 3, -1j), (1, 2, -1j)],
                    "ryy": [(0, 3, 1j), (1, 2, -1j)]}[gate]:
        g = 1 if gate == "ry" else f
        x, y = c * r[a] + (f * q) * r[b], c * r[b] + (g * q) * r[a]
        r[a].copy_(x)
        r[b].copy_(y)


def _generator(s, n, gate, qs):
    """-i/2 P s for the rotation's Pauli string P."""
    out = torch.empty_like(s)
    r, o = _rows(s, n, qs), _rows(out, n, qs)
    h = -0.5j
    src = {"rx": [(1, h), (0, h)], "ry": [(1, -1j * h), (0, 1j * h)], "rz": [(0, h), (1, -h)],
           "rzz": [(0, h), (1, -h), (2, -h), (3, h)], "rxx": [(3, h), (2, h), (1, h), (0, h)],
           "ryy": [(3, -h), (2, h), (1, h), (0, -h)]}[gate]
    for dst, (i, f) in zip(o, src):
        torch.mul(r[i], f, out=dst)
    return out


def _start(c, B):
    n = c["n"]
    s = torch.zeros((B, 1 << n), dtype=torch.complex128, device="cuda")
    if c["circuit"] == "tfim":
        s.fill_(2.0 ** (-n / 2))
    else:
        s[:, ((1 << (n // 2)) - 1) << (n - n // 2) if c["circuit"] in ("xxz", "fsim") else 0] = 1.0
    return s


def _evolve(c, ang):
    """States (B, 2^n) for angles (B, P)."""
    s = _start(c, ang.shape[0])
    for gate, qs, sl in _program(c):
        _apply(s, c["n"], gate, qs, [ang[:, k] for k in sl])
    return s


def exact(case, seed):
    kind, n = case["kind"], case["n"]
    if kind == "entangle":
        out = []
        for s in _states(case, seed).split(max(1, (1 << 26) >> n)):
            s = s.to(torch.complex128)
            pur = 0.0
            for q in range(n):
                a, b = _rows(s, n, (q,))
                r0, r1 = (v.abs().square().sum(dim=(1, 2)) for v in (a, b))
                pur = pur + r0 ** 2 + r1 ** 2 + 2 * (a * b.conj()).sum(dim=(1, 2)).abs() ** 2
            out.append(2 * (1 - pur / n))
        return torch.cat(out)
    if kind == "magic":
        s, d = _states(case, seed).to(torch.complex128), 1 << n
        j = torch.arange(d, device="cuda")
        out = []
        for row in s:
            f = row.conj()[None, :] * row[j[None, :] ^ j[:, None]]
            for b in range(n):
                v = f.view(d, -1, 2, 1 << b)
                f = torch.stack([v[:, :, 0] + v[:, :, 1], v[:, :, 0] - v[:, :, 1]], dim=2)
            out.append(((f.abs() ** 2 / d) ** case["alpha"]).sum())
        tot = torch.stack(out).cpu().numpy()
        return np.log(tot) / (1 - case["alpha"]) - n * np.log(2)
    if kind == "allpairs":
        s = _states(case, seed).to(torch.complex128)
        a, b = np.triu_indices(case["batch"], k=1)
        g = s.conj() @ s.t().contiguous()
        return g[torch.as_tensor(a, device="cuda"), torch.as_tensor(b, device="cuda")].abs() ** 2
    ang = torch.as_tensor(_angles(case, seed), device="cuda")
    if kind == "state":
        return _evolve(case, ang[None])[0]
    if kind in ("sample", "pairs"):
        s = torch.cat([_evolve(case, a) for a in ang.split(max(1, (1 << 26) >> n))])
        return s if kind == "sample" else [s, (s[0::2].conj() * s[1::2]).sum(dim=1)]
    prog, th = _program(case), ang.tolist()
    s = _start(case, 1)
    if kind == "qfim":
        J = torch.zeros((len(th), 1 << n), dtype=torch.complex128, device="cuda")
        for gate, qs, sl in prog:
            _apply(s, n, gate, qs, [th[k] for k in sl])
            _apply(J, n, gate, qs, [th[k] for k in sl])
            if sl:
                J[sl[0]] += _generator(s, n, gate, qs)[0]
        ov = J.conj() @ s[0]
        return [s[0], 4 * ((J.conj() @ J.t().contiguous()) - ov[:, None] * ov.conj()[None, :]).real]
    for gate, qs, sl in prog:
        _apply(s, n, gate, qs, [th[k] for k in sl])
    psi, lam = s.clone(), s.clone()
    for i in (1, 2):
        _rows(lam, n, (0, 1))[i].neg_()
    grad = torch.zeros(len(th), dtype=torch.float64, device="cuda")
    for gate, qs, sl in reversed(prog):
        if sl:
            grad[sl[0]] += 2 * torch.vdot(lam[0], _generator(psi, n, gate, qs)[0]).real
        for v in (psi, lam):
            _apply(v, n, gate, qs, [th[k] for k in sl], inverse=True)
    return [s[0], grad]
