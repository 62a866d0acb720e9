"""Performance cases: the calls a program makes on one GPU, over their real range.

Families (the `path` of a case):

* `circuit`: a compiled plan run on a state from |0...0> (brickwall, hardware-efficient ansatz),
  with generated pass kernels or the compiled op loop, in FP64 or FP32;
* `qft`: the compiled quantum Fourier transform applied to the state in hand;
* `dense`: a compiled circuit of dense k-qubit unitaries;
* `vqe`: one energy evaluation of a variational loop: plan, run, Pauli sum;
* `energy`: the energy of a prepared state under a transverse-field Ising chain or a MaxCut sum;
* `readout`: shots and a marginal distribution of a prepared state;
* `syndrome`: gates one by one with mid-circuit measurements (a repetition-code cycle);
* `qaoa`: a batch of QAOA MaxCut instances, each an uneven number of qubits;
* `noise`: Monte-Carlo noise trajectories.
"""

from __future__ import annotations

import math

import numpy as np
import torch

from aleph_amd import _lib as L
from aleph_amd import noise as N
from aleph_amd import workloads as W
from aleph_amd.backend import HipSvBackend
from aleph_amd.batch import HipBatch
from aleph_amd.circuit import Circuit, Gate, GateInstance, PauliString

DEV = "cuda"


def listed():
    return [
        # The headline benchmark: a deep random circuit on the largest FP64 state in everyday use.
        {"name": "brickwall_f64_n30", "path": "circuit", "kind": "brickwall", "n": 30, "depth": 20, "precision": 64,
         "jit": True},
        # The same kind of circuit in single precision.
        {"name": "brickwall_f32_n28", "path": "circuit", "kind": "brickwall", "n": 28, "depth": 20, "precision": 32,
         "jit": True},
        # An ansatz run with the library's defaults (no kernel generation) on a mid-size state.
        {"name": "hea_f64_n23_oploop", "path": "circuit", "kind": "hea", "n": 23, "depth": 5, "precision": 64,
         "jit": False},
        # The QFT as a subroutine on a state that the program already has.
        {"name": "qft_f64_n27", "path": "qft", "n": 27, "precision": 64, "jit": True},
        # Dense 5-qubit unitaries (block-encoded or synthesised operators).
        {"name": "dense5_f64_n25", "path": "dense", "n": 25, "k": 5, "gates": 12, "precision": 64},
        # The smallest calls: one step of a variational loop at a textbook size.
        {"name": "vqe_f64_n11", "path": "vqe", "n": 11, "depth": 3, "precision": 64},
        # Energy of a large state: one Pauli sum with diagonal and off-diagonal strings.
        {"name": "ising_energy_f64_n26", "path": "energy", "kind": "ising", "n": 26, "precision": 64},
        # Shots and a register's distribution after a large run.
        {"name": "readout_f64_n27", "path": "readout", "n": 27, "shots": 4096, "marginal": 9, "precision": 64},
        # Error-correction style execution: every gate a call, measurements in between.
        {"name": "syndrome_f64_n19", "path": "syndrome", "n": 19, "precision": 64},
        # A parameter sweep: many instances of 12 to 20 qubits run and scored together.
        {"name": "qaoa_sweep_f32", "path": "qaoa", "count": 160, "n_min": 12, "n_max": 20, "p": 4, "precision": 32,
         "new_angles": False},
        # One step of an optimiser over a few small instances: new angles, run, score.
        {"name": "qaoa_step_f64", "path": "qaoa", "count": 24, "n_min": 10, "n_max": 16, "p": 3, "precision": 64,
         "new_angles": True},
        # Noisy shots of a small device-style circuit.
        {"name": "noise_n12", "path": "noise", "n": 12, "depth": 10, "shots": 20000},
    ]


def draw(rng):
    path = rng.choice(["circuit", "circuit", "circuit", "qft", "dense", "vqe", "energy", "readout", "syndrome",
                       "qaoa", "noise"])
    prec = rng.choice([64, 64, 32])
    if path == "circuit":
        kind = rng.choice(["brickwall", "hea"])
        jit = rng.random() < 0.6
        return {"path": path, "kind": kind, "n": rng.randint(14, 28 if jit else 26),
                "depth": rng.randint(6, 24) if kind == "brickwall" else rng.randint(2, 7), "precision": prec,
                "jit": jit}
    if path == "qft":
        return {"path": path, "n": rng.randint(13, 28), "precision": prec, "jit": rng.random() < 0.6}
    if path == "dense":
        return {"path": path, "n": rng.randint(12, 26), "k": rng.randint(3, 6), "gates": rng.randint(4, 16),
                "precision": prec}
    if path == "vqe":
        return {"path": path, "n": rng.randint(6, 16), "depth": rng.randint(1, 6), "precision": 64}
    if path == "energy":
        return {"path": path, "kind": rng.choice(["ising", "maxcut"]), "n": 2 * rng.randint(5, 13) + rng.randint(0, 1),
                "precision": prec}
    if path == "readout":
        return {"path": path, "n": rng.randint(10, 28), "shots": int(round(2 ** rng.uniform(6, 14))),
                "marginal": rng.randint(2, 10), "precision": prec}
    if path == "syndrome":
        return {"path": path, "n": 2 * rng.randint(4, 11) + 1, "precision": prec}
    if path == "qaoa":
        n_max = 2 * rng.randint(6, 11)
        return {"path": path, "count": int(round(2 ** rng.uniform(4, 8))), "n_min": max(8, n_max - 8),
                "n_max": n_max, "p": rng.randint(1, 5), "precision": rng.choice([32, 32, 64]),
                "new_angles": rng.random() < 0.5}
    return {"path": path, "n": rng.randint(4, 14), "depth": rng.randint(4, 12),
            "shots": int(round(2 ** rng.uniform(10, 14)))}


# ---------------------------------------------------------------- inputs

def _ising(n):
    """H = -sum Z_q Z_{q+1} - 0.7 sum X_q on an open chain."""
    zz = [PauliString.new(-1.0, [(q, "Z"), (q + 1, "Z")]) for q in range(n - 1)]
    return zz + [PauliString.new(-0.7, [(q, "X")]) for q in range(n)]


def _edges(case, seed):
    n = case["n"]
    m = n - (n & 1)
    return W.random_3_regular(m, seed + 17) + ([(0, n - 1)] if n & 1 else [])


def _maxcut(n, edges):
    return [PauliString.identity(0.5 * len(edges))] + [PauliString.new(-0.5, [(u, "Z"), (v, "Z")]) for u, v in edges]


def _terms(case, seed):
    return _ising(case["n"]) if case.get("kind") != "maxcut" else _maxcut(case["n"], _edges(case, seed))


def _circuit(case, seed):
    if case["kind"] == "hea":
        return W.hea(case["n"], case["depth"], seed=seed)
    return W.brickwall(case["n"], case["depth"], seed=seed)


def _random_state(n, seed, precision):
    """A normalised complex Gaussian vector on the GPU, interleaved re/im."""
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    v = torch.randn(2 << n, generator=g, device=DEV, dtype=torch.float64 if precision == 64 else torch.float32)
    return v.mul_(1.0 / float(torch.linalg.vector_norm(v, dtype=torch.float64)))


def _unitaries(case, seed):
    rng = np.random.default_rng(seed)
    d, out = 1 << case["k"], []
    for _ in range(case["gates"]):
        q, r = np.linalg.qr(rng.standard_normal((d, d)) + 1j * rng.standard_normal((d, d)))
        u = q * (np.diag(r) / np.abs(np.diag(r)))
        out.append((u, [int(x) for x in rng.permutation(case["n"])[:case["k"]]]))
    return out


def _cycle(case, seed):
    """A repetition-code cycle: data qubits on even positions are rotated a little, each ancilla between two
    of them takes their parity and is measured.  Items: GateInstance, or (ancilla, uniform)."""
    rng = np.random.default_rng(seed)
    n, out = case["n"], []
    for _ in range(2):
        for q in range(0, n, 2):
            out.append(GateInstance(Gate.Rx(float(rng.uniform(0.2, 0.8))), [q]))
        for a in range(1, n - 1, 2):
            out += [GateInstance(Gate.Cnot(), [a - 1, a]), GateInstance(Gate.Cnot(), [a + 1, a]),
                    (a, float(rng.uniform()))]
    return out


def _qaoa(case, seed):
    return W.qaoa_batch(case["count"], seed=seed, n_min=case["n_min"], n_max=case["n_max"], p=case["p"])


class _DeviceArray:
    """A state's amplitudes as (2^n, 2) reals, for torch.as_tensor (no copy)."""

    def __init__(self, state):
        t = "<f8" if state.precision == 64 else "<f4"
        self.state = state
        self.__cuda_array_interface__ = {"data": (state.device_ptr(), False), "shape": (1 << state.num_qubits, 2),
                                         "typestr": t, "strides": None, "version": 2}


def _view(state):
    return torch.as_tensor(_DeviceArray(state), device=DEV)


def _load(backend, state, amps):
    torch.cuda.synchronize()
    backend._check(L.load().aleph_hip_state_load_device(backend._ctx, state.handle, amps.data_ptr()))


def _reset(s):
    s["backend"]._check(L.load().aleph_hip_state_reset(s["backend"]._ctx, s["state"].handle))


def prepare(case, seed):
    path = case["path"]
    prec = case.get("precision", 64)
    b = HipSvBackend(seed=seed, precision=prec)
    s = {"path": path, "backend": b}
    if path == "noise":
        s["circuit"], s["model"] = W.noisy_brickwall(case["n"], case["depth"], seed=seed)
        s.update(shots=case["shots"], seed=seed)
        return s
    if path == "qaoa":
        graphs, ga, be = _qaoa(case, seed)
        s["batch"] = HipBatch.qaoa(b, graphs, ga, be, precision=prec)
        s["angles"] = (ga, be) if case["new_angles"] else None
        return s
    s["state"] = b.allocate(case["n"])
    if path == "circuit":
        s["plan"] = b.compile(_circuit(case, seed), jit=case["jit"])
    elif path == "qft":
        s["plan"] = b.compile(W.qft(case["n"]), jit=case["jit"])
        _load(b, s["state"], _random_state(case["n"], seed, prec))
    elif path == "dense":
        c = Circuit(case["n"])
        for u, qs in _unitaries(case, seed):
            c.gate(Gate.unitary_kq(u), qs)
        s["plan"] = b.compile(c)
        _load(b, s["state"], _random_state(case["n"], seed, prec))
    elif path == "vqe":
        s["circuit"] = W.hea(case["n"], case["depth"], seed=seed)
        s["terms"] = _ising(case["n"])
    elif path == "energy":
        s["terms"] = _terms(case, seed)
        _load(b, s["state"], _random_state(case["n"], seed, prec))
    elif path == "readout":
        rng = np.random.default_rng(seed)
        s["uniforms"] = rng.uniform(size=case["shots"])
        s["qubits"] = [int(q) for q in rng.permutation(case["n"])[:min(case["marginal"], case["n"])]]
        _load(b, s["state"], _random_state(case["n"], seed, prec))
    else:
        s["cycle"] = _cycle(case, seed)
    s["view"] = _view(s["state"])
    return s


# ---------------------------------------------------------------- one pass

def run(s):
    path, b = s["path"], s["backend"]
    if path == "circuit":
        _reset(s)
        s["plan"].execute(s["state"])
        return s["view"]
    if path in ("qft", "dense"):
        s["plan"].execute(s["state"])
        return s["view"]
    if path == "vqe":
        _reset(s)
        b.run_program(s["state"], s["circuit"])
        return [b.expectation_pauli_sum(s["state"], s["terms"]), s["view"]]
    if path == "energy":
        return b.expectation_pauli_sum(s["state"], s["terms"])
    if path == "readout":
        shots = b.sample(s["state"], len(s["uniforms"]), s["uniforms"])
        return [shots.view(np.int64), b.probabilities(s["state"], s["qubits"])]
    if path == "syndrome":
        _reset(s)
        bits = []
        for item in s["cycle"]:
            if isinstance(item, GateInstance):
                b.apply_gate(s["state"], item)
            else:
                bits.append(int(b.measure_with_uniform(s["state"], *item)[0]))
        return [np.array(bits, dtype=np.int64), s["view"]]
    if path == "qaoa":
        if s["angles"]:
            s["batch"].set_qaoa_angles(*s["angles"])
        s["batch"].run()
        return s["batch"].expect_maxcut()
    return N.outcomes(s["circuit"], s["model"], s["shots"], s["seed"], backend=b).view(np.int64)


# ---------------------------------------------------------------- what a pass cannot do without

def _gate_flops(case):
    """Floating-point operations per amplitude: 14 for a 2x2 (two complex products and a sum), 6 for a phase;
    sign flips and permutations are free, neighbouring one-qubit gates count once."""
    n, d = case["n"], case.get("depth", 1)
    if case["path"] == "qft":
        return 14 * n + 6 * 0.5 * n
    return 14 * n * d


def work(case):
    path, prec = case["path"], case.get("precision", 64)
    if path == "noise":
        gates = case["n"] * case["depth"]
        return {"bytes": 8.0 * case["shots"], "flops": 14.0 * gates * case["shots"] * 2.0 ** case["n"]}
    if path == "qaoa":
        sizes = [n for n, _ in _qaoa(case, 1)[0]]
        amps = float(sum(2.0 ** n for n in sizes))
        flops = sum(2.0 ** n * case["p"] * (14 * n + 6) for n in sizes)
        return {"bytes": amps * (prec // 4), "flops": flops}
    state = 2.0 ** case["n"] * (prec // 4)
    amps = 2.0 ** case["n"]
    if path == "circuit":
        return {"bytes": state, "flops": amps * _gate_flops(case)}
    if path == "vqe":
        return {"bytes": state, "flops": amps * (_gate_flops(case) + 4 * (2 * case["n"] - 1))}
    if path == "qft":
        return {"bytes": 2 * state, "flops": amps * _gate_flops(case)}
    if path == "dense":
        return {"bytes": 2 * state, "flops": amps * case["gates"] * (8.0 * 2 ** case["k"] - 2)}
    if path == "energy":
        terms = 2 * case["n"] - 1 if case["kind"] == "ising" else 1.5 * case["n"]
        return {"bytes": state, "flops": amps * 4 * terms}
    if path == "readout":
        return {"bytes": state, "flops": amps * 5}
    gates = sum(1 for i in _cycle(case, 1) if isinstance(i, GateInstance) and i.gate.name == "Rx")
    meas = 2 * ((case["n"] - 1) // 2)
    return {"bytes": state, "flops": amps * (14 * gates + 5 * meas)}


# ---------------------------------------------------------------- the same in 64 bits, by torch alone

def _u3(t, p, l):
    c, s = math.cos(t / 2), math.sin(t / 2)
    return np.array([[c, -np.exp(1j * l) * s], [np.exp(1j * p) * s, np.exp(1j * (p + l)) * c]])


def _rx(t):
    c, s = math.cos(t / 2), math.sin(t / 2)
    return np.array([[c, -1j * s], [-1j * s, c]])


def _layer(psi, n, mats):
    """mats[q] on every qubit q: blocks of up to 5 of the top qubits at a time, each moved to the bottom."""
    q = n
    while q > 0:
        g = min(5, q)
        m = np.ones((1, 1))
        for j in range(g):
            m = np.kron(m, mats[q - 1 - j])
        m = torch.from_numpy(np.ascontiguousarray(m.astype(np.complex128))).to(DEV)
        psi = (m @ psi.view(1 << g, -1)).t().contiguous().view(-1)
        q -= g
    return psi


def _one(psi, q, m):
    v = psi.view(-1, 2, 1 << q)
    a, b = v[:, 0].clone(), v[:, 1].clone()
    m = [[complex(z) for z in row] for row in m]
    v[:, 0] = m[0][0] * a + m[0][1] * b
    v[:, 1] = m[1][0] * a + m[1][1] * b


def _cx(psi, n, c, t):
    v = psi.view(-1, 2, 1 << (abs(c - t) - 1), 2, 1 << min(c, t))
    x, y = (v[:, 0, :, 1], v[:, 1, :, 1]) if t > c else (v[:, 1, :, 0], v[:, 1, :, 1])
    k = x.clone()
    x.copy_(y)
    y.copy_(k)


def _zero(n):
    psi = torch.zeros(1 << n, dtype=torch.complex128, device=DEV)
    psi[0] = 1
    return psi


def _exact_circuit(case, seed):
    n, psi = case["n"], _zero(case["n"])
    insts = _circuit(case, seed).instructions if case["path"] == "circuit" else W.hea(n, case["depth"], seed=seed).instructions
    mats, pending = [np.eye(2, dtype=complex) for _ in range(n)], False
    for i in insts:
        g = i.gate
        if g.name in ("U3", "Ry", "Rz"):
            p = g.params
            m = (_u3(*p) if g.name == "U3" else _u3(p[0], 0.0, 0.0) if g.name == "Ry"
                 else np.diag([np.exp(-0.5j * p[0]), np.exp(0.5j * p[0])]))
            mats[i.qubits[0]] = m @ mats[i.qubits[0]]
            pending = True
            continue
        if pending:
            psi = _layer(psi, n, mats)
            mats, pending = [np.eye(2, dtype=complex) for _ in range(n)], False
        a, b = i.qubits
        if g.name == "Cz":
            psi.view(-1, 2, 1 << (abs(a - b) - 1), 2, 1 << min(a, b))[:, 1, :, 1].neg_()
        else:
            _cx(psi, n, a, b)
    return _layer(psi, n, mats) if pending else psi


def _reversed_bits(n):
    x = torch.arange(1 << n, device=DEV)
    r = torch.zeros_like(x)
    for q in range(n):
        r |= ((x >> q) & 1) << (n - 1 - q)
    return r


def _exact_qft(case, seed):
    n = case["n"]
    psi = torch.view_as_complex(_random_state(n, seed, case["precision"]).double().view(-1, 2))
    h = math.sqrt(0.5)
    for j in range(n):
        _one(psi, j, [[h, h], [h, -h]])
        y = torch.arange(1 << (n - 1 - j), device=DEV)
        ang = torch.zeros(y.shape, dtype=torch.float64, device=DEV)
        for i in range(n - 1 - j):
            ang += ((y >> i) & 1).double() * (2.0 * math.pi / 2.0 ** (i + 2))
        psi.view(-1, 2, 1 << j)[:, 1].mul_(torch.polar(torch.ones_like(ang), ang)[:, None])
    return psi[_reversed_bits(n)]


def _exact_dense(case, seed):
    n, k = case["n"], case["k"]
    psi = torch.view_as_complex(_random_state(n, seed, case["precision"]).double().view(-1, 2))
    for u, qs in _unitaries(case, seed):
        rest = [q for q in range(n) if q not in qs]
        y = torch.arange(1 << (n - k), device=DEV)
        base = torch.zeros_like(y)
        for i, q in enumerate(rest):
            base |= ((y >> i) & 1) << q
        off = torch.tensor([sum(((r >> (k - 1 - i)) & 1) << q for i, q in enumerate(qs)) for r in range(1 << k)],
                           device=DEV)
        idx = off[:, None] | base[None, :]
        psi[idx] = torch.from_numpy(np.ascontiguousarray(u)).to(DEV) @ psi[idx]
    return psi


def _exact_terms(psi, terms):
    """sum of coefficient * <psi|P|psi> for strings of one X or of Z's."""
    p = psi.real.square() + psi.imag.square()
    total = 0.0
    for t in terms:
        if not t.terms:
            total += t.coefficient * float(p.sum())
        elif t.terms[0][1] == "X":
            v = psi.view(-1, 2, 1 << t.terms[0][0])
            a, b = v[:, 0], v[:, 1]
            total += t.coefficient * 2.0 * float((a.real * b.real + a.imag * b.imag).sum())
        else:
            lo, hi = (q for q, _ in t.terms)
            m = p.view(-1, 2, 1 << (hi - lo - 1), 2, 1 << lo).sum(dim=(0, 2, 4)).cpu()
            total += t.coefficient * float(m[0, 0] + m[1, 1] - m[0, 1] - m[1, 0])
    return total


def _exact_qaoa(case, seed):
    out = []
    for (n, edges), ga, be in zip(*_qaoa(case, seed)):
        x = torch.arange(1 << n, device=DEV)
        cut = torch.zeros(1 << n, dtype=torch.float64, device=DEV)
        for u, v in edges:
            cut += (((x >> u) ^ (x >> v)) & 1).double()
        psi = torch.full((1 << n,), 2.0 ** (-n / 2), dtype=torch.complex128, device=DEV)
        for g, b in zip(ga, be):
            ang = (-0.5 * float(g)) * (len(edges) - 2.0 * cut)
            psi = _layer(psi * torch.polar(torch.ones_like(ang), ang), n, [_rx(float(b))] * n)
        out.append(float(((psi.real.square() + psi.imag.square()) * cut).sum()))
    return np.array(out)


def _exact_syndrome(case, seed):
    n, psi, bits = case["n"], _zero(case["n"]), []
    for item in _cycle(case, seed):
        if isinstance(item, GateInstance) and item.gate.name == "Rx":
            _one(psi, item.qubits[0], _rx(item.gate.params[0]))
        elif isinstance(item, GateInstance):
            _cx(psi, n, *item.qubits)
        else:
            v = psi.view(-1, 2, 1 << item[0])
            p1 = float(v[:, 1].abs().square().sum())
            bit = int(p1 >= 1e-300 and item[1] < p1)
            v[:, 1 - bit] = 0
            v[:, bit] *= 1.0 / math.sqrt(p1 if bit else 1.0 - p1)
            bits.append(bit)
    return [None, torch.view_as_real(psi)]


def exact(case, seed):
    path = case["path"]
    if path == "circuit":
        return torch.view_as_real(_exact_circuit(case, seed))
    if path == "qft":
        return torch.view_as_real(_exact_qft(case, seed))
    if path == "dense":
        return torch.view_as_real(_exact_dense(case, seed))
    if path == "vqe":
        psi = _exact_circuit(case, seed)
        return [_exact_terms(psi, _ising(case["n"])), torch.view_as_real(psi)]
    if path in ("energy", "readout"):
        psi = torch.view_as_complex(_random_state(case["n"], seed, case["precision"]).double().view(-1, 2))
        if path == "energy":
            return _exact_terms(psi, _terms(case, seed))
        p = psi.real.square() + psi.imag.square()
        rng = np.random.default_rng(seed)
        rng.uniform(size=case["shots"])
        x = torch.arange(1 << case["n"], device=DEV)
        sel = torch.zeros_like(x)
        qubits = [int(q) for q in rng.permutation(case["n"])[:min(case["marginal"], case["n"])]]
        for j, q in enumerate(qubits):
            sel |= ((x >> q) & 1) << j
        return [None, torch.stack([p[sel == k].sum() for k in range(1 << len(qubits))])]
    if path == "qaoa":
        return _exact_qaoa(case, seed)
    if path == "syndrome":
        return _exact_syndrome(case, seed)
    return None
