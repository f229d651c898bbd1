"""Performance cases of the state-vector engine.

Each case is one piece of work a user's program has the engine do through the
public Python API, from a 3-qubit teleportation to 32-qubit registers: the
random-circuit, Grover and ansatz workloads of ``quaru_amd.circuits`` and
``bench.py``, the textbook algorithms of the examples (teleportation, Shor's
period finding, the quantum Fourier transform), dense multi-qubit blocks and
the readouts.  ``listed()`` names the fixed cases, ``draw(rng)`` makes further
ones of the same ranges; ``prepare`` makes what the program holds before the
call, ``run`` is one pass, ``work`` what a pass cannot do without and
``exact`` its result in 64-bit arithmetic from plain torch and numpy.

``circuit`` in a case is the seed of what a program keeps from run to run (the
wiring of a random circuit); the seed of ``prepare`` makes the values (gate
matrices, angles, uniforms, input states).  States of 22 and more qubits run
sweep kernels compiled at run time for the circuit's wiring, so ``prepare``
runs such a circuit once and waits for them, as ``bench.py`` does.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from quaru_amd import Register, _lib, circuits
from quaru_amd import operation as ops
from quaru_amd.adjoint import Expectation, ParamCircuit
from quaru_amd.operation import Operation, QuantumCircuit

READOUT = 1 << 16  # amplitudes read from a state too large to copy whole
WHOLE = 20         # qubits up to which a program reads the whole state
JIT_FROM = 22      # index bits from which sweeps run specialised kernels


def listed():
    return [
        # teleportation of one qubit: the smallest program, measurements and
        # conditional corrections kept on the device
        dict(name="teleport_3q", kind="teleport", hops=1, dtype="c128"),
        # the 12-qubit, 20-layer random circuit, then every qubit measured in
        # turn: many small gates on a state that fits one compute unit
        dict(name="circuit_12q_c128", kind="circuit", n=12, layers=20, triples=0, dtype="c128",
             circuit=1, measure="each"),
        # the 26-qubit circuit of the same shape with a full readout: 1 GiB
        dict(name="circuit_26q_c128", kind="circuit", n=26, layers=20, triples=0, dtype="c128",
             circuit=2, measure="all"),
        # the benchmark's 30-qubit circuit with Toffoli and CCZ gates, and
        # amplitudes of given bit strings: 16 GiB, the largest state in FP64
        dict(name="circuit_30q_c128", kind="circuit", n=30, layers=20, triples=8, dtype="c128",
             circuit=3, measure="none"),
        dict(name="circuit_30q_c64", kind="circuit", n=30, layers=20, triples=8, dtype="c64",
             circuit=3, measure="none"),
        # a Fourier transform of a state that the program loads and reads
        # back: controlled phases, an ordinary size
        dict(name="qft_20q_c64", kind="qft", n=20, dtype="c64"),
        # Shor's period finding as the example writes it, N = 21 on 5 bits:
        # dense Hadamard and Fourier matrices on 10 qubits, controlled modular
        # multiplications
        dict(name="shor_15q_c128", kind="shor", bits=5, dtype="c128"),
        # dense 5-qubit blocks on any qubits: circuits that a program fused
        # itself, an odd register size
        dict(name="blocks_27q_c128", kind="blocks", n=27, k=5, count=8, dtype="c128", circuit=4),
        # Grover iterations with Hadamard layers as 5-qubit blocks at the
        # largest size of the benchmark: 32 GiB
        dict(name="grover_32q_c64", kind="grover", n=32, iterations=4, fused=True, dtype="c64"),
        # readouts of a state at rest: shots, amplitudes of bit strings,
        # norm and overlap with another state
        dict(name="readout_26q_c128", kind="readout", n=26, shots=1000, dtype="c128"),
        # energies and gradients of the benchmark's ansatz, 400 parameters in
        # 64 sets
        dict(name="adjoint_20q_b64_c128", kind="adjoint", n=20, layers=10, batch=64,
             checkpoint=2, dtype="c128"),
        # a smaller ansatz in a batch that is no power of two, as an
        # optimiser's population
        dict(name="adjoint_13q_b20_c64", kind="adjoint", n=13, layers=6, batch=20, checkpoint=0,
             dtype="c64"),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    dtype = rng.choice(["c128", "c64"])
    kind = rng.choice(["teleport", "circuit", "circuit", "qft", "shor", "blocks", "grover",
                       "readout", "adjoint", "adjoint"])
    if kind == "teleport":
        return dict(kind=kind, hops=rng.randint(2, 7), dtype=dtype)
    if kind == "circuit":
        n = rng.randint(2, 30)
        return dict(kind=kind, n=n, layers=_log_int(rng, 1, 20),
                    triples=rng.choice([0, 3, 8]) if n >= 3 else 0, dtype=dtype,
                    circuit=rng.randrange(1 << 20), measure=rng.choice(["none", "each", "all"]))
    if kind == "qft":
        return dict(kind=kind, n=rng.randint(3, 22), dtype=dtype)
    if kind == "shor":
        return dict(kind=kind, bits=rng.randint(3, 5), dtype=dtype)
    if kind == "blocks":
        n, k = rng.randint(10, 28), rng.randint(2, 6)
        most = 1 << max(0, 38 - n - k)  # the listed case's operations
        return dict(kind=kind, n=n, k=k, count=min(most, _log_int(rng, 1, 16)), dtype=dtype,
                    circuit=rng.randrange(1 << 20))
    if kind == "grover":
        n = rng.randint(4, 31)
        return dict(kind=kind, n=n, iterations=rng.randint(1, 4 if n > 28 else 12),
                    fused=rng.choice([True, False]), dtype=dtype)
    if kind == "readout":
        return dict(kind=kind, n=rng.randint(8, 27), shots=_log_int(rng, 1, 4096), dtype=dtype)
    return dict(kind=kind, n=rng.randint(3, 20), layers=rng.randint(1, 10),
                batch=_log_int(rng, 1, 64), checkpoint=rng.choice([0, 2]), dtype=dtype)


# ---- values from a seed ---------------------------------------------------------

def _rng(seed, what=0):
    return np.random.Generator(np.random.PCG64([int(seed), what]))


def _haar(rng, d, count):
    """`count` Haar-random d x d unitaries (QR of a complex Gaussian matrix,
    phases fixed by the diagonal of R)."""
    z = rng.standard_normal((count, d, d)) + 1j * rng.standard_normal((count, d, d))
    q, r = np.linalg.qr(z)
    ph = np.einsum("cii->ci", r)
    return q * (ph / np.abs(ph))[:, None, :]


def _triples(case):
    """Distinct qubit triples per layer: the circuit's wiring."""
    rng = _rng(case["circuit"], 1)
    return [[[int(q) for q in rng.permutation(case["n"])[:3]] for _ in range(case["triples"])]
            for _ in range(case["layers"])]


def _haar_layers(case, seed):
    n, layers = case["n"], case["layers"]
    return _haar(_rng(seed, 2), 2, layers * n).reshape(layers, n, 2, 2)


def _indices(n, seed):
    """Basis states whose amplitudes a program asks for."""
    return _rng(seed, 3).integers(0, 1 << n, min(READOUT, 1 << n), dtype=np.uint64)


def _random_state(n, seed, what):
    """A normalised Gaussian state (the probabilities of a deep random
    circuit)."""
    g = torch.Generator(device=_device())
    g.manual_seed(1000003 * int(seed) + what)
    x = torch.view_as_complex(torch.randn((1 << n, 2), generator=g, device=_device(),
                                          dtype=torch.float64))
    return x / torch.linalg.vector_norm(x)


def _uniforms(seed, count):
    return _rng(seed, 4).random(count)


def _block_targets(case):
    rng = _rng(case["circuit"], 5)
    return [[int(q) for q in rng.permutation(case["n"])[:case["k"]]]
            for _ in range(case["count"])]


def _winner(n, seed):
    """The basis state that a Grover oracle marks."""
    return int(_rng(seed, 10).integers(0, 1 << n))


def _shor(case, seed):
    """(N, a) of the period finding: N of the given bit length, a coprime."""
    number = {3: 7, 4: 15, 5: 21}[case["bits"]]
    coprime = [a for a in range(2, number) if math.gcd(a, number) == 1]
    return number, coprime[int(_rng(seed, 6).integers(len(coprime)))]


# ---- prepare ----------------------------------------------------------------------

def _teleport_circuit(hops):
    """The state of qubit 0 handed on over `hops` Bell pairs to the last
    qubit; the corrections of all hops follow the measurements."""
    c = QuantumCircuit()
    last = 2 * hops
    for h in range(hops):
        c.add_operation(ops.hadamard(2 * h + 1))
        c.add_operation(ops.cnot(2 * h + 1, 2 * h + 2))
    for h in range(hops):
        c.add_operation(ops.cnot(2 * h, 2 * h + 1))
        c.add_operation(ops.hadamard(2 * h))
    for q in range(last):
        c.add_measurement(q)
    for h in range(hops):
        c.add_conditional_operation(ops.not_(last), [(2 * h + 1, True)])
        c.add_conditional_operation(ops.pauli_z(last), [(2 * h, True)])
    return c


def _circuit_ops(case, seed):
    n, out = case["n"], []
    for mats, triples in zip(_haar_layers(case, seed), _triples(case)):
        out += [Operation(mats[q], [q]) for q in range(n)]
        out += [ops.cnot(q, q + 1) for q in range(n - 1)]
        out += [ops.cnx([a, b], c) if g % 2 == 0 else ops.cnz([a, b], c)
                for g, (a, b, c) in enumerate(triples)]
    return out


def _qft_ops(n):
    """Fourier transform: H and controlled phases from the top qubit down,
    then the swaps."""
    out = []
    for q in reversed(range(n)):
        out.append(ops.hadamard(q))
        for c in reversed(range(q)):
            ph = np.diag([1.0, np.exp(1j * math.pi / (1 << (q - c)))])
            out.append(Operation.controlled([c], ph, [q]))
    out += [ops.swap(q, n - 1 - q) for q in range(n // 2)]
    return out


def _shor_ops(case, seed):
    b = case["bits"]
    number, a = _shor(case, seed)
    count, work = list(range(2 * b)), list(range(2 * b, 3 * b))
    out = [ops.hadamard_transform(count), ops.not_(2 * b)]
    for i in count:
        f = pow(a, 1 << i, number)
        gate = ops.to_quantum_gate(lambda w, f=f: w * f % number if w < number else w, work)
        out.append(ops.to_controlled(gate, i))
    d = 1 << (2 * b)
    x = np.arange(d)
    out.append(Operation(np.exp(2j * math.pi / d * (np.outer(x, x) % d)) / math.sqrt(d), count))
    return out


def _grover_ops(case, w):
    """H on every qubit, then per iteration the oracle (-1 on w) and the
    diffusion H^n diag(1, -1, ..., -1) H^n, as ``circuits.grover_operations``
    builds them."""
    n = case["n"]
    layer = circuits.hadamard_layer(n, case["fused"])
    minus = Operation(-np.eye(2), [0])
    turn = [circuits.phase_flip(n, w)] + layer + [circuits.phase_flip(n, 0), minus] + layer
    return layer + turn * case["iterations"]


def prepare(case, seed):
    kind = case["kind"]
    s = dict(case=case, kind=kind)
    if kind == "teleport":
        q = _rng(seed, 7).standard_normal((1, 4)) @ np.eye(4)
        payload = (q[0, :2] + 1j * q[0, 2:]) / np.linalg.norm(q)
        zero = np.array([1.0, 0.0], dtype=np.complex128)
        s.update(qubits=[payload] + [zero] * (2 * case["hops"]), seed=int(seed),
                 circuit=_teleport_circuit(case["hops"]))
        return s
    if kind == "adjoint":
        ansatz = circuits.hardware_efficient_ansatz(case["n"], case["layers"])
        masks, coeffs = circuits.zz_chain_observable(case["n"])
        s["thetas"] = _rng(seed, 8).random((case["batch"], ansatz.nparams)) * 2 * math.pi
        s["expectation"] = Expectation(ParamCircuit.from_ansatz(ansatz), masks, coeffs,
                                       dtype=case["dtype"], checkpoint_every=case["checkpoint"])
        bits = case["n"] + (case["batch"] - 1).bit_length()
    elif kind == "readout":
        n = case["n"]
        s["registers"] = []
        x = _random_state(n, seed, 1)
        for v in (x, x + 0.3 * _random_state(n, seed, 2)):
            r = Register.from_int(n, 0, dtype=case["dtype"], seed=0)
            r.state = (v / torch.linalg.vector_norm(v)).cpu().numpy()
            s["registers"].append(r)
        s.update(uniforms=_uniforms(seed, case["shots"]), indices=_indices(n, seed))
        return s
    else:
        n = s["n"] = 3 * case["bits"] if kind == "shor" else case["n"]
        bits = n
        s["indices"] = _indices(n, seed) if n > WHOLE else None
        s["uniforms"] = _uniforms(seed, n)
        s["measure"] = case.get("measure", "none")
        s["measured"] = list(range(n))
        if kind == "circuit":
            s["ops"] = _circuit_ops(case, seed)
        elif kind == "qft":
            s["ops"] = _qft_ops(n)
            s["input"] = _random_state(n, seed, 3).cpu().numpy()
            s["indices"] = None
        elif kind == "shor":
            s["ops"] = _shor_ops(case, seed)
            s.update(measure="each", measured=list(range(2 * case["bits"])))
        elif kind == "blocks":
            mats = _haar(_rng(seed, 9), 1 << case["k"], case["count"])
            s["ops"] = [ops.hadamard(q) for q in range(n)]
            s["ops"] += [Operation(m, t) for m, t in zip(mats, _block_targets(case))]
        else:
            w = _winner(n, seed)
            s["ops"] = _grover_ops(case, w)
            if s["indices"] is not None:
                s["indices"][0] = w
    if bits >= JIT_FROM:
        run(s)
        _lib.load().qs_sweep_jit_wait()
    return s


# ---- run ---------------------------------------------------------------------------

def run(s):
    kind = s["kind"]
    if kind == "teleport":
        r = Register.from_qubits(s["qubits"], dtype=s["case"]["dtype"], seed=s["seed"])
        bits = r.apply_circuit(s["circuit"])
        out = {"bits": [v for _, v in bits], "state": r.state}
        r.close()
        return out
    if kind == "adjoint":
        e = s["expectation"].forward(s["thetas"])
        return {"energies": e, "gradients": s["expectation"].backward()}
    if kind == "readout":
        a, b = s["registers"]
        overlap = a.inner(b)
        return {"shots": a.sample(s["uniforms"]).astype(np.int64),
                "amplitudes": a.amplitudes(s["indices"]),
                "norm_overlap": np.array([a.norm_sqr(), overlap.real, overlap.imag])}
    n = s["n"]
    r = Register.from_int(n, 0, dtype=s["case"]["dtype"], seed=0)
    if "input" in s:
        r.state = s["input"]
    for op in s["ops"]:
        r.apply(op)
    out = {"state": r.state} if s["indices"] is None else {"amplitudes": r.amplitudes(s["indices"])}
    if s["measure"] == "each":
        out["bits"] = np.array([r.measure(q, s["uniforms"][q]) for q in s["measured"]])
    elif s["measure"] == "all":
        out["index"] = r.measure_all(s["uniforms"])
    r.close()
    return out


# ---- work --------------------------------------------------------------------------

def work(case):
    """Bytes: the state written once (read too where the case brings one),
    what is returned, and dense matrices.  Flops: complex products of the
    gates with a dense factor (a 2 x 2 on a pair of amplitudes 28, a D x D
    block 8 D per amplitude), phases at 6 per amplitude that changes."""
    kind = case["kind"]
    s = 16 if case["dtype"] == "c128" else 8
    if kind == "adjoint":
        n, p = case["n"], 2 * case["n"] * case["layers"]
        amps = case["batch"] * 2.0 ** n
        # forward, psi and lambda back, and the inner product of every rotation
        return {"bytes": 2 * s * amps + 16.0 * case["batch"] * p,
                "flops": amps * case["layers"] * n * (3 * (6 + 3) + 2 * 4.0)}
    n = {"teleport": lambda: 2 * case["hops"] + 1,
         "shor": lambda: 3 * case["bits"]}.get(kind, lambda: case["n"])()
    amps = 2.0 ** n
    few = 24.0 * min(READOUT, amps)
    out = 16.0 * amps if n <= WHOLE else few
    if kind == "teleport":
        return {"bytes": s * amps + out, "flops": amps * (3 * case["hops"] + 2) * 4.0}
    if kind == "circuit":
        return {"bytes": s * amps + out, "flops": 14 * amps * n * case["layers"]}
    if kind == "qft":
        return {"bytes": 2 * s * amps + 32 * amps,
                "flops": amps * (4.0 * n + 6 * 0.25 * n * (n - 1) / 2)}
    if kind == "shor":
        d = 4.0 ** case["bits"]
        return {"bytes": s * amps + out + 2 * 16 * d * d, "flops": 8 * amps * d}
    if kind == "blocks":
        d = 2.0 ** case["k"]
        return {"bytes": s * amps + out + 16 * d * d * case["count"],
                "flops": amps * (4 * n + 8 * d * case["count"])}
    if kind == "grover":
        return {"bytes": s * amps + out, "flops": 4 * amps * n * (2 * case["iterations"] + 1)}
    return {"bytes": 2 * s * amps + few, "flops": 12 * amps}


# ---- exact -------------------------------------------------------------------------

def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _c(a):
    return torch.as_tensor(np.ascontiguousarray(a, dtype=np.complex128), device=_device())


def _basis(n):
    x = torch.zeros(1 << n, dtype=torch.complex128, device=_device())
    x[0] = 1
    return x


def _one_per_qubit(x, mats, n):
    """mats[q] on every qubit q: the low qubits of x in groups, each product
    moving its group to the top, so that the order is the first again."""
    for lo in range(0, n, 5):
        m = np.eye(1)
        for q in range(lo, min(lo + 5, n)):
            m = np.kron(mats[q], m)
        x = torch.mm(_c(m), x.view(-1, m.shape[0]).t()).view(-1)
    return x


def _cnot_ladder(x, n):
    """cnot(q, q + 1) for q = 0 .. n - 2: bit q becomes the parity of bits
    0 .. q."""
    out = torch.empty_like(x)
    step = min(1 << n, 1 << 24)
    for at in range(0, 1 << n, step):
        y = torch.arange(at, at + step, device=x.device)
        out[at:at + step] = x[(y ^ (y << 1)) & ((1 << n) - 1)]
    return out


def _bits_first(x, qubits, n):
    """A view of x with one axis of 2 for each of `qubits`, in that order,
    before the other axes."""
    order = sorted(qubits)
    shape, top = [], n
    for q in reversed(order):
        shape += [1 << (top - q - 1), 2]
        top = q
    shape.append(1 << top)
    axis = {q: 2 * i + 1 for i, q in enumerate(reversed(order))}
    v = x.view(shape)
    first = [axis[q] for q in qubits]
    return v.permute(first + [i for i in range(len(shape)) if i not in first])


def _exact_circuit(case, seed):
    n = case["n"]
    x = _basis(n)
    for mats, triples in zip(_haar_layers(case, seed), _triples(case)):
        x = _cnot_ladder(_one_per_qubit(x, mats, n), n)
        for g, (a, b, c) in enumerate(triples):
            v = _bits_first(x, [a, b, c], n)[1, 1]
            if g % 2 == 0:
                old = v[0].clone()
                v[0] = v[1]
                v[1] = old
            else:
                v[1].mul_(-1)
    return x


def _exact_blocks(case, seed):
    n, k = case["n"], case["k"]
    x = torch.full((1 << n,), 2.0 ** (-n / 2), dtype=torch.complex128, device=_device())
    for m, targets in zip(_haar(_rng(seed, 9), 1 << k, case["count"]), _block_targets(case)):
        v = _bits_first(x, targets[::-1], n)
        w = torch.mm(_c(m), v.reshape(1 << k, -1)).view(v.shape)
        out = torch.empty_like(x)
        _bits_first(out, targets[::-1], n).copy_(w)
        x = out
    return x


def _exact_shor(case, seed):
    b = case["bits"]
    number, a = _shor(case, seed)
    d = 1 << (2 * b)
    f = np.zeros((1 << b, d), dtype=np.complex128)
    value = 1
    for x in range(d):
        f[value, x] = 1.0 / math.sqrt(d)
        value = value * a % number
    return np.fft.ifft(f, axis=1, norm="ortho").reshape(-1)


def _exact_adjoint(case, seed):
    n, layers, batch = case["n"], case["layers"], case["batch"]
    dev = _device()
    th = torch.as_tensor(_rng(seed, 8).random((batch, 2 * n * layers)) * 2 * math.pi, device=dev)
    idx = torch.arange(1 << n, device=dev)
    z = [1.0 - 2.0 * ((idx >> q) & 1).double() for q in range(n)]
    h = sum(z) + 0.5 * sum((z[q] * z[q + 1] for q in range(n - 1)), torch.zeros_like(z[0]))
    ring = torch.ones_like(z[0])
    for q in range(n):
        if q != (q + 1) % n:
            ring = ring * (1.0 - 2.0 * (((idx >> q) & (idx >> ((q + 1) % n))) & 1).double())

    def turn(x, axis, q, angle):
        v = x.view(batch, 1 << (n - q - 1), 2, 1 << q)
        c, t = torch.cos(angle / 2).view(-1, 1, 1), torch.sin(angle / 2).view(-1, 1, 1)
        out = torch.empty_like(v)
        if axis == "y":
            out[:, :, 0] = c * v[:, :, 0] - t * v[:, :, 1]
            out[:, :, 1] = t * v[:, :, 0] + c * v[:, :, 1]
        else:
            out[:, :, 0] = torch.complex(c, -t) * v[:, :, 0]
            out[:, :, 1] = torch.complex(c, t) * v[:, :, 1]
        return out.view(batch, -1)

    steps = [(axis, q, layer * 2 * n + i * n + q) for layer in range(layers)
             for i, axis in enumerate("yz") for q in range(n)]
    x = torch.zeros((batch, 1 << n), dtype=torch.complex128, device=dev)
    x[:, 0] = 1
    for i, (axis, q, p) in enumerate(steps):
        x = turn(x, axis, q, th[:, p])
        if (i + 1) % (2 * n) == 0:
            x = x * ring
    energies = ((x.real ** 2 + x.imag ** 2) * h).sum(1)
    lam = x * h
    grads = torch.zeros_like(th)
    for i in reversed(range(len(steps))):
        axis, q, p = steps[i]
        if (i + 1) % (2 * n) == 0:
            x, lam = x * ring, lam * ring
        xv = x.view(batch, 1 << (n - q - 1), 2, 1 << q)
        lv = lam.view(batch, 1 << (n - q - 1), 2, 1 << q)
        if axis == "y":  # Im <lam| Y |x>, Y = [[0, -i], [i, 0]]
            g = (lv[:, :, 1].conj() * xv[:, :, 0]).real - (lv[:, :, 0].conj() * xv[:, :, 1]).real
        else:
            g = (lv[:, :, 0].conj() * xv[:, :, 0]).imag - (lv[:, :, 1].conj() * xv[:, :, 1]).imag
        grads[:, p] = g.sum((1, 2))
        x, lam = turn(x, axis, q, -th[:, p]), turn(lam, axis, q, -th[:, p])
    return {"energies": energies, "gradients": grads}


def _numpy(x):
    return x.cpu().numpy() if isinstance(x, torch.Tensor) else x


def exact(case, seed):
    kind = case["kind"]
    if kind == "adjoint":
        return {k: v.cpu().numpy() for k, v in _exact_adjoint(case, seed).items()}
    if kind == "teleport":
        return None  # the collapsed state follows the drawn outcomes
    if kind == "readout":
        n = case["n"]
        x = _random_state(n, seed, 1)
        y = x + 0.3 * _random_state(n, seed, 2)
        y = y / torch.linalg.vector_norm(y)
        overlap = complex((x.conj() * y).sum())
        return {"shots": None, "amplitudes": _numpy(x[torch.as_tensor(
            _indices(n, seed).astype(np.int64), device=x.device)]),
            "norm_overlap": np.array([float((x.abs() ** 2).sum()), overlap.real, overlap.imag])}
    if kind == "qft":
        return {"state": np.fft.ifft(_random_state(case["n"], seed, 3).cpu().numpy(),
                                     norm="ortho")}
    if kind == "grover":
        n = case["n"]
        w, size = _winner(n, seed), 2.0 ** n
        angle = (2 * case["iterations"] + 1) * math.asin(1.0 / math.sqrt(size))
        on, off = math.sin(angle), math.cos(angle) / math.sqrt(size - 1.0)
        at = np.arange(1 << n, dtype=np.uint64) if n <= WHOLE else _indices(n, seed)
        if n > WHOLE:
            at[0] = w
        out = np.where(at == w, on, off).astype(np.complex128)
        return {"state" if n <= WHOLE else "amplitudes": out}
    if kind == "shor":
        return {"state": _exact_shor(case, seed), "bits": None}
    x = _exact_circuit(case, seed) if kind == "circuit" else _exact_blocks(case, seed)
    if case["n"] <= WHOLE:
        return {"state": _numpy(x)}
    return {"amplitudes": _numpy(x[torch.as_tensor(_indices(case["n"], seed).astype(np.int64),
                                                   device=x.device)])}
