"""GPU adjoint gradients against parameter shift (CPU oracle / numpy
goldens), central finite differences on the GPU, and closed forms."""
import math
import os

import numpy as np
import pytest

import oracle
from quaru_amd import circuits
from quaru_amd import operation as ops
from quaru_amd.adjoint import Expectation, ParamCircuit, expectation_function

pytestmark = pytest.mark.gpu


def oracle_energy(ans, theta, masks, coeffs):
    """Forward pass of the ansatz with the CPU oracle (FP64)."""
    s = oracle.new([False] * ans.n)
    for op in ans.ops:
        if op[0] == "ry":
            g = ops.ry(theta[op[2]], op[1])
        elif op[0] == "rz":
            g = ops.rz(theta[op[2]], op[1])
        else:
            g = ops.cz(op[1], op[2])
        s = oracle.apply_fast(s, g.matrix(), g.targets())
    return oracle.expect_zstrings(s, masks, coeffs)


def test_one_qubit_closed_form():
    pc = ParamCircuit(1).rotation("y", 0, 0).layer()
    ex = Expectation(pc, [1], [1.0])
    th = np.array([[0.3], [1.2], [2.9]])
    e = ex.forward(th)
    g = ex.backward()
    assert np.max(np.abs(e - np.cos(th[:, 0]))) < 1e-14
    assert np.max(np.abs(g[:, 0] + np.sin(th[:, 0]))) < 1e-14


@pytest.mark.parametrize("axis", ["x", "y", "z"])
def test_single_rotation_axes(axis):
    # <Z> after H then R_axis(t): X -> cos t on |0>, Y, Z via an H first
    pc = ParamCircuit(1)
    h = ops.hadamard(0)
    pc.gate(h.matrix(), [0]).rotation(axis, 0, 0).gate(h.matrix(), [0]).layer()
    ex = Expectation(pc, [1], [1.0])
    t = np.array([[0.77]])
    e = ex.forward(t)
    g = ex.backward()
    # finite difference on the same engine
    d = 1e-6
    fd = (ex.energies(t + d) - ex.energies(t - d)) / (2 * d)
    assert abs(g[0, 0] - fd[0]) < 1e-8
    assert np.isfinite(e).all()


@pytest.mark.parametrize("dtype,tol", [("c128", 1e-12), ("c64", 1e-5)])
def test_golden_4q_parameter_shift(golden, dtype, tol):
    g = golden("adj_4q.npz")
    ans = circuits.hardware_efficient_ansatz(int(g["n"]), int(g["layers"]))
    pc = ParamCircuit.from_ansatz(ans)
    ex = Expectation(pc, g["masks"], g["coeffs"], dtype=dtype)
    e = ex.forward(g["thetas"])
    gr = ex.backward()
    assert np.max(np.abs(e - g["energies"])) < tol
    assert np.max(np.abs(gr - g["grads"])) < tol


@pytest.mark.parametrize("checkpoint", [0, 2])
def test_adjoint_vs_fd_and_parameter_shift(checkpoint):
    n, layers, batch = 8, 3, 5
    ans = circuits.hardware_efficient_ansatz(n, layers)
    masks, coeffs = circuits.zz_chain_observable(n)
    th = circuits.seeded_thetas(batch, ans.nparams, seed=3)
    pc = ParamCircuit.from_ansatz(ans)
    ex = Expectation(pc, masks, coeffs, checkpoint_every=checkpoint)
    e = ex.forward(th)
    g = ex.backward()
    # energies vs the oracle
    for b in range(batch):
        assert abs(e[b] - oracle_energy(ans, th[b], masks, coeffs)) < 1e-12
    # central FD (h = 1e-4, FP64) on the GPU for every parameter of set 0,2
    h = 1e-4
    for b in (0, 2):
        plus = np.repeat(th[b:b + 1], ans.nparams, axis=0)
        minus = plus.copy()
        idx = np.arange(ans.nparams)
        plus[idx, idx] += h
        minus[idx, idx] -= h
        fd = (ex.energies(plus) - ex.energies(minus)) / (2 * h)
        assert np.max(np.abs(fd - g[b])) < 1e-6
    # parameter shift with the CPU oracle on a sample of parameters
    for p in (0, 7, ans.nparams - 1):
        tp, tm = th[1].copy(), th[1].copy()
        tp[p] += math.pi / 2
        tm[p] -= math.pi / 2
        ps = 0.5 * (oracle_energy(ans, tp, masks, coeffs) - oracle_energy(ans, tm, masks, coeffs))
        assert abs(ps - g[1, p]) < 1e-11


def _mixed_circuit(n, seed):
    """Rotations (X, Y, Z; some parameters used twice) between fixed gates of
    every kind the reverse pass handles: H and CNOT (one dense target, the
    CNOT's control off a 10-qubit tile), a controlled phase and a CZ (diagonal
    on any qubits), a SWAP and a Haar 2-qubit gate (two dense targets: run
    by the per-gate kernels between tiled blocks).  Returns (ops, nparams):
    op = ("rot", axis, q, p) or ("gate", matrix, targets)."""
    from tests.conftest import random_unitary
    rng = np.random.default_rng(seed)
    out, p = [], 0
    for layer in range(3):
        for q in rng.permutation(n)[:8]:
            out.append(("rot", "xyz"[int(rng.integers(3))], int(q), p))
            p += 1
        out.append(("rot", "y", int(rng.integers(n)), p - 3))  # a shared parameter
        g = ops.hadamard(int(rng.integers(n)))
        out.append(("gate", g.matrix(), g.targets()))
        g = ops.cnot(n - 1, 2)
        out.append(("gate", g.matrix(), g.targets()))
        cp = np.diag([1, 1, 1, np.exp(0.7j)])
        out.append(("gate", cp, [3, n - 2]))
        g = ops.cz(0, n - 3)
        out.append(("gate", g.matrix(), g.targets()))
        g = ops.swap(1, 9)
        out.append(("gate", g.matrix(), g.targets()))
        out.append(("gate", random_unitary(rng, 4), [5, n - 1]))
        for q in rng.permutation(n)[:6]:
            out.append(("rot", "xyz"[int(rng.integers(3))], int(q), p))
            p += 1
    return out, p


def _mixed_oracle_energy(n, circ, angles, masks, coeffs):
    """angles[i]: the angle of the i-th rotation occurrence."""
    s = oracle.new([False] * n)
    k = 0
    for op in circ:
        if op[0] == "rot":
            g = {"x": ops.rx, "y": ops.ry, "z": ops.rz}[op[1]](angles[k], op[2])
            k += 1
            s = oracle.apply_fast(s, g.matrix(), g.targets())
        else:
            s = oracle.apply_fast(s, op[1], op[2])
    return oracle.expect_zstrings(s, masks, coeffs)


@pytest.mark.parametrize("dtype,tol", [("c128", 1e-11), ("c64", 2e-5)])
def test_mixed_gates_shared_parameters_vs_parameter_shift(dtype, tol):
    n = 13
    circ, nparams = _mixed_circuit(n, seed=21)
    masks, coeffs = circuits.zz_chain_observable(n)
    th = circuits.seeded_thetas(2, nparams, seed=4)
    pc = ParamCircuit(n)
    for op in circ:
        if op[0] == "rot":
            pc.rotation(op[1], op[2], op[3])
        else:
            pc.gate(op[1], op[2])
        pc.layer()
    ex = Expectation(pc, masks, coeffs, dtype=dtype, checkpoint_every=4)
    e = ex.forward(th)
    g = ex.backward()
    occ = [op[3] for op in circ if op[0] == "rot"]
    for b in range(2):
        ang = np.array([th[b, p] for p in occ])
        assert abs(e[b] - _mixed_oracle_energy(n, circ, ang, masks, coeffs)) < tol
        # parameter shift per occurrence, summed over a parameter's uses
        ref = np.zeros(nparams)
        for i, p in enumerate(occ):
            ap, am = ang.copy(), ang.copy()
            ap[i] += math.pi / 2
            am[i] -= math.pi / 2
            ref[p] += 0.5 * (_mixed_oracle_energy(n, circ, ap, masks, coeffs)
                             - _mixed_oracle_energy(n, circ, am, masks, coeffs))
        assert np.max(np.abs(g[b] - ref)) < tol


def test_c64_adjoint_agrees_with_c128():
    n, layers, batch = 10, 4, 4
    ans = circuits.hardware_efficient_ansatz(n, layers)
    masks, coeffs = circuits.zz_chain_observable(n)
    th = circuits.seeded_thetas(batch, ans.nparams, seed=9)
    pc = ParamCircuit.from_ansatz(ans)
    g = {}
    for dt in ("c128", "c64"):
        ex = Expectation(pc, masks, coeffs, dtype=dt, checkpoint_every=2)
        ex.forward(th)
        g[dt] = ex.backward()
    assert np.max(np.abs(g["c64"] - g["c128"])) < 1e-5


def test_torch_autograd_function():
    torch = pytest.importorskip("torch")
    n, layers = 6, 2
    ans = circuits.hardware_efficient_ansatz(n, layers)
    masks, coeffs = circuits.zz_chain_observable(n)
    ex = Expectation(ParamCircuit.from_ansatz(ans), masks, coeffs)
    th = torch.tensor(circuits.seeded_thetas(3, ans.nparams, seed=1), requires_grad=True)
    E = expectation_function().apply(th, ex)
    w = torch.tensor([1.0, -2.0, 0.5], dtype=torch.float64)
    (E * w).sum().backward()
    ex2 = Expectation(ParamCircuit.from_ansatz(ans), masks, coeffs)
    ex2.forward(th.detach().numpy())
    ref = ex2.backward() * w.numpy()[:, None]
    assert np.max(np.abs(th.grad.numpy() - ref)) < 1e-12


def test_torch_two_forwards_before_one_backward():
    """loss = f(t1) + 2 f(t2) through one Expectation: each application keeps
    its own device state, so both gradients are right; a 1-D thetas gets a
    gradient of its own shape."""
    torch = pytest.importorskip("torch")
    n, layers = 5, 2
    ans = circuits.hardware_efficient_ansatz(n, layers)
    masks, coeffs = circuits.zz_chain_observable(n)
    ex = Expectation(ParamCircuit.from_ansatz(ans), masks, coeffs)
    t_all = circuits.seeded_thetas(2, ans.nparams, seed=21)
    t1 = torch.tensor(t_all[0], requires_grad=True)          # 1-D
    t2 = torch.tensor(t_all[1:2], requires_grad=True)        # (1, P)
    f = expectation_function()
    loss = f.apply(t1, ex).sum() + 2.0 * f.apply(t2, ex).sum()
    loss.backward()
    assert t1.grad.shape == t1.shape and t2.grad.shape == t2.shape
    ref = Expectation(ParamCircuit.from_ansatz(ans), masks, coeffs)
    ref.forward(t_all)
    g = ref.backward()
    assert np.max(np.abs(t1.grad.numpy() - g[0])) < 1e-12
    assert np.max(np.abs(t2.grad.numpy()[0] - 2.0 * g[1])) < 1e-12


def _omp_threads() -> int:
    return max(1, min(16, os.cpu_count() or 1))


def oracle_layer_states(ans, theta):
    """The oracle's state at the start of every layer (and at the end), by
    the multi-core try_apply_fast restatement (bit-identical to the scalar
    one)."""
    n = ans.n
    s = oracle.new([False] * n)
    scratch = np.empty_like(s)
    states = [s.copy()]
    start = 0
    for end in ans.layer_ends:
        for op in ans.ops[start:end]:
            g = _ansatz_gate(op, theta)
            oracle.apply_fast_omp(s, scratch, g.matrix(), g.targets(), _omp_threads())
        states.append(s.copy())
        start = end
    return states


def _ansatz_gate(op, theta):
    if op[0] == "ry":
        return ops.ry(theta[op[2]], op[1])
    if op[0] == "rz":
        return ops.rz(theta[op[2]], op[1])
    return ops.cz(op[1], op[2])


def oracle_energy_from(ans, theta, state, layer, masks, coeffs):
    """Finish the forward pass on the oracle from the start of `layer`."""
    s = state.copy()
    scratch = np.empty_like(s)
    start = 0 if layer == 0 else ans.layer_ends[layer - 1]
    for op in ans.ops[start:]:
        g = _ansatz_gate(op, theta)
        oracle.apply_fast_omp(s, scratch, g.matrix(), g.targets(), _omp_threads())
    return oracle.expect_zstrings(s, masks, coeffs)


_ANSATZ20 = {}


def _ansatz20_reference():
    """The differentiation workload at its own size: 20 qubits, 10 layers of
    RY/RZ on every qubit and a CZ ring (400 parameters), H = sum Z_i + 0.5
    sum Z_i Z_{i+1}, a batch of 64 seeded parameter sets.  FP64 checks:
    oracle energies of sets 0 and 1; central finite differences (h = 1e-4)
    of 16 seeded parameters of set 1 on the complex128 engine; oracle
    parameter shift of 4 parameters of set 1 in layers 9, 8, 7 and 5
    (started from the oracle's cached layer states)."""
    if _ANSATZ20:
        return _ANSATZ20
    n, layers, batch = 20, 10, 64
    ans = circuits.hardware_efficient_ansatz(n, layers)
    masks, coeffs = circuits.zz_chain_observable(n)
    th = circuits.seeded_thetas(batch, ans.nparams, seed=5)
    print("20-qubit ansatz: oracle forward of sets 0 and 1", flush=True)
    e0 = oracle_energy_from(ans, th[0], oracle.new([False] * n), 0, masks, coeffs)
    states1 = oracle_layer_states(ans, th[1])
    e1 = oracle.expect_zstrings(states1[-1], masks, coeffs)
    ps = {}
    per_layer = 2 * n
    for layer, k in ((9, 3), (8, n + 7), (7, 11), (5, n + 19)):
        p = layer * per_layer + k
        tp, tm = th[1].copy(), th[1].copy()
        tp[p] += math.pi / 2
        tm[p] -= math.pi / 2
        ps[p] = 0.5 * (oracle_energy_from(ans, tp, states1[layer], layer, masks, coeffs)
                       - oracle_energy_from(ans, tm, states1[layer], layer, masks, coeffs))
        print(f"20-qubit ansatz: parameter shift of parameter {p} done", flush=True)
    rng = np.random.default_rng(55)
    fd_params = np.sort(rng.choice(ans.nparams, 16, replace=False))
    h = 1e-4
    plus = np.repeat(th[1:2], fd_params.size, axis=0)
    minus = plus.copy()
    plus[np.arange(fd_params.size), fd_params] += h
    minus[np.arange(fd_params.size), fd_params] -= h
    ex = Expectation(ParamCircuit.from_ansatz(ans), masks, coeffs, dtype="c128")
    fd = (ex.energies(plus) - ex.energies(minus)) / (2 * h)
    _ANSATZ20.update(ans=ans, masks=masks, coeffs=coeffs, th=th, e=(e0, e1), ps=ps,
                    fd_params=fd_params, fd=fd)
    return _ANSATZ20


@pytest.mark.parametrize("dtype", ["c128", "c64"])
def test_ansatz20_full_size(dtype):
    """20 qubits x 10 layers x batch 64, checkpoint every 2 layers, in both
    precisions: energies against the oracle, gradients against central FD
    (FP64, h = 1e-4) and oracle parameter shift, all within 1e-5 (complex128
    energies within 1e-10)."""
    ref = _ansatz20_reference()
    ans, th = ref["ans"], ref["th"]
    ex = Expectation(ParamCircuit.from_ansatz(ans), ref["masks"], ref["coeffs"], dtype=dtype,
                     checkpoint_every=2)
    print(f"20-qubit ansatz {dtype}: forward + backward, batch {th.shape[0]}", flush=True)
    e = ex.forward(th)
    g = ex.backward()
    assert e.shape == (64,) and g.shape == (64, 400)
    assert np.isfinite(g).all() and np.max(np.abs(g)) > 0.1
    etol = 1e-10 if dtype == "c128" else 1e-5
    assert abs(e[0] - ref["e"][0]) < etol and abs(e[1] - ref["e"][1]) < etol
    assert np.max(np.abs(g[1, ref["fd_params"]] - ref["fd"])) < 1e-5
    for p, v in ref["ps"].items():
        assert abs(g[1, p] - v) < 1e-5, (p, g[1, p], v)
    if dtype == "c128":
        # the same batch without checkpoints gives the same gradients
        ex0 = Expectation(ParamCircuit.from_ansatz(ans), ref["masks"], ref["coeffs"])
        ex0.forward(th[:8])
        assert np.max(np.abs(ex0.backward() - g[:8])) < 1e-10


@pytest.mark.parametrize("dtype,tol", [("c128", 1e-12), ("c64", 2e-5)])
@pytest.mark.parametrize("n,batch", [(1, 3), (5, 5), (9, 3), (10, 33), (11, 5), (13, 9)])
def test_batches_equal_their_parameter_sets_alone(n, batch, dtype, tol):
    # padding states of a batch are left out; tiles of every size
    ans = circuits.hardware_efficient_ansatz(n, 3)
    masks, coeffs = circuits.zz_chain_observable(n)
    th = circuits.seeded_thetas(batch, ans.nparams, seed=17)
    pc = ParamCircuit.from_ansatz(ans)
    ex = Expectation(pc, masks, coeffs, dtype=dtype, checkpoint_every=2)
    e = ex.forward(th)
    g = ex.backward()
    one = Expectation(pc, masks, coeffs, dtype="c128")
    for b in sorted({0, batch // 2, batch - 1}):
        eb = one.forward(th[b])
        gb = one.backward()
        assert np.max(np.abs(e[b] - eb[0])) < tol * n
        assert np.max(np.abs(g[b] - gb[0])) < tol * n


@pytest.mark.parametrize("dtype,tol", [("c128", 1e-9), ("c64", 2e-3)])
@pytest.mark.parametrize("n", [2, 8, 9, 11, 14])
def test_reverse_blocks_with_every_record(n, dtype, tol):
    # rotations about all axes in any order, several Z rotations of one qubit
    # in a row, phases and diagonals on and off the tile, controlled 2x2s:
    # against central differences of the engine's own FP64 energies
    rng = np.random.default_rng(n)
    pc = ParamCircuit(n)
    p = 0
    for _ in range(70):
        k = rng.integers(0, 8)
        a, b = (int(q) for q in rng.permutation(n)[:2])
        if k < 4:
            pc.rotation("xyzz"[k], a, p)
            p += 1
        elif k == 4:
            pc.gate(np.diag(np.exp(1j * rng.random(4) * 6)), [a, b])
        elif k == 5:
            pc.gate(ops.cz(a, b).matrix(), [a, b])
        elif k == 6:
            pc.gate(np.diag([1, 1, 1, np.exp(0.7j)]), [a, b])
        else:
            pc.gate(ops.cnot(a, b).matrix(), ops.cnot(a, b).targets())
    masks, coeffs = circuits.zz_chain_observable(n)
    th = rng.random((3, p)) * 6.2
    ex = Expectation(pc, masks, coeffs, dtype=dtype)
    ex.forward(th)
    g = ex.backward()
    fd = Expectation(pc, masks, coeffs, dtype="c128")
    for q in sorted({0, p // 3, p // 2, p - 1}):
        d = np.zeros(p)
        d[q] = 1e-4
        want = (fd.energies(th + d) - fd.energies(th - d)) / 2e-4
        assert np.max(np.abs(g[:, q] - want)) < max(tol, 1e-6)


def shift_gradients(ex, th):
    """dE/dtheta by the shift rule, exact for rotations exp(-i t sigma / 2)
    with a parameter each, in batches of shifted sets."""
    p = th.shape[1]
    out = np.empty_like(th)
    for b, t in enumerate(th):
        e = ex.energies(np.concatenate([t + np.eye(p) * np.pi / 2, t - np.eye(p) * np.pi / 2]))
        out[b] = (e[:p] - e[p:]) / 2
    return out


@pytest.mark.parametrize("dtype,tol", [("c128", 1e-11), ("c64", 1e-4)])
@pytest.mark.parametrize("n", [3, 6, 9, 12, 14])
def test_gates_that_are_not_unitary_before_the_rotations(n, dtype, tol):
    """A preparation that is no unitary (columns of zeros, weights on the
    diagonal) in front of the rotations: nothing that commutes with it may be
    taken after it in the reverse pass."""
    rng = np.random.default_rng(600 + n)
    pc = ParamCircuit(n)
    for q in range(n):
        pc.gate(np.array([[0.8, 0.1], [0.5j, -0.3]]), [q])
    pc.gate(np.diag([1.0, 0.7]), [n - 1])
    pc.gate(np.diag([1.0, 1.0, 1.0, 0.4j]), [0, n - 1])
    pc.gate(np.diag([1.0, 0.9, 0.8, 0.6]), [1, 0])
    for layer in range(3):
        for q in range(n):
            pc.rotation("yxz"[(q + layer) % 3], q, pc.nparams)
            pc.rotation("z", q, pc.nparams)
        for q in range(n - 1):
            g = ops.cnot(q, q + 1) if q % 2 else ops.cz(q, q + 1)
            pc.gate(g.matrix(), g.targets())
    masks, coeffs = circuits.zz_chain_observable(n)
    th = rng.random((2, pc.nparams)) * 6.2
    ex = Expectation(pc, masks, coeffs, dtype=dtype)
    ex.forward(th)
    g = ex.backward()
    want = shift_gradients(Expectation(pc, masks, coeffs, dtype="c128"), th)
    assert np.max(np.abs(want)) > 1e-4
    assert np.max(np.abs(g - want)) < tol * n


def long_gradients(n, ansatz, masks, coeffs, th):
    """Gradients of RY / RZ / CZ circuits in 80-bit arithmetic."""
    idx = np.arange(1 << n)
    h = np.zeros(1 << n, dtype=np.longdouble)
    for m, c in zip(masks, coeffs):
        odd = np.array([bin(int(m) & i).count("1") & 1 for i in range(1 << n)])
        h += np.where(odd == 1, -np.longdouble(c), np.longdouble(c))

    def turn(x, op, t):
        if op[0] == "cz":
            x[(idx >> op[1]) & (idx >> op[2]) & 1 == 1] *= -1
            return
        v = x.reshape(-1, 2, 1 << op[1])
        a, b = v[:, 0].copy(), v[:, 1].copy()
        c, s = np.cos(t / 2), np.sin(t / 2)
        v[:, 0], v[:, 1] = ((c * a - s * b, s * a + c * b) if op[0] == "ry"
                            else ((c - 1j * s) * a, (c + 1j * s) * b))

    out = np.zeros(th.shape, dtype=np.longdouble)
    for g, t in zip(out, th.astype(np.longdouble)):
        x = np.zeros(1 << n, dtype=np.clongdouble)
        x[0] = 1
        for op in ansatz.ops:
            turn(x, op, t[op[2]])
        lam = h * x
        for op in reversed(ansatz.ops):
            if op[0] != "cz":
                v, w = (y.reshape(-1, 2, 1 << op[1]) for y in (x, np.conj(lam)))
                g[op[2]] += np.sum(w[:, 1] * v[:, 0] - w[:, 0] * v[:, 1]).real if op[0] == "ry" \
                    else np.sum(w[:, 0] * v[:, 0] - w[:, 1] * v[:, 1]).imag
            for y in (x, lam):
                turn(y, op, -t[op[2]])
    return out


@pytest.mark.parametrize("n,batch,bound", [(8, 24, 2.9e-16), (13, 8, 4.1e-16)])
def test_gradients_as_close_as_one_operation_at_a_time(n, batch, bound):
    """Root mean square of the error of complex128 gradients against 80-bit
    arithmetic; the bounds are what the reverse pass with one kernel per
    operation leaves (each rotation rounded by itself on each amplitude)."""
    ans = circuits.hardware_efficient_ansatz(n, 10)
    masks, coeffs = circuits.zz_chain_observable(n)
    th = np.random.default_rng(700 + n).random((batch, ans.nparams)) * 2 * np.pi
    ex = Expectation(ParamCircuit.from_ansatz(ans), masks, coeffs)
    ex.forward(th)
    err = ex.backward() - long_gradients(n, ans, masks, coeffs, th)
    assert np.sqrt(np.mean(err ** 2)) < bound


@pytest.mark.parametrize("dtype,tol", [("c128", 1e-11), ("c64", 1e-4)])
@pytest.mark.parametrize("n", [2, 5, 8, 10, 12, 13])
def test_reverse_blocks_against_the_shift_rule(n, dtype, tol):
    """Every parameter of circuits with every record of the reverse blocks
    (rotations about all axes, several Z rotations of one qubit in a row,
    phases and diagonals on and off the tile, dense and controlled 2x2s, a 4x4
    in between), of all parameter sets of a batch that is no power of two."""
    rng = np.random.default_rng(40 + n)
    pc = ParamCircuit(n)
    for step in range(90):
        k = int(rng.integers(0, 10))
        a, b = (int(q) for q in rng.permutation(n)[:2])
        if k < 5:
            pc.rotation("xyzzz"[k], a, pc.nparams)
            if k == 4:
                pc.rotation("z", a, pc.nparams)
        elif k == 5:
            pc.gate(np.diag(np.exp(1j * rng.random(4) * 6)), [a, b])
        elif k == 6:
            pc.gate(ops.cz(a, b).matrix(), [a, b])
        elif k == 7:
            pc.gate(np.diag([1, 1, 1, np.exp(0.7j)]), [a, b])
        elif k == 8:
            g = ops.cnot(a, b) if step % 2 else ops.to_controlled(ops.Operation(random_u(rng, 2), [a]), b)
            pc.gate(g.matrix(), g.targets())
        else:
            pc.gate(random_u(rng, 4 if step % 3 == 0 else 2), [a, b] if step % 3 == 0 else [a])
        if step % 30 == 29:
            pc.layer()
    masks, coeffs = circuits.zz_chain_observable(n)
    th = rng.random((3, pc.nparams)) * 6.2
    want = shift_gradients(Expectation(pc, masks, coeffs), th)
    for every in (0, 1):
        ex = Expectation(pc, masks, coeffs, dtype=dtype, checkpoint_every=every)
        ex.forward(th)
        assert np.max(np.abs(ex.backward() - want)) < tol


def random_u(rng, d):
    q, r = np.linalg.qr(rng.standard_normal((d, d)) + 1j * rng.standard_normal((d, d)))
    return q * (np.diag(r) / np.abs(np.diag(r)))


@pytest.mark.parametrize("dtype,batch,tol", [("c128", 8200, 1e-11), ("c64", 2050, 1e-4)])
def test_batches_beyond_a_sweeps_descriptor(dtype, batch, tol):
    """Rotations of so many parameter sets that a sweep has no room for their
    matrices: energies and gradients of some of the sets alone."""
    n = 12
    ans = circuits.hardware_efficient_ansatz(n, 1)
    masks, coeffs = circuits.zz_chain_observable(n)
    th = circuits.seeded_thetas(batch, ans.nparams, seed=23)
    pc = ParamCircuit.from_ansatz(ans)
    ex = Expectation(pc, masks, coeffs, dtype=dtype)
    e = ex.forward(th)
    g = ex.backward()
    some = [0, batch // 3, batch - 1]
    one = Expectation(pc, masks, coeffs)
    assert np.max(np.abs(e[some] - one.forward(th[some]))) < tol * n
    assert np.max(np.abs(g[some] - one.backward())) < tol * n
