"""Operation lists at the circuit-capture boundary (qmxCircuit*, qmxApplyOperations)
against the oracle of QuantumLab's own loop (oracle/ops_oracle.py: one QuEST
call per EBasicOperation, QLGate.cpp:652-803, and the density simulator's
after-gate noise, QLSimulatorDensityMatrix.cpp:88-153) run on the C restatement
of QuEST's CPU backend.

CPU tests: record-time validation (no GPU). GPU tests: FP64 state vectors and
density matrices within 1e-12 of the oracle, fused or not; FP32 fused MFMA
blocks within FP32 resolution; collapse probabilities equal."""
import ctypes as C

import numpy as np
import pytest

from oracle import ops_oracle as O
from quantumlab_amd import workloads as W
from quantumlab_amd.quest import QMX_PREC_FP32, BasicOperation, NoiseAfterGate, QuESTError
from tests.cases import ints

TOL = 1e-12


def _lib_cpu():
    import os

    import quantumlab_amd
    lib = C.CDLL(quantumlab_amd.library_path(), mode=os.RTLD_LOCAL)
    lib.qmxSetErrorMode(1)
    lib.qmxCircuitCreate.restype = C.c_void_p
    lib.qmxCircuitCreate.argtypes = [C.c_int]
    lib.qmxCircuitDestroy.argtypes = [C.c_void_p]
    lib.qmxCircuitNumGates.argtypes = [C.c_void_p]
    lib.qmxCircuitAddOperation.argtypes = [C.c_void_p, C.c_int, C.POINTER(C.c_int), C.c_int, C.c_double]
    lib.qmxCircuitFuse.argtypes = [C.c_void_p, C.c_int]
    lib.qmxCircuitSetNoiseAfterGate.argtypes = [C.c_void_p, NoiseAfterGate]
    lib.qmxLastError.argtypes = [C.c_char_p, C.c_int]
    lib.qmxClearError()
    return lib


def _last_error(lib):
    buf = C.create_string_buffer(1024)
    had = lib.qmxLastError(buf, 1024)
    lib.qmxClearError()
    return buf.value.decode() if had else None


@pytest.mark.parametrize("code,qubits,param,substr", [
    (O.H, [5], 0.0, "Invalid target"),
    (O.H, [-1], 0.0, "Invalid target"),
    (O.CX, [2, 2], 0.0, "Control qubit cannot equal target"),
    (O.CRZ, [7, 1], 0.3, "Invalid control"),
    (O.CX, [1], 0.0, "exactly two qubits"),
    (O.RX, [0, 1], 0.1, "exactly one qubit"),
    (O.CC, [1], 2.0, "Invalid measurement outcome"),
    (O.NOISE_DEPHASING, [1], 0.6, "cannot exceed 1/2"),
    (O.NOISE_DEPOLARISING, [1], 0.8, "cannot exceed 3/4"),
    (O.NOISE_TWO_DEPOLARISING, [1, 1], 0.1, "target qubits must be unique"),
    (O.NOISE_DAMPING, [0], -0.1, "Probabilities must be in [0, 1]"),
    (99, [0], 0.0, "Invalid operation code"),
])
def test_circuit_records_reject_invalid_operations(code, qubits, param, substr):
    lib = _lib_cpu()
    c = lib.qmxCircuitCreate(5)
    lib.qmxCircuitAddOperation(c, code, ints(qubits), len(qubits), param)
    err = _last_error(lib)
    assert err is not None and substr in err, err
    assert lib.qmxCircuitNumGates(c) == 0
    lib.qmxCircuitDestroy(c)


def test_circuit_width_and_block_size_validated():
    lib = _lib_cpu()
    assert lib.qmxCircuitCreate(0) is None
    assert "Invalid number of qubits" in _last_error(lib)
    c = lib.qmxCircuitCreate(4)
    lib.qmxCircuitAddOperation(c, O.H, ints([3]), 1, 0.0)
    lib.qmxCircuitAddOperation(c, O.CX, ints([3, 0]), 2, 0.0)
    assert _last_error(lib) is None and lib.qmxCircuitNumGates(c) == 2
    for bad in (0, 11):
        lib.qmxCircuitFuse(c, bad)
        assert "Invalid block size" in _last_error(lib)
    assert lib.qmxCircuitFuse(c, 2) == 1
    lib.qmxCircuitSetNoiseAfterGate(c, NoiseAfterGate(0.1, 0.7, 0, 0, 0, 0))
    assert "cannot exceed 1/2" in _last_error(lib)
    lib.qmxCircuitDestroy(c)


# ---- GPU parity --------------------------------------------------------------------------

def resolve_collapses(qe, q, ops, noise=None):
    """Run ops on the oracle, fixing each collapse's outcome to the likelier one
    (so its probability is well away from 0); returns the completed list."""
    out = []
    for code, qs, t in ops:
        if code == O.CC and t < 0:
            p0 = qe.calcProbOfOutcome(q, qs[0], 0)
            t = 0.0 if p0 >= 0.5 else 1.0
        op = (code, qs, t)
        out.append(op)
        O.perform(qe, q, op)
        if noise and q.isDensityMatrix:
            O.noise_after_gate(qe, q, op, noise)
    return out


def record(gpu, n, ops, noise=None):
    c = gpu.lib.qmxCircuitCreate(n)
    for code, qs, t in ops:
        gpu.call("qmxCircuitAddOperation", c, code, ints(qs), len(qs), t)
    if noise:
        gpu.call("qmxCircuitSetNoiseAfterGate", c, NoiseAfterGate(**noise))
    return c


def oracle_state(cpuref, n, ops, density=False, noise=None, init=None):
    q = cpuref.qureg(n, density=density)
    if init is not None:
        init(cpuref, q)
    prob = O.run_ops(cpuref, q, ops, noise)
    st = cpuref.state(q)
    cpuref.destroy(q)
    return st, prob


def _init_plus(lib, q):
    lib.initPlusState(q)


@pytest.mark.gpu
@pytest.mark.parametrize("fuse", [0, 3, 5])
def test_state_vector_op_list_matches_oracle(gpu, cpuref, fuse):
    n = 12
    raw = O.random_ops(n, 400, seed=21, noise=True, collapses=3)
    raw.insert(7, (O.PHASE, [2], 0.4))
    q0 = cpuref.qureg(n)
    cpuref.initPlusState(q0)
    ops = resolve_collapses(cpuref, q0, raw)
    cpuref.destroy(q0)
    ref, pref = oracle_state(cpuref, n, ops, init=_init_plus)
    c = record(gpu, n, ops)
    q = gpu.qureg(n)
    gpu.initPlusState(q)
    if fuse:
        assert gpu.qmxCircuitFuse(c, fuse) > 0
    prob = gpu.qmxCircuitApply(q, c, 1 if fuse else 0)
    assert abs(prob - pref) < TOL
    assert np.max(np.abs(gpu.state(q) - ref)) < TOL
    gpu.destroy(q)
    gpu.qmxCircuitDestroy(c)


@pytest.mark.gpu
def test_apply_operations_entry_matches_circuit(gpu, cpuref):
    n = 10
    q0 = cpuref.qureg(n)
    ops = resolve_collapses(cpuref, q0, O.random_ops(n, 150, seed=5, collapses=2))
    cpuref.destroy(q0)
    ref, pref = oracle_state(cpuref, n, ops)
    arr = (BasicOperation * len(ops))()
    for i, (code, qs, t) in enumerate(ops):
        arr[i].operation = code
        arr[i].numQubits = len(qs)
        for j, x in enumerate(qs):
            arr[i].qubits[j] = x
        arr[i].param = t
    for fuse in (0, 4):
        q = gpu.qureg(n)
        prob = gpu.qmxApplyOperations(q, arr, len(ops), None, fuse)
        assert abs(prob - pref) < TOL
        assert np.max(np.abs(gpu.state(q) - ref)) < TOL
        gpu.destroy(q)


NOISES = [
    dict(damping=0.03, dephasing=0.02, depolarising=0.01, mixPauli=0.005),
    dict(damping=0.01, dephasing=0.02, depolarising=0.01, twoQubitDephasing=0.03, twoQubitDepolarising=0.02),
]


@pytest.mark.gpu
@pytest.mark.parametrize("noise_idx", [0, 1])
def test_density_op_list_with_noise_matches_oracle(gpu, cpuref, noise_idx):
    """Noise operations and the simulator's after-gate noise on a density register."""
    n = 6
    noise = NOISES[noise_idx]
    q0 = cpuref.qureg(n, density=True)
    ops = resolve_collapses(cpuref, q0, O.random_ops(n, 120, seed=30 + noise_idx, noise=True, collapses=2),
                            noise)
    cpuref.destroy(q0)
    ref, pref = oracle_state(cpuref, n, ops, density=True, noise=noise)
    c = record(gpu, n, ops, noise)
    q = gpu.qureg(n, density=True)
    prob = gpu.qmxCircuitApply(q, c, 1)  # fused on a density register: the ops in order
    assert abs(prob - pref) < TOL
    assert np.max(np.abs(gpu.state(q) - ref)) < TOL
    gpu.destroy(q)
    gpu.qmxCircuitDestroy(c)


@pytest.mark.gpu
def test_circuit_apply_rejects_other_widths(gpu):
    c = record(gpu, 6, [(O.H, [5], 0.0)])
    q = gpu.qureg(5)
    with pytest.raises(QuESTError, match="different numbers of qubits"):
        gpu.qmxCircuitApply(q, c, 0)
    gpu.destroy(q)
    q = gpu.qureg(3, density=True)
    with pytest.raises(QuESTError, match="different numbers of qubits"):
        gpu.qmxCircuitApply(q, c, 1)
    gpu.destroy(q)
    gpu.qmxCircuitDestroy(c)


@pytest.mark.gpu
@pytest.mark.parametrize("n,k", [(10, 5), (14, 5), (16, 5), (16, 3)])
def test_fused_brick_fp64_matches_oracle(gpu, cpuref, n, k):
    """Brick circuit with the 3-control and 5-target extras, fused into dense
    FP64 blocks (5-qubit blocks on the FP64 MFMA tiles from 11 qubits, kDense
    for 2-4 qubits and below 11), against the oracle's per-gate run."""
    gates = W.brick_circuit(n, 10, seed=40 + n, extra_every=5)
    qc = cpuref.qureg(n)
    W.apply_gates(cpuref, qc, gates)
    ref = cpuref.state(qc)
    cpuref.destroy(qc)
    c = W.build_circuit(gpu, n, gates)
    assert gpu.qmxCircuitFuse(c, k) < len(gates)
    q = gpu.qureg(n)
    gpu.qmxCircuitApply(q, c, 1)
    assert np.max(np.abs(gpu.state(q) - ref)) < TOL
    gpu.destroy(q)
    gpu.qmxCircuitDestroy(c)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [14, 18])
def test_fused_brick_fp32_mfma_matches_oracle(gpu, cpuref, n):
    """The same fused into 5-qubit MFMA blocks on FP32 amplitudes (kFused5):
    max-abs amplitude error <= 2e-6 and 1 - F <= 1e-6 against the oracle."""
    gates = W.brick_circuit(n, 10, seed=60 + n, extra_every=5)
    qc = cpuref.qureg(n)
    W.apply_gates(cpuref, qc, gates)
    ref = cpuref.state(qc)
    cpuref.destroy(qc)
    c = W.build_circuit(gpu, n, gates)
    gpu.qmxCircuitFuse(c, 5)
    q = gpu.qureg(n, precision=QMX_PREC_FP32)
    gpu.qmxCircuitApply(q, c, 1)
    got = gpu.state(q)
    assert np.max(np.abs(got - ref)) < 2e-6
    f = abs(np.vdot(ref, got)) ** 2 / (np.vdot(got, got).real * np.vdot(ref, ref).real)
    assert 1 - f < 1e-6
    gpu.destroy(q)
    gpu.qmxCircuitDestroy(c)


def _edge_gates(n, count, seed):
    """Brick and random gates with 2- to 4-control and 2- to 6-target ones where the
    register has the qubits: every form a tile, an LDS circuit or a lone kernel takes."""
    rng = np.random.default_rng(seed)
    gates = W.brick_circuit(n, 2, seed=seed, extra_every=2 if n >= 5 else 0)
    for i in range(count):
        qs = [int(x) for x in rng.permutation(n)]
        kind = i % 6
        if kind == 0 and n >= 3:
            c = min(n - 1, 2 + i % 3)
            gates.append(("mcu", qs[:c], qs[c], W.haar_unitary(rng, 2)))
        elif kind == 1 and n >= 2 and i % 24 == 1:
            k = min(n, 2 + (i // 24) % 5)
            gates.append(("mqu", qs[:k], W.haar_unitary(rng, 1 << k)))
        elif kind in (2, 3) and n >= 2:
            gates.append(("cnot", qs[0], qs[1]))
        elif kind == 4:
            gates.append(("rz", qs[0], float(rng.uniform(0, 6))))
        else:
            a = W.compact_pair(rng)
            gates.append(("cu", qs[0], *a))
    return gates


@pytest.mark.gpu
@pytest.mark.parametrize("n,count", [(1, 5), (2, 20), (3, 40), (6, 60), (9, 200), (11, 60), (12, 200),
                                     (13, 3), (13, 400), (14, 150), (17, 300), (20, 150)])
@pytest.mark.parametrize("precision", [None, QMX_PREC_FP32])
def test_circuits_at_the_edges_of_their_kernels(gpu, cpuref, n, count, precision):
    """A recorded circuit applied fused (twice: the prepared blocks serve every
    application) and unfused, where the register is one workgroup's (n <= 12), the
    smallest and larger tile sweeps, lists of one and of many sweeps."""
    gates = _edge_gates(n, count, 900 + n)
    qc = cpuref.qureg(n)
    for j in range(n):
        cpuref.lib.rotateY(qc, j, 0.3 + 0.1 * j)
    W.apply_gates(cpuref, qc, gates)
    once = cpuref.state(qc)
    W.apply_gates(cpuref, qc, gates)
    twice = cpuref.state(qc)
    cpuref.destroy(qc)
    # every gate is unitary: an amplitude's error is at most the sum of the gates'
    # roundings, a few ulps of an amplitude each (2^-53 or 2^-24)
    tol = 1e-12 if precision is None else 2.0 ** -22 * np.sqrt(2 * len(gates))
    for fused in (1, 0):
        c = W.build_circuit(gpu, n, gates)
        if fused:
            assert gpu.qmxCircuitFuse(c, 5) >= 1
        q = gpu.qureg(n, precision=precision)
        for j in range(n):
            gpu.lib.rotateY(q, j, 0.3 + 0.1 * j)
        for ref in (once, twice):
            gpu.qmxCircuitApply(q, c, fused)
            assert np.max(np.abs(gpu.state(q) - ref)) < tol
        gpu.destroy(q)
        gpu.qmxCircuitDestroy(c)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [2, 5, 12, 13, 15])
@pytest.mark.parametrize("fuse", [0, 5])
def test_operation_lists_with_collapses_between_sweeps(gpu, cpuref, n, fuse):
    """qmxApplyOperations on lists whose collapses cut the sweeps (and the LDS
    circuits), with noise and undispatched operations among them: state and
    probability as the oracle's loop."""
    rng = np.random.default_rng(n)
    ops = []
    for i in range(240):
        qs = [int(x) for x in rng.permutation(n)[:2]]
        code = int(rng.choice([O.H, O.X, O.Y, O.Z, O.P, O.RX, O.RY, O.RZ, O.CX, O.CY, O.CZ, O.CP, O.CRX, O.CRY, O.CRZ]))
        ops.append((code, qs if code >= O.CX else qs[:1], float(rng.uniform(0, 6))))
        if i in (60, 61, 150):
            ops.append((O.H, qs[:1], 0.0))
            ops.append((O.RY, qs[:1], 0.9))
            ops.append((O.CC, qs[:1], float(i & 1)))
        if i == 100:
            ops.append((O.NOISE_DEPHASING, qs[:1], 0.1))
            ops.append((O.PHASE, qs[:1], 0.2))  # accepted, not dispatched
    qc = cpuref.qureg(n)
    want = O.run_ops(cpuref, qc, [o for o in ops if o[0] != O.PHASE])
    ref = cpuref.state(qc)
    cpuref.destroy(qc)
    arr = (BasicOperation * len(ops))()
    for a, (code, qs, t) in zip(arr, ops):
        a.operation, a.numQubits, a.param = code, len(qs), t
        for j, x in enumerate(qs):
            a.qubits[j] = x
    q = gpu.qureg(n)
    got = gpu.qmxApplyOperations(q, arr, len(ops), None, fuse)
    assert abs(got - want) < TOL
    assert np.max(np.abs(gpu.state(q) - ref)) < TOL
    gpu.destroy(q)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 2, 3, 5, 6, 7, 8, 10])
@pytest.mark.parametrize("precision", [None, QMX_PREC_FP32])
@pytest.mark.parametrize("after", [None, dict(damping=0.03, dephasing=0.02, depolarising=0.01),
                                   dict(mixPauli=0.02)])
def test_density_lists_match_oracle(gpu, cpuref, n, precision, after):
    """qmxApplyOperations on density registers at the edges of its two forms (the
    register in one workgroup's LDS up to 5 or 6 qubits, tile sweeps of the rows and
    columns above): every gate, every one-qubit channel and a collapse, from a state
    that is not symmetric between rows and columns."""
    rng = np.random.default_rng(40 + n)
    one = [O.H, O.X, O.Y, O.Z, O.P, O.RX, O.RY, O.RZ]
    two = [O.CX, O.CY, O.CZ, O.CP, O.CRX, O.CRY, O.CRZ]
    channels = [O.NOISE_DAMPING, O.NOISE_DEPHASING, O.NOISE_DEPOLARISING, O.NOISE_MIX_X, O.NOISE_MIX_Y,
                O.NOISE_MIX_Z, O.NOISE_MIX_ALL]
    ops = []
    for i in range(60):
        qs = [int(x) for x in rng.permutation(n)[:2]]
        code = int(rng.choice(one + two if n > 1 else one))
        ops.append((code, qs if code in two else qs[:1], float(rng.uniform(0, 6))))
        if i % 3 == 0:
            ops.append((int(rng.choice(channels)), qs[:1], float(rng.uniform(0, 0.2))))
        if i == 40:
            ops += [(O.RY, qs[:1], 0.9), (O.CC, qs[:1], 0.0)]

    def start(lib, q):
        lib.initPlusState(q)
        for j in range(n):
            lib.rotateZ(q, j, 0.4 + 0.2 * j)

    qc = cpuref.qureg(n, density=True)
    start(cpuref, qc)
    ops = resolve_collapses(cpuref, qc, [(c, q, -1.0 if c == O.CC else t) for c, q, t in ops], after)
    ref = cpuref.state(qc)
    cpuref.destroy(qc)
    arr = (BasicOperation * len(ops))()
    for a, (code, qs, t) in zip(arr, ops):
        a.operation, a.numQubits, a.param = code, len(qs), t
        for j, x in enumerate(qs):
            a.qubits[j] = x
    noise = C.byref(NoiseAfterGate(**after)) if after else None
    # entries are at most 1 and no operation enlarges an error by more than the
    # collapse's 1/p <= 2: a few ulps an operation
    tol = TOL if precision is None else 2.0 ** -21 * np.sqrt(len(ops))
    for fuse in (0, 5):
        q = gpu.qureg(n, density=True, precision=precision)
        start(gpu, q)
        gpu.qmxApplyOperations(q, arr, len(ops), noise, fuse)
        assert np.max(np.abs(gpu.state(q) - ref)) < tol
        gpu.destroy(q)


def _operation_array(ops):
    arr = (BasicOperation * len(ops))()
    for a, (code, qs, t) in zip(arr, ops):
        a.operation, a.numQubits, a.param = code, len(qs), t
        for j, x in enumerate(qs):
            a.qubits[j] = x
    return arr


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 2, 6])
def test_repeated_noise_does_not_drift(gpu, n):
    """The same three channels after each of 2000 bit flips (exact permutations), on
    registers of one workgroup's LDS and of tile sweeps, against 80-bit arithmetic. The
    channels' product is made once: rounded to FP64, its error is the same in every
    channel and the trace drifts (1.1e-16 a channel where the qubit is 1, 1e-13 in all).
    What rounds entry by entry walks: about twice 2^-53 an operation, in random
    directions."""
    damping, dephasing, depolarising = 0.007, 0.003, 0.012
    ops = [(O.X, [i % n], 0.0) for i in range(2000)]
    q = gpu.qureg(n, density=True)
    gpu.lib.initPlusState(q)
    for j in range(n):
        gpu.lib.rotateY(q, j, 0.4 + 0.2 * j)
    rho = gpu.state(q).astype(np.clongdouble)
    gpu.qmxApplyOperations(q, _operation_array(ops), len(ops),
                           C.byref(NoiseAfterGate(damping=damping, dephasing=dephasing, depolarising=depolarising)), 5)
    got = gpu.state(q)
    gpu.destroy(q)
    exact = np.longdouble  # of the channels' FP64 numbers
    level = 4 * depolarising / 3.0
    h, keep = exact(level / 2), exact(1 - level / 2)
    f = exact(np.sqrt(1 - damping)) * exact(1 - 2 * dephasing) * exact(1 - level)
    for _, (t,), _ in ops:
        v = rho.reshape(-1, 2, 1 << (n - 1), 2, 1 << t)
        x11, x10, x01, x00 = (v[:, i, :, j].copy() for i in (0, 1) for j in (0, 1))
        x00, x11 = x00 + exact(damping) * x11, exact(1 - damping) * x11
        v[:, 0, :, 0], v[:, 1, :, 1] = keep * x00 + h * x11, h * x00 + keep * x11
        v[:, 0, :, 1], v[:, 1, :, 0] = f * x01, f * x10
    err = float(np.sqrt(np.sum(np.abs(got - rho) ** 2) / np.sum(np.abs(rho) ** 2)))
    assert err < 4 * 2.0 ** -53 * np.sqrt(len(ops))


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 3, 4, 5, 8, 9, 10, 11, 12])
@pytest.mark.parametrize("precision", [None, QMX_PREC_FP32])
def test_small_registers_in_blocks(gpu, cpuref, n, precision):
    """Fused circuits on registers of one workgroup's LDS: 4-qubit blocks, 5-qubit ones
    (of which tiles of 9 to 11 bits have fewer chunks than waves), more than 64 in a
    sweep, collapses and a gate too wide for a block between sweeps; applied twice."""
    rng = np.random.default_rng(50 + n)
    gates = W.brick_circuit(n, 12, seed=n, extra_every=4 if n >= 6 else 0) if n > 1 else []
    for i in range(100):
        qs = [int(x) for x in rng.permutation(n)]
        if n >= 5 and i % 5 == 0:
            gates.append(("mqu", qs[:5], W.haar_unitary(rng, 32)))
        elif n >= 2 and i % 3 == 0:
            gates.append(("cnot", qs[0], qs[1]))
        else:
            gates.append(("cu", qs[0], *W.compact_pair(rng)))
    if n >= 6:
        gates.insert(40, ("mcu", qs[:5], qs[5], W.haar_unitary(rng, 2)))
    c = W.build_circuit(gpu, n, gates)
    gpu.qmxCircuitAddOperation(c, O.CC, ints([0]), 1, 1.0)
    gpu.qmxCircuitAddOperation(c, O.H, ints([0]), 1, 0.0)
    assert gpu.qmxCircuitFuse(c, 5) >= 1
    q, qc = gpu.qureg(n, precision=precision), cpuref.qureg(n)
    for lib, r in ((gpu, q), (cpuref, qc)):
        for j in range(n):
            lib.lib.rotateY(r, j, 0.3 + 0.1 * j)
    # FP32: each launch (4 an application) and the n rotations round an amplitude once, by
    # 2^-24; a collapse divides what came before by the root of its probability (> 0.05)
    tol = 1e-12 if precision is None else 2.0 ** -24 * (n + 8) / 0.05
    for _ in range(2):
        W.apply_gates(cpuref, qc, gates)
        want = cpuref.call("collapseToOutcome", qc, 0, 1)
        cpuref.call("hadamard", qc, 0)
        got = gpu.qmxCircuitApply(q, c, 1)
        assert want > 0.05 and abs(got - want) < tol
        assert np.max(np.abs(gpu.state(q) - cpuref.state(qc))) < tol
    gpu.destroy(q)
    cpuref.destroy(qc)
    gpu.qmxCircuitDestroy(c)


@pytest.mark.gpu
@pytest.mark.parametrize("count", [32, 33, 400])
@pytest.mark.parametrize("precision", [None, QMX_PREC_FP32])
def test_long_lists_on_two_qubits(gpu, cpuref, count, precision):
    """Runs of more than 32 gates (none joined: two-qubit ones between one-qubit ones)
    become one matrix each; a collapse ends a run."""
    rng = np.random.default_rng(count)
    two = [O.CX, O.CY, O.CZ, O.CP, O.CRX, O.CRY, O.CRZ]
    run = []
    for i in range(count):
        a = int(rng.integers(2))
        run.append((int(rng.choice(two)), [a, 1 - a], float(rng.uniform(0, 6))) if i % 2 else
                   (int(rng.choice([O.H, O.X, O.Y, O.P, O.RX, O.RY, O.RZ])), [a], float(rng.uniform(0, 6))))
    ops = run + [(O.CC, [0], 1.0), (O.H, [0], 0.0)] + run
    qc = cpuref.qureg(2)
    cpuref.lib.rotateY(qc, 0, 0.4)
    cpuref.lib.rotateX(qc, 1, 1.1)
    want = O.run_ops(cpuref, qc, ops)
    ref = cpuref.state(qc)
    cpuref.destroy(qc)
    assert want > 0.04
    # each run and each operation beside it rounds an amplitude once by 2^-24
    tol = TOL if precision is None else 2.0 ** -24 * 8 / 0.04
    q = gpu.qureg(2, precision=precision)
    gpu.lib.rotateY(q, 0, 0.4)
    gpu.lib.rotateX(q, 1, 1.1)
    got = gpu.qmxApplyOperations(q, _operation_array(ops), len(ops), None, 2)
    assert abs(got - want) < tol
    assert np.max(np.abs(gpu.state(q) - ref)) < tol
    gpu.destroy(q)


@pytest.mark.gpu
@pytest.mark.parametrize("n,k", [(13, 6), (14, 7), (16, 6)])
def test_five_qubit_blocks_of_wider_circuits(gpu, cpuref, n, k):
    """FP32 circuits fused into blocks of more than 5 qubits keep the device form of the
    blocks that have exactly 5: applied twice, fused again, applied again."""
    gates = _edge_gates(n, 60, 70 + n)
    qc = cpuref.qureg(n)
    c = W.build_circuit(gpu, n, gates)
    q = gpu.qureg(n, precision=QMX_PREC_FP32)
    for lib, r in ((gpu, q), (cpuref, qc)):
        for j in range(n):
            lib.lib.rotateY(r, j, 0.3 + 0.1 * j)
    sizes = []
    for i in range(3):
        if i != 1:
            blocks = gpu.qmxCircuitFuse(c, k)
            sizes = [gpu.qmxCircuitStep(c, s, None, None, None) for s in range(blocks)]
        assert 5 in sizes
        W.apply_gates(cpuref, qc, gates)
        gpu.qmxCircuitApply(q, c, 1)
        # as in test_circuits_at_the_edges_of_their_kernels, for i + 1 applications
        assert np.max(np.abs(gpu.state(q) - cpuref.state(qc))) < 2.0 ** -22 * np.sqrt((i + 1) * len(gates))
    gpu.destroy(q)
    cpuref.destroy(qc)
    gpu.qmxCircuitDestroy(c)


@pytest.mark.gpu
@pytest.mark.parametrize("precision,most", [(None, 7), (QMX_PREC_FP32, 4)])
def test_a_planned_circuit_holds_its_blocks_only(gpu, precision, most):
    """Device memory that a circuit's first application takes and keeps: a 4-qubit block's
    vectors are 4 KiB in FP32 and 7 in FP64 and its description 20 bytes; the gates are
    needed while the blocks are built. 2000 blocks and more, and two allocations' slack."""
    with open("/proc/self/maps") as f:  # the HIP runtime that the library runs on
        hip = C.CDLL(next(line.split()[-1] for line in f if "libamdhip64" in line))

    def free():
        gpu.qmxSync()
        f, total = C.c_size_t(), C.c_size_t()
        assert hip.hipMemGetInfo(C.byref(f), C.byref(total)) == 0
        return f.value

    n = 14
    rng = np.random.default_rng(14)
    gates = []
    for i in range(9000):
        qs = [int(x) for x in rng.choice(n, 2, replace=False)]
        gates += [("cnot", qs[0], qs[1]), ("cu", qs[0], *W.compact_pair(rng))]
    c = W.build_circuit(gpu, n, gates)
    gpu.qmxCircuitFuse(c, 5)
    small = large = sweep = 0
    while True:
        k = gpu.lib.qmxCircuitSweepBlock(c, 0 if precision is None else 1, sweep, 0, None, None, None)
        if k < 0:
            break
        block = 0
        while k > 0:
            small, large, block = small + (k <= 4), large + (k == 5), block + 1
            k = gpu.lib.qmxCircuitSweepBlock(c, 0 if precision is None else 1, sweep, block, None, None, None)
        sweep += 1
    assert small > 2000
    q = gpu.qureg(n, precision=precision)
    gpu.lib.hadamard(q, 0)
    before = free()
    gpu.qmxCircuitApply(q, c, 1)
    kept = before - free()
    gpu.destroy(q)
    gpu.qmxCircuitDestroy(c)
    assert kept <= small * (most * 1024 + 20) + large * (26 * 1024 + 20) + 2 * (4 << 20)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [2, 10])
def test_noise_does_not_cut_a_state_vectors_list(gpu, n):
    """Noise is ignored on state vectors: an unfused circuit with noise after every gate
    gives the bits of the circuit without it (FP32 is rounded once a launch, so a list
    that noise cuts into launches gives others)."""
    rng = np.random.default_rng(n)
    states = []
    gates = [(O.RY if i % 2 else O.RX, int(rng.integers(n)), float(rng.uniform(0, 6))) for i in range(60)]
    for noisy in (False, True):
        c = gpu.qmxCircuitCreate(n)
        for code, target, angle in gates:
            gpu.qmxCircuitAddOperation(c, code, ints([target]), 1, angle)
            if noisy:
                gpu.qmxCircuitAddOperation(c, O.NOISE_DAMPING, ints([target]), 1, 0.1)
        q = gpu.qureg(n, precision=QMX_PREC_FP32)
        gpu.qmxCircuitApply(q, c, 0)
        states.append(gpu.state(q))
        gpu.destroy(q)
        gpu.qmxCircuitDestroy(c)
    assert np.array_equal(states[0], states[1])


@pytest.mark.gpu
@pytest.mark.parametrize("n", [3, 13])
@pytest.mark.parametrize("fuse", [0, 3, 5])
def test_undispatched_operations_say_so(gpu, capfd, n, fuse):
    """Lists of operations that QuantumLab's loop does not dispatch report each of them,
    fused or not (QLGate.cpp:652-803); among gates that are fused they are passed over."""
    libc = C.CDLL(None)
    q = gpu.qureg(n)
    for ops, said in (([(O.PHASE, [0], 0.2), (O.PHASE, [1], 0.3)], 2),
                      ([(O.H, [0], 0.0), (O.PHASE, [0], 0.2)], 0 if fuse else 1)):
        libc.fflush(None)
        capfd.readouterr()
        assert gpu.qmxApplyOperations(q, _operation_array(ops), len(ops), None, fuse) == 1.0
        libc.fflush(None)
        assert capfd.readouterr().out.count("not supported type!") == said
    gpu.destroy(q)


@pytest.mark.gpu
@pytest.mark.parametrize("n,precision", [(21, None), (25, None), (22, QMX_PREC_FP32), (26, QMX_PREC_FP32)])
def test_tile_sweeps_of_large_registers(gpu, n, precision):
    """The tile kernel's forms for registers that fill the CUs with four-wave workgroups:
    the smallest such register, and the smallest that outgrows the last-level cache (whose
    accesses are nontemporal); a recorded circuit against its gates one by one."""
    gates = W.brick_circuit(n, 4, seed=n, extra_every=2)
    a, b = gpu.qureg(n, precision=precision), gpu.qureg(n, precision=precision)
    for q in (a, b):
        for j in range(n):
            gpu.lib.rotateY(q, j, 0.9 + 0.05 * j)
            gpu.lib.rotateZ(q, j, 0.2 * j)
    c = W.build_circuit(gpu, n, gates)
    gpu.qmxCircuitFuse(c, 5)
    gpu.qmxCircuitApply(a, c, 1)
    W.apply_gates(gpu, b, gates)
    # as in test_circuits_at_the_edges_of_their_kernels, for the two paths
    assert gpu.lib.qmxMaxAbsDiff(a, b) < (1e-12 if precision is None else 2.0 ** -22 * np.sqrt(2 * len(gates)))
    assert abs(gpu.calcTotalProb(a) - 1) < (1e-12 if precision is None else 2.0 ** -22 * np.sqrt(2 * len(gates)))
    gpu.destroy(a)
    gpu.destroy(b)
    gpu.qmxCircuitDestroy(c)


def _mixed_ops(rng, n, count, qubits=None):
    pool = np.arange(n) if qubits is None else np.array(qubits)
    ops = []
    for i in range(count):
        qs = [int(x) for x in rng.choice(pool, 2, replace=False)]
        two = i % 3 == 2
        code = int(rng.choice([O.CX, O.CY, O.CZ, O.CP, O.CRX, O.CRY, O.CRZ] if two else
                              [O.H, O.X, O.Y, O.Z, O.P, O.RX, O.RY, O.RZ]))
        ops.append((code, qs if two else qs[:1], float(rng.uniform(0, 6))))
    return ops


@pytest.mark.gpu
@pytest.mark.parametrize("n,precision", [(11, None), (13, None), (12, QMX_PREC_FP32), (13, QMX_PREC_FP32)])
def test_density_lists_of_large_registers(gpu, n, precision):
    """The same kernel forms on density registers (22 to 26 row and column bits): a list
    with noise against the recorded circuit, which composes superoperators call by call."""
    ops = _mixed_ops(np.random.default_rng(n), n, 40)
    noise = NoiseAfterGate(damping=0.01, dephasing=0.02, depolarising=0.015)
    c = gpu.qmxCircuitCreate(n)
    for code, qs, t in ops:
        gpu.qmxCircuitAddOperation(c, code, ints(qs), len(qs), t)
    gpu.qmxCircuitSetNoiseAfterGate(c, noise)
    a, b = gpu.qureg(n, density=True, precision=precision), gpu.qureg(n, density=True, precision=precision)
    for q in (a, b):
        gpu.lib.initPlusState(q)
        for j in range(n):
            gpu.lib.rotateX(q, j, 0.3 + 0.1 * j)
    gpu.qmxApplyOperations(a, _operation_array(ops), len(ops), C.byref(noise), 5)
    gpu.qmxCircuitApply(b, c, 0)
    gpu.qmxCircuitDestroy(c)
    # as in test_density_lists_match_oracle, whose entries reach 1 where these are near 2^-n
    assert gpu.lib.qmxMaxAbsDiff(a, b) < (TOL if precision is None else 2.0 ** -21 * np.sqrt(len(ops))) * 1e-2
    assert abs(gpu.calcTotalProb(a) - 1) < (TOL if precision is None else 2.0 ** -21 * np.sqrt(len(ops)))
    gpu.destroy(a)
    gpu.destroy(b)


@pytest.mark.gpu
@pytest.mark.parametrize("n,count,qubits,fuse", [
    (13, 9000, None, 5),                  # more blocks than a batch of the workspace holds (256)
    (13, 2000, [0, 5, 8, 12], 5),         # one set of 4 qubits: more gates than a block may hold (512) or stages at a time (64)
    (10, 12000, None, 5), (3, 12000, None, 0)])  # more gates than a launch takes (4096 after joins)
@pytest.mark.parametrize("precision", [None, QMX_PREC_FP32])
def test_lists_longer_than_a_launch(gpu, cpuref, n, count, qubits, fuse, precision):
    ops = _mixed_ops(np.random.default_rng(n + count), n, count, qubits)
    qc = cpuref.qureg(n)
    O.run_ops(cpuref, qc, ops)
    ref = cpuref.state(qc)
    cpuref.destroy(qc)
    # every operation rounds an amplitude by a few ulps, in random directions
    tol = 2.0 ** -51 * np.sqrt(count) * 8 if precision is None else 2.0 ** -22 * np.sqrt(count)
    q = gpu.qureg(n, precision=precision)
    gpu.qmxApplyOperations(q, _operation_array(ops), len(ops), None, fuse)
    assert np.max(np.abs(gpu.state(q) - ref)) < tol
    gpu.destroy(q)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [12, 13])
@pytest.mark.parametrize("precision", [None, QMX_PREC_FP32])
def test_recorded_circuits_of_many_blocks(gpu, cpuref, n, precision):
    """More blocks than are built at a time (256), some with matrices of their own, in one
    sweep on 12 qubits and in many on 13."""
    rng = np.random.default_rng(n)
    gates = []
    for i in range(2400):
        qs = [int(x) for x in rng.permutation(n)]
        if i % 50 == 0:
            gates.append(("mqu", qs[:5], W.haar_unitary(rng, 32)))
        elif i % 3:
            gates.append(("cu", qs[0], *W.compact_pair(rng)))
        else:
            gates.append(("cnot", qs[0], qs[1]))
    c = W.build_circuit(gpu, n, gates)
    gpu.qmxCircuitFuse(c, 5)
    q, qc = gpu.qureg(n, precision=precision), cpuref.qureg(n)
    W.apply_gates(cpuref, qc, gates)
    gpu.qmxCircuitApply(q, c, 1)
    tol = 1e-12 if precision is None else 2.0 ** -22 * np.sqrt(2 * len(gates))
    assert np.max(np.abs(gpu.state(q) - cpuref.state(qc))) < tol
    gpu.destroy(q)
    cpuref.destroy(qc)
    gpu.qmxCircuitDestroy(c)
