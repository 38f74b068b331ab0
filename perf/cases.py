"""The workloads this library is timed on.

Each case is work that a user's program hands to the library in one piece:

  ops      QuantumLab's simulators: a list of SBasicOperations applied to a state
           vector in one call (qmxApplyOperations), then the outcome
           probabilities of a few qubits;
  gates    QuEST's C API called gate by gate (the brick circuit);
  circuit  a circuit recorded and fused once and applied to a register
           (qmxCircuitApply), as simulators of large registers do;
  density  the density-matrix simulator: an operation list with noise after
           every gate, then purity and the P(0) of every qubit;
  trotter  Hamiltonian simulation, applyTrotterCircuit on the chain family;
  kmeans   quantum k-means: swap tests of all points against all centroids,
           assignments and new centroids, a few iterations from given centroids.

Sizes run from registers of a few qubits, where a call's latency counts, to
registers of several GiB. States are returned as views of the registers' device
buffers.
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

import quantumlab_amd
from quantumlab_amd import hamiltonians as H
from quantumlab_amd import qkmeans as K
from quantumlab_amd import workloads as W

FP64, FP32 = 0, 1


def listed():
    return [
        # a small application circuit (QuantumLab's default float build): latency of one call
        {"name": "ops_f32_10", "kind": "ops", "qubits": 10, "count": 80, "precision": "f32", "fuse": 5},
        # an ordinary simulator run, double precision, ragged size
        {"name": "ops_f64_17", "kind": "ops", "qubits": 17, "count": 300, "precision": "f64", "fuse": 5},
        # QuEST callers, one API call per gate: a register that the caches hold
        {"name": "gates_f64_20", "kind": "gates", "qubits": 20, "layers": 3, "precision": "f64"},
        # the same at 8 GiB, where every gate streams the register
        {"name": "gates_f64_29", "kind": "gates", "qubits": 29, "layers": 5, "precision": "f64"},
        # recorded circuits: a cache-sized register, and large ones in both precisions
        {"name": "circuit_f32_21", "kind": "circuit", "qubits": 21, "layers": 5, "precision": "f32"},
        {"name": "circuit_f64_27", "kind": "circuit", "qubits": 27, "layers": 5, "precision": "f64"},
        {"name": "circuit_f32_30", "kind": "circuit", "qubits": 30, "layers": 5, "precision": "f32"},
        # the noisy swap-test job's register size, and a large density matrix
        {"name": "density_f64_7", "kind": "density", "qubits": 7, "count": 60, "precision": "f64"},
        {"name": "density_f32_13", "kind": "density", "qubits": 13, "count": 120, "precision": "f32"},
        # Hamiltonian simulation: the 24-qubit instances, and a smaller FP64 register
        {"name": "trotter_f32_24", "kind": "trotter", "qubits": 24, "order": 2, "reps": 8, "precision": "f32"},
        {"name": "trotter_f64_19", "kind": "trotter", "qubits": 19, "order": 4, "reps": 2, "precision": "f64"},
        # k-means on points of uneven size
        {"name": "kmeans_f32_4096", "kind": "kmeans", "points": 4096, "clusters": 16, "q_lo": 4, "q_hi": 10,
         "iterations": 5, "precision": "f32"},
    ]


def draw(rng):
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["ops", "gates", "circuit", "density", "trotter", "kmeans"])
    prec = rng.choice(["f32", "f64"])
    if kind == "ops":
        return {"kind": kind, "qubits": rng.randint(3, 22), "count": log(20, 400), "precision": prec,
                "fuse": rng.choice([0, 5, 5])}
    if kind == "gates":
        return {"kind": kind, "qubits": rng.randint(6, 28), "layers": rng.randint(1, 5), "precision": prec}
    if kind == "circuit":
        return {"kind": kind, "qubits": rng.randint(9, 29), "layers": rng.randint(1, 6), "precision": prec}
    if kind == "density":
        return {"kind": kind, "qubits": rng.randint(2, 13), "count": log(20, 150), "precision": prec}
    if kind == "trotter":
        order = rng.choice([1, 2, 4])
        reps = log(1, 40 if order == 1 else 20 if order == 2 else 4)
        return {"kind": kind, "qubits": rng.randint(6, 25), "order": order, "reps": reps, "precision": prec}
    lo = rng.randint(3, 6)
    return {"kind": kind, "points": log(100, 6000), "clusters": log(2, 24), "q_lo": lo,
            "q_hi": rng.randint(lo, 10), "iterations": rng.randint(1, 6), "precision": prec}


# ---- inputs ---------------------------------------------------------------------

_LIBS = {}


def _library(flavour):
    if flavour not in _LIBS:
        _LIBS[flavour] = quantumlab_amd.load(flavour=flavour)
    return _LIBS[flavour]


class Register:
    """A register and a view of its device amplitudes, (2^n, 2) reals."""

    def __init__(self, qe, n, precision, density=False):
        self.qe = qe
        self.q = qe.qureg(n, density=density, precision=precision)
        ptr = C.cast(self.q.deviceStateVec.real, C.c_void_p).value
        self.__cuda_array_interface__ = {"shape": (int(self.q.numAmpsTotal), 2), "version": 3, "strides": None,
                                         "typestr": "<f8" if precision == FP64 else "<f4", "data": (ptr, False)}

    def view(self):
        return torch.as_tensor(self, device="cuda")

    def __del__(self):
        self.qe.destroy(self.q)


def _precision(case):
    return FP64 if case["precision"] == "f64" else FP32


def _seeded(case, seed):
    return np.random.default_rng([seed, case["qubits"]])


def _angles(case, seed):
    """RY and RZ angles of a product state: what the register holds before the pass."""
    rng = np.random.default_rng([seed, case["qubits"], 5])
    return rng.uniform(0, np.pi, case["qubits"]), rng.uniform(0, 2 * np.pi, case["qubits"])


# QuantumLab's operation codes (EBasicOperation)
_SINGLE = {"H": 0, "X": 1, "Y": 2, "Z": 3, "P": 4, "RX": 6, "RY": 7, "RZ": 8}
_DOUBLE = {"CX": 9, "CY": 10, "CZ": 11, "CP": 12, "CRX": 13, "CRY": 14, "CRZ": 15}


def operations(case, seed):
    """A seeded list of basic operations: (name, qubits, angle). Two thirds act on
    one qubit (rotations more often than Paulis), the rest on two, three in four
    of them neighbours."""
    rng, n = _seeded(case, seed), case["qubits"]
    out = []
    for _ in range(case["count"]):
        t = float(rng.uniform(0, 2 * np.pi))
        if case["precision"] == "f32":
            t = float(np.float32(t))
        if n == 1 or rng.random() < 2 / 3:
            name = str(rng.choice(["H", "H", "X", "Y", "Z", "P", "RX", "RY", "RZ", "RY", "RZ"]))
            out.append((name, (int(rng.integers(n)),), t))
            continue
        name = str(rng.choice(["CX", "CX", "CX", "CY", "CZ", "CP", "CRX", "CRY", "CRZ"]))
        if rng.random() < 0.75:
            a = int(rng.integers(n - 1))
            pair = (a, a + 1) if rng.random() < 0.5 else (a + 1, a)
        else:
            pair = tuple(int(x) for x in rng.choice(n, size=2, replace=False))
        out.append((name, pair, t))
    return out


def _noise(case, seed):
    """Damping, dephasing and depolarising rates after every gate."""
    r = np.random.default_rng([seed, 77]).uniform(0.002, 0.02, 3)
    return tuple(float(np.float32(x)) for x in r)


def _operation_array(qe, ops):
    arr = (qe.t.BasicOperation * len(ops))()
    for o, (name, qubits, t) in zip(arr, ops):
        o.operation = _SINGLE.get(name, _DOUBLE.get(name))
        o.numQubits = len(qubits)
        for j, q in enumerate(qubits):
            o.qubits[j] = q
        o.param = t
    return arr


def _product_state(qe, q, case, seed):
    qe.lib.initZeroState(q)
    theta, phi = _angles(case, seed)
    for j in range(case["qubits"]):
        qe.lib.rotateY(q, j, float(theta[j]))
        qe.lib.rotateZ(q, j, float(phi[j]))


def _brick(case, seed):
    return W.brick_circuit(case["qubits"], case["layers"], seed, extra_every=case["layers"])


def _dataset(case, seed):
    return K.make_dataset(case["points"], case["clusters"], case["q_lo"], case["q_hi"], seed=seed)


def _hamiltonian(case, seed):
    return H.trotter_instance(case["qubits"], seed, 0)


def prepare(case, seed):
    kind, n = case["kind"], case.get("qubits")
    s = {"kind": kind}
    if kind in ("ops", "density"):
        # these callers use the library of their own real type
        qe = _library(case["precision"])
        reg = Register(qe, n, _precision(case), density=kind == "density")
        ops = operations(case, seed)
        s.update(qe=qe, reg=reg, ops=_operation_array(qe, ops), count=len(ops))
        if kind == "ops":
            k = min(n, 6)
            s.update(noise=None, fuse=case["fuse"], qubits=(C.c_int * k)(*range(k)), k=k,
                     probs=(qe.t.qreal * (1 << k))())
        else:
            s.update(noise=qe.t.NoiseAfterGate(*_noise(case, seed), 0, 0, 0), n=n)
    else:
        qe = s["qe"] = _library("f64")
    if kind in ("gates", "circuit", "trotter"):
        reg = s["reg"] = Register(qe, n, _precision(case))
    if kind == "gates":
        s["calls"], s["keep"] = _calls(qe, reg.q, _brick(case, seed))
    elif kind == "circuit":
        s["circuit"] = Circuit(qe, n, _brick(case, seed))
    elif kind == "trotter":
        s["inst"] = _hamiltonian(case, seed)
        s["batch"] = H.HamilBatch([s["inst"]])
        s["steps"] = (float(s["inst"].time), case["order"], case["reps"])
    elif kind == "kmeans":
        data = _dataset(case, seed)
        s["plan"] = K.SwapPlan(qe, data, _precision(case))
        s["plan"].autotune()
        s["init"], s["iterations"] = data.init, case["iterations"]
    if kind != "kmeans":
        _product_state(qe, reg.q, case, seed)
        qe.lib.qmxSync()
        s["state"] = reg.view()
    return s


class Circuit:
    """A recorded circuit, fused into blocks of at most five qubits."""

    def __init__(self, qe, n, gates):
        self.qe, self.c = qe, W.build_circuit(qe, n, gates)
        qe.call("qmxCircuitFuse", self.c, 5)

    def __del__(self):
        self.qe.lib.qmxCircuitDestroy(self.c)


def _calls(qe, q, gates):
    """The gate list as (function, arguments) of the C API."""
    lib, out, keep = qe.lib, [], []
    for g in gates:
        if g[0] == "cu":
            out.append((lib.compactUnitary, (q, g[1], qe.t.cplx(g[2]), qe.t.cplx(g[3]))))
        elif g[0] == "cnot":
            out.append((lib.controlledNot, (q, g[1], g[2])))
        elif g[0] == "rz":
            out.append((lib.rotateZ, (q, g[1], g[2])))
        elif g[0] == "mcu":
            out.append((lib.multiControlledUnitary, (q, (C.c_int * len(g[1]))(*g[1]), len(g[1]), g[2],
                                                     qe.t.matrix2(g[3]))))
        else:
            m = qe.matrixN(g[2])
            keep.append(m)
            out.append((lib.multiQubitUnitary, (q, (C.c_int * len(g[1]))(*g[1]), len(g[1]), m)))
    return out, keep


# ---- one pass -------------------------------------------------------------------

def run(s):
    kind, qe = s["kind"], s["qe"]
    if kind == "kmeans":
        plan = s["plan"]
        plan.set_centroids(s["init"])
        plan.run(s["iterations"])
        return {"p0": plan.p0(), "assignments": plan.assignments(), "centroids": plan.centroids()}
    lib, q = qe.lib, s["reg"].q
    if kind == "ops":
        prob = lib.qmxApplyOperations(q, s["ops"], s["count"], s["noise"], s["fuse"])
        lib.calcProbOfAllOutcomes(s["probs"], q, s["qubits"], s["k"])
        qe.check()
        return {"prob": np.float64(prob), "probs": np.array(s["probs"]), "state": s["state"]}
    if kind == "density":
        lib.qmxApplyOperations(q, s["ops"], s["count"], s["noise"], 5)
        purity = lib.calcPurity(q)
        zeros = np.array([lib.calcProbOfOutcome(q, j, 0) for j in range(s["n"])])
        qe.check()
        return {"purity": np.float64(purity), "zeros": zeros, "state": s["state"]}
    if kind == "gates":
        for fn, args in s["calls"]:
            fn(*args)
    elif kind == "circuit":
        lib.qmxCircuitApply(q, s["circuit"].c, 1)
    else:
        time, order, reps = s["steps"]
        lib.applyTrotterCircuit(q, s["batch"][0], time, order, reps)
    qe.check()
    return {"state": s["state"]}


# ---- what a pass cannot do without ----------------------------------------------

def _gate_flops(gates, amps):
    """Real operations of a gate list applied gate by gate: 14 an amplitude for a
    2x2, 8 2^k for a 2^k x 2^k, a 2^c-th of that with c controls, none for CNOTs."""
    f = 0.0
    for g in gates:
        if g[0] == "cu":
            f += 14.0 * amps
        elif g[0] == "rz":
            f += 6.0 * amps
        elif g[0] == "mcu":
            f += 14.0 * amps / (1 << len(g[1]))
        elif g[0] == "mqu":
            f += 8.0 * (1 << len(g[1])) * amps
    return f


def _op_flops(name, amps):
    name, share = (name[1:], 0.5) if name[0] == "C" else (name, 1.0)
    return share * amps * {"X": 0, "Y": 1, "Z": 0.5, "P": 3, "RZ": 6, "H": 4}.get(name, 14)


def work(case):
    size = 16 if case["precision"] == "f64" else 8
    kind = case["kind"]
    if kind == "kmeans":
        # points once, P0 out; one multiply-add for each coordinate, centroid and iteration
        mean = np.mean([2.0 ** q for q in range(case["q_lo"], case["q_hi"] + 1)])
        return {"bytes": case["points"] * (8 * mean + 8 * case["clusters"]),
                "flops": 2 * mean * case["points"] * case["clusters"] * case["iterations"]}
    amps = float(1 << (case["qubits"] * (2 if kind == "density" else 1)))
    if kind in ("gates", "circuit"):
        return {"bytes": 2 * amps * size, "flops": _gate_flops(_brick(case, 1), amps)}
    if kind == "trotter":
        terms = _hamiltonian(case, 1).terms
        return {"bytes": 2 * amps * size, "flops": 6 * amps * terms * H.stages(case["order"]) * case["reps"]}
    ops = operations(case, 1)
    if kind == "ops":
        return {"bytes": 2 * amps * size, "flops": sum(_op_flops(o[0], amps) for o in ops)}
    # a gate acts on rows and columns; each of its qubits meets three channels
    return {"bytes": 2 * amps * size, "flops": sum(2 * _op_flops(o[0], amps) + 9 * amps * len(o[1]) for o in ops)}


# About four times the largest difference from exact() seen over these ranges:
# amplitudes and their arithmetic in the register's own precision, gate after
# gate (rel 6e-7 and max 2e-5 in FP32, 1e-14 and 4e-14 in FP64; 3e-6 for the
# hundreds of rotations of an FP32 Trotter circuit, whose rounding repeats);
# k-means registers rounded once to FP32 (5e-8, 2e-7), sums in FP64.
def tolerance(case):
    single = case["precision"] == "f32"
    if case["kind"] == "kmeans":
        return {"rel": 2e-7, "max": 1e-6, "differ": 0.002} if single else {"rel": 2e-15, "max": 1e-14, "differ": 0.002}
    if not single:
        return {"rel": 5e-14, "max": 2e-13}
    return {"rel": 1.2e-5 if case["kind"] == "trotter" else 3e-6, "max": 1.2e-4}


# ---- the same in 64 bits --------------------------------------------------------

def _on(psi, target):
    return psi.view(-1, 2, 1 << target)


def _m2(psi, target, u, control=None):
    """A 2x2 on `target`, where the control qubit (if any) is 1; in place."""
    if control is None:
        v = _on(psi, target)
        a, b = v[:, 0].clone(), v[:, 1]
        v[:, 0] = u[0][0] * a + u[0][1] * b
        v[:, 1] = u[1][0] * a + u[1][1] * b
        return
    hi, lo = max(target, control), min(target, control)
    v = psi.view(-1, 2, 1 << (hi - lo - 1), 2, 1 << lo)
    a, b = (v[:, 0, :, 1], v[:, 1, :, 1]) if hi == target else (v[:, 1, :, 0], v[:, 1, :, 1])
    x = a.clone()
    a_new, b_new = u[0][0] * x + u[0][1] * b, u[1][0] * x + u[1][1] * b
    a.copy_(a_new)
    b.copy_(b_new)


def _operator(psi, n, targets, u):
    """A 2^k x 2^k matrix on targets (targets[0] the lowest index bit); a new tensor."""
    dims = [n - 1 - t for t in reversed(targets)]  # axis of the highest index bit first
    rest = [d for d in range(n) if d not in dims]
    if n > 20:  # merge the axes between the targets: fewer, larger ones
        cuts = sorted(targets, reverse=True)
        shape, axis, top = [], {}, n
        for t in cuts:
            shape += [1 << (top - t - 1), 2]
            axis[t] = len(shape) - 1
            top = t
        shape.append(1 << top)
        dims = [axis[t] for t in reversed(targets)]
        rest = [d for d in range(len(shape)) if d not in dims]
    else:
        shape = [2] * n
    order = dims + rest
    v = psi.view(shape).permute(order)
    m = torch.as_tensor(np.asarray(u), device=psi.device) @ v.reshape(1 << len(targets), -1)
    back = [order.index(d) for d in range(len(order))]
    return m.view([shape[d] for d in order]).permute(back).reshape(-1).contiguous()


def _matrix(name, t):
    c, s, r, e = math.cos(t / 2), math.sin(t / 2), math.sqrt(0.5), complex(math.cos(t), math.sin(t))
    return {"H": [[r, r], [r, -r]], "X": [[0, 1], [1, 0]], "Y": [[0, -1j], [1j, 0]], "Z": [[1, 0], [0, -1]],
            "P": [[1, 0], [0, e]], "RX": [[c, -1j * s], [-1j * s, c]], "RY": [[c, -s], [s, c]],
            "RZ": [[c - 1j * s, 0], [0, c + 1j * s]]}[name]


def _product(case, seed, twice=False):
    theta, phi = _angles(case, seed)
    if case["precision"] == "f32" and case["kind"] in ("ops", "density"):  # that library takes floats
        theta, phi = theta.astype(np.float32).astype(float), phi.astype(np.float32).astype(float)
    psi = torch.ones(1, dtype=torch.complex128, device="cuda")
    for a, b in zip(theta, phi):
        lo = math.cos(a / 2) * complex(math.cos(b / 2), -math.sin(b / 2))
        up = math.sin(a / 2) * complex(math.cos(b / 2), math.sin(b / 2))
        psi = torch.cat([lo * psi, up * psi])
    return torch.outer(psi.conj(), psi).reshape(-1) if twice else psi


def _out(psi):
    return torch.view_as_real(psi)


def _exact_kmeans(case, seed):
    data = _dataset(case, seed)
    cents = np.array(data.init)
    points = [data.point(p) / np.linalg.norm(data.point(p)) for p in range(case["points"])]
    groups = {q: np.flatnonzero(data.qubits == q) for q in set(data.qubits.tolist())}
    stacked = {q: np.stack([points[p] for p in ix]) for q, ix in groups.items()}
    p0 = np.empty((case["points"], case["clusters"]))
    for _ in range(case["iterations"]):
        for q, ix in groups.items():
            c = cents[:, :1 << q]
            norm = np.linalg.norm(c, axis=1, keepdims=True)
            p0[ix] = 0.5 + 0.5 * (stacked[q] @ (c / np.where(norm > 0, norm, 1)).T) ** 2
        assigned = np.argmax(p0, axis=1)
        sums, counts = np.zeros_like(cents), np.zeros_like(cents)
        for q, ix in groups.items():
            np.add.at(sums[:, :1 << q], assigned[ix], stacked[q])
            np.add.at(counts[:, :1 << q], assigned[ix], 1.0)
        cents = np.where(counts > 0, sums / np.maximum(counts, 1), cents)
    return {"p0": p0, "assignments": None, "centroids": cents.reshape(case["clusters"], -1)}


def _exact_density(case, seed):
    n = case["qubits"]
    rho = _product(case, seed, twice=True)
    damp, deph, depol = _noise(case, seed)
    d = 4 * depol / 3

    def channel(q, f, d00, d01, d10, d11):
        v = rho.view(-1, 2, 1 << (n - 1), 2, 1 << q)
        v[:, 0, :, 1] *= f
        v[:, 1, :, 0] *= f
        a, b = v[:, 0, :, 0].clone(), v[:, 1, :, 1].clone()
        v[:, 0, :, 0] = d00 * a + d01 * b
        v[:, 1, :, 1] = d10 * a + d11 * b

    for name, qubits, t in operations(case, seed):
        u = np.array(_matrix(name[1:] if len(qubits) == 2 else name, t), dtype=complex)
        control = qubits[0] if len(qubits) == 2 else None
        _m2(rho, qubits[-1], u.tolist(), control)
        _m2(rho, qubits[-1] + n, u.conj().tolist(), None if control is None else control + n)
        for q in qubits:
            channel(q, math.sqrt(1 - damp), 1, damp, 0, 1 - damp)
        for q in qubits:
            channel(q, 1 - 2 * deph, 1, 0, 0, 1)
        for q in qubits:
            channel(q, 1 - d, 1 - d / 2, d / 2, d / 2, 1 - d / 2)
    diag = torch.diagonal(rho.view(1 << n, 1 << n)).real
    zeros = np.array([float(diag.reshape(-1, 2, 1 << q)[:, 0].sum()) for q in range(n)])
    return {"purity": np.float64(float(_out(rho).square().sum())), "zeros": zeros, "state": _out(rho)}


def _exact_trotter(case, seed):
    inst, psi = _hamiltonian(case, seed), _product(case, seed)
    dim = psi.numel()
    index = torch.arange(dim, device="cuda")

    def parity(x):
        for k in (16, 8, 4, 2, 1):
            x = x ^ (x >> k)
        return x & 1

    bits = 1 << np.arange(case["qubits"])
    terms = [(int(bits[(row == 1) | (row == 2)].sum()), int(bits[(row == 2) | (row == 3)].sum()),
              int((row == 2).sum()), float(c)) for row, c in zip(inst.codes, inst.coeffs)]

    def one(t, z):
        x, zm, ny, c = terms[t]
        angle = 2 * z * c
        partner = index ^ x
        sign = 1 - 2 * parity(partner & zm).to(torch.float64)
        if x:
            return math.cos(angle / 2) * psi + (-1j * math.sin(angle / 2) * (1j ** ny)) * (sign * psi[partner])
        return psi * torch.complex(torch.full_like(sign, math.cos(angle / 2)), -math.sin(angle / 2) * sign)

    def sequence(z, order):
        if order == 1:
            return [(t, z) for t in range(len(terms))]
        if order == 2:
            half = [(t, z / 2) for t in range(len(terms))]
            return half + half[::-1]
        p = 1 / (4 - 4 ** (1 / (order - 1)))
        outer = sequence(p * z, order - 2)
        return outer * 2 + sequence((1 - 4 * p) * z, order - 2) + outer * 2

    for t, z in sequence(inst.time / case["reps"], case["order"]) * case["reps"]:
        psi = one(t, z)
    return {"state": _out(psi)}


def exact(case, seed):
    kind, n = case["kind"], case.get("qubits")
    if kind == "kmeans":
        return _exact_kmeans(case, seed)
    if kind == "density":
        return _exact_density(case, seed)
    if kind == "trotter":
        rotations = _hamiltonian(case, 1).terms * H.stages(case["order"]) * case["reps"]
        return _exact_trotter(case, seed) if rotations * 2.0 ** n < 6e10 else None
    psi = _product(case, seed)
    if kind == "ops":
        for name, qubits, t in operations(case, seed):
            if len(qubits) == 1:
                _m2(psi, qubits[0], _matrix(name, t))
            else:
                _m2(psi, qubits[1], _matrix(name[1:], t), qubits[0])
        k = min(n, 6)
        probs = _out(psi).square().sum(-1).view(-1, 1 << k).sum(0)
        return {"prob": np.float64(1.0), "probs": probs, "state": _out(psi)}
    for g in _brick(case, seed):
        if g[0] == "cu":
            a, b = g[2], g[3]
            _m2(psi, g[1], [[a, -b.conjugate()], [b, a.conjugate()]])
        elif g[0] == "cnot":
            _m2(psi, g[2], _matrix("X", 0.0), g[1])
        elif g[0] == "rz":
            _m2(psi, g[1], _matrix("RZ", g[2]))
        elif g[0] == "mcu":
            u = np.eye(1 << (len(g[1]) + 1), dtype=complex)
            u[-2:, -2:] = g[3]
            psi = _operator(psi, n, [g[2]] + list(g[1]), u)
        else:
            psi = _operator(psi, n, list(g[1]), g[2])
    return {"state": _out(psi)}
