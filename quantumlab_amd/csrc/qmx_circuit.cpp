// Operation lists and the fusion planner.
//
// A qmxCircuit records the operations of one register width: QuantumLab's
// basic operations (EBasicOperation, QL/Circuit/QLGate.h:18-104, same codes)
// and the QuEST gate calls of the older recorders (compactUnitary, unitary,
// rotateZ, controlledNot, multiControlledUnitary, multiQubitUnitary). Every
// operation is validated when it is recorded, with QuEST's messages.
//
// Applied unfused, each operation is the QuEST call that
// QLGate::PerformBasicOperation makes for it (QL/Circuit/QLGate.cpp:652-803):
// noise operations act on density registers only, a controlled collapse
// (EBO_CC) returns its outcome's probability, and the product of those
// probabilities is returned, as the simulators accumulate it
// (QL/Simulator/QLSimulatorVector.cpp:53-59). On density registers every
// operation that is neither noise nor a collapse is followed by the density
// simulator's after-gate noise (QLSimulatorDensityMatrix.cpp:88-153).
//
// Applied fused (state vectors), the unitaries between collapses run as dense
// blocks, and each collapse is a barrier no block crosses. Blocks of at most 5
// qubits on registers of more than 12 qubits share sweeps (qmx_plan.cpp plans
// them, qmx_sweep.hip builds and applies them: many gates to a read and write of
// the register); other block sizes take one sweep a block (qmx::applyMatrixN).
// State vectors of at most 12 qubits lie in one workgroup's LDS: a fused circuit
// runs there in blocks of 4 and 5 qubits, a list applied once or unfused gate by
// gate, in one launch between collapses and gates too wide for it. On density
// registers, fused application is the unfused sequence: a recorded circuit's operations are the QuEST
// calls, which compose into superoperator sweeps two qubits at a time, and
// qmxApplyOperations plans its list as gates on the row and column bits.
//
// The block planner below (qmxCircuitFuse's steps) is greedy and dependency-aware:
// see fuseSegment. Block matrices are products of the expanded gate matrices,
// formed on the host in FP64.
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <limits>
#include <vector>

#include "QuEST.h"
#include "qmx_internal.h"
#include "qmx_sweep.h"
#include "quest_mi355x.h"
#include "quest_validation.h"

using qmx::Cplx;
using qmx::FlatGate;

namespace {

enum GateKind { G_NONE = -1, G_MATRIX2 = 0, G_NOT = 1, G_MATRIXN = 2 };

struct Gate {
    int kind = G_NONE;
    int target = -1;            // G_MATRIX2 / G_NOT
    uint64_t ctrlMask = 0;      // all kinds
    std::vector<int> targs;     // G_MATRIXN (targs[0] = LSB)
    std::vector<Cplx> u;        // 4 entries (MATRIX2) or dim*dim (MATRIXN), row-major
    uint64_t qubitMask() const {
        uint64_t m = ctrlMask;
        if (kind == G_MATRIXN)
            for (int t : targs) m |= 1ull << t;
        else
            m |= 1ull << target;
        return m;
    }
};

// codes of the older recorders (QuEST calls), after QuantumLab's codes
enum : int {
    OP_COMPACT_UNITARY = 100,
    OP_UNITARY,
    OP_ROTATE_Z,
    OP_MULTI_CONTROLLED_UNITARY,
    OP_MULTI_QUBIT_UNITARY
};

struct Op {
    int code = 0;
    std::vector<int> qubits;    // as QuantumLab lists them (controls first); targets of a multi-qubit unitary
    int target = -1;            // older recorders: the 2x2 target
    double param = 0;           // angle, probability or outcome
    Complex alpha{}, beta{};    // OP_COMPACT_UNITARY
    ComplexMatrix2 m2{};        // OP_UNITARY, OP_MULTI_CONTROLLED_UNITARY
    ComplexMatrixN mN{};        // OP_MULTI_QUBIT_UNITARY (owned)
    Gate gate;                  // matrix form for fusion; G_NONE: not a unitary
    bool barrier = false;       // a collapse: no block crosses it
};

struct Block {
    uint64_t mask = 0;          // qubits of the block
    std::vector<int> gates;     // indices into the operation list, in order
    std::vector<int> targs;     // ascending qubits (targs[0] = LSB of the block matrix)
    std::vector<Cplx> u;        // dense block matrix, row-major; empty until something wants it
    void *prepared5 = nullptr;  // its device form for FP32 registers (5 qubits)
    int barrierOp = -1;         // >= 0: this step is the collapse ops[barrierOp]
};

Cplx cmul(Cplx a, Cplx b) { return Cplx{a.re * b.re - a.im * b.im, a.re * b.im + a.im * b.re}; }
Cplx cadd(Cplx a, Cplx b) { return Cplx{a.re + b.re, a.im + b.im}; }

// apply gate g to a k-qubit column vector v (local bit j <-> qubit qs[j])
void applyLocal(const Gate &g, const std::vector<int> &qs, std::vector<Cplx> &v) {
    const int k = (int)qs.size();
    auto local = [&](int q) {
        for (int j = 0; j < k; ++j)
            if (qs[j] == q) return j;
        return -1;
    };
    uint64_t lctrl = 0;
    for (int q = 0; q < 64; ++q)
        if ((g.ctrlMask >> q) & 1ull) lctrl |= 1ull << local(q);
    const size_t dim = v.size();
    if (g.kind == G_MATRIX2 || g.kind == G_NOT) {
        const int t = local(g.target);
        const size_t bit = 1ull << t;
        for (size_t i = 0; i < dim; ++i) {
            if (i & bit) continue;
            if ((i & lctrl) != lctrl) continue;
            Cplx a = v[i], b = v[i | bit];
            if (g.kind == G_NOT) {
                v[i] = b;
                v[i | bit] = a;
            } else {
                v[i] = cadd(cmul(g.u[0], a), cmul(g.u[1], b));
                v[i | bit] = cadd(cmul(g.u[2], a), cmul(g.u[3], b));
            }
        }
        return;
    }
    const int gk = (int)g.targs.size();
    const int gd = 1 << gk;
    std::vector<int> lt(gk);
    uint64_t tmask = 0;
    for (int j = 0; j < gk; ++j) {
        lt[j] = local(g.targs[j]);
        tmask |= 1ull << lt[j];
    }
    std::vector<Cplx> in(gd), out(gd);
    std::vector<size_t> idx(gd);
    for (size_t base = 0; base < dim; ++base) {
        if (base & tmask) continue;
        if ((base & lctrl) != lctrl) continue;
        for (int c = 0; c < gd; ++c) {
            size_t i = base;
            for (int j = 0; j < gk; ++j)
                if ((c >> j) & 1) i |= 1ull << lt[j];
            idx[c] = i;
            in[c] = v[i];
        }
        for (int r = 0; r < gd; ++r) {
            Cplx s{0, 0};
            for (int c = 0; c < gd; ++c) s = cadd(s, cmul(g.u[(size_t)r * gd + c], in[c]));
            out[r] = s;
        }
        for (int r = 0; r < gd; ++r) v[idx[r]] = out[r];
    }
}

// 2x2 gate forms of QuantumLab's single-qubit operations, as the QuEST call
// each one maps to applies it (rotations: QuEST_common.c:117-124, compact form
// [[a, -conj(b)], [b, conj(a)]])
void setMatrix2(Gate &g, int target, uint64_t ctrl, Cplx u00, Cplx u01, Cplx u10, Cplx u11) {
    g.kind = G_MATRIX2;
    g.target = target;
    g.ctrlMask = ctrl;
    g.u = {u00, u01, u10, u11};
}

void setCompact(Gate &g, int target, uint64_t ctrl, Cplx a, Cplx b) {
    setMatrix2(g, target, ctrl, a, Cplx{-b.re, b.im}, b, Cplx{a.re, -a.im});
}

// the rotation about axis (x, y, z) by `angle` as a compact pair
void rotationPair(double angle, double x, double y, double z, Cplx &a, Cplx &b) {
    const double c = std::cos(angle / 2.0), s = std::sin(angle / 2.0);
    a = Cplx{c, -s * z};
    b = Cplx{s * y, -s * x};
}

void setRotation(Gate &g, int target, uint64_t ctrl, double angle, double x, double y, double z) {
    Cplx a, b;
    rotationPair(angle, x, y, z, a, b);
    setCompact(g, target, ctrl, a, b);
}

// QuantumLab's operation `code` on qubits q with angle t in matrix form; false
// where it has none (noise, collapses, undispatched codes)
bool basicGate(int code, const int *q, double t, FlatGate &g) {
    const double r = 1.0 / std::sqrt(2.0);
    auto matrix = [&](int target, uint64_t ctrl, Cplx u00, Cplx u01, Cplx u10, Cplx u11) {
        g.kind = FlatGate::MATRIX2;
        g.target = target;
        g.ctrl = ctrl;
        g.u[0] = u00;
        g.u[1] = u01;
        g.u[2] = u10;
        g.u[3] = u11;
        return true;
    };
    auto rotation = [&](int target, uint64_t ctrl, double x, double y, double z) {
        Cplx a, b;
        rotationPair(t, x, y, z, a, b);
        return matrix(target, ctrl, a, Cplx{-b.re, b.im}, b, Cplx{a.re, -a.im});
    };
    auto bitNot = [&](int target, uint64_t ctrl) {
        g.kind = FlatGate::NOT;
        g.target = target;
        g.ctrl = ctrl;
        return true;
    };
    const Cplx zero{0, 0}, one{1, 0};
    switch (code) {
        case QMX_OP_H: return matrix(q[0], 0, {r, 0}, {r, 0}, {r, 0}, {-r, 0});
        case QMX_OP_X: return bitNot(q[0], 0);
        case QMX_OP_Y: return matrix(q[0], 0, zero, {0, -1}, {0, 1}, zero);
        case QMX_OP_Z: return matrix(q[0], 0, one, zero, zero, {-1, 0});
        case QMX_OP_P: return matrix(q[0], 0, one, zero, zero, {std::cos(t), std::sin(t)});
        case QMX_OP_RX: return rotation(q[0], 0, 1, 0, 0);
        case QMX_OP_RY: return rotation(q[0], 0, 0, 1, 0);
        case QMX_OP_RZ: return rotation(q[0], 0, 0, 0, 1);
        case QMX_OP_CX: return bitNot(q[1], 1ull << q[0]);
        case QMX_OP_CY: return matrix(q[1], 1ull << q[0], zero, {0, -1}, {0, 1}, zero);
        case QMX_OP_CZ: return matrix(q[1], 1ull << q[0], one, zero, zero, {-1, 0});
        case QMX_OP_CP: return matrix(q[1], 1ull << q[0], one, zero, zero, {std::cos(t), std::sin(t)});
        case QMX_OP_CRX: return rotation(q[1], 1ull << q[0], 1, 0, 0);
        case QMX_OP_CRY: return rotation(q[1], 1ull << q[0], 0, 1, 0);
        case QMX_OP_CRZ: return rotation(q[1], 1ull << q[0], 0, 0, 1);
        default: return false;
    }
}

bool basicGate(Op &o) {
    FlatGate f;
    if (!basicGate(o.code, o.qubits.data(), o.param, f)) return false;
    o.gate.kind = f.kind == FlatGate::NOT ? G_NOT : G_MATRIX2;
    o.gate.target = f.target;
    o.gate.ctrlMask = f.ctrl;
    if (f.kind == FlatGate::MATRIX2) o.gate.u.assign(f.u, f.u + 4);
    return true;
}

FlatGate flatGate(const Gate &g) {
    FlatGate f;
    f.target = g.target;
    f.ctrl = g.ctrlMask;
    if (g.kind == G_MATRIXN) {
        f.kind = FlatGate::MATRIXN;
        f.k = (int)g.targs.size();
        f.targs = g.targs.data();
        f.uN = g.u.data();
    } else if (g.kind == G_NOT) {
        f.kind = FlatGate::NOT;
    } else {
        std::copy(g.u.begin(), g.u.end(), f.u);
    }
    return f;
}

// the one-qubit channel `code` of strength p on qubit q of an n-qubit density
// register, with the numbers of its QuEST call; false for two-qubit channels
bool channelGate(int code, int q, int n, double p, FlatGate &g) {
    auto channel = [&](double f, double swap, double d00, double d01, double d10, double d11) {
        g.kind = FlatGate::CHANNEL;
        g.target = q;
        g.ctrl = 0;
        g.k = q + n;
        g.u[0] = Cplx{f, swap};
        g.u[1] = Cplx{d00, d01};
        g.u[2] = Cplx{d10, d11};
        g.u[3] = Cplx{0, 0};
        return true;
    };
    auto pauli = [&](double x, double y, double z) {
        const double none = 1 - (x + y + z);
        return channel(none - z, x - y, none + z, x + y, x + y, none + z);
    };
    switch (code) {
        case QMX_OP_NOISE_DAMPING: return channel(std::sqrt(1 - p), 0, 1, p, 0, 1 - p);
        case QMX_OP_NOISE_DEPHASING: return channel(1 - 2 * p, 0, 1, 0, 0, 1);
        case QMX_OP_NOISE_DEPOLARISING: {
            const double level = (4 * p) / 3.0, h = level / 2;
            return channel(1 - level, 0, 1 - h, h, h, 1 - h);
        }
        case QMX_OP_NOISE_MIX_PAULI_X: return pauli(p, 0, 0);
        case QMX_OP_NOISE_MIX_PAULI_Y: return pauli(0, p, 0);
        case QMX_OP_NOISE_MIX_PAULI_Z: return pauli(0, 0, p);
        case QMX_OP_NOISE_MIX_PAULI_ALL: return pauli(p, p, p);
        default: return false;
    }
}

bool lone1(const FlatGate &g) { return (g.kind == FlatGate::MATRIX2 || g.kind == FlatGate::NOT) && !g.ctrl; }

// gate b after gate a, both on the same one qubit, as one
void joinGate(FlatGate &a, const FlatGate &b) {
    static const Cplx swap[4] = {{0, 0}, {1, 0}, {1, 0}, {0, 0}};
    Cplx x[4], y[4];
    std::copy(b.kind == FlatGate::NOT ? swap : b.u, (b.kind == FlatGate::NOT ? swap : b.u) + 4, x);
    std::copy(a.kind == FlatGate::NOT ? swap : a.u, (a.kind == FlatGate::NOT ? swap : a.u) + 4, y);
    a.kind = FlatGate::MATRIX2;
    for (int r = 0; r < 2; ++r)
        for (int c = 0; c < 2; ++c) a.u[2 * r + c] = cadd(cmul(x[2 * r], y[c]), cmul(x[2 * r + 1], y[2 + c]));
}

// Gate g at the end of `gates`, or inside the last one where that is the last to touch
// its one qubit (last[qubit]: index of the last gate on it, -1 for none): in lists of
// two one-qubit gates to each two-qubit one, a third of the gates go that way (10
// qubits FP32, 80 gates: 53 steps of the LDS kernel, 62 -> 49 us with the reads).
void appendGate(std::vector<FlatGate> &gates, int *last, const FlatGate &g) {
    if (lone1(g) && last[g.target] >= 0 && lone1(gates[last[g.target]])) {
        joinGate(gates[last[g.target]], g);
        return;
    }
    for (uint64_t m = g.mask(); m; m &= m - 1) last[__builtin_ctzll(m)] = (int)gates.size();
    gates.push_back(g);
}

// Channel b after channel a on the same qubit, as one; false where the pair does not
// join. The same rates after every gate make the same product, and the rounding of its
// numbers, alike in hundreds of channels, does not average out: those near 1 keep what
// FP64 does not hold of them, and products with large numbers beside them are not made.
// (60 operations with noise on 7 qubits FP64, error of the state over 8 draws against
// 80-bit arithmetic: 1.6e-15 to 3.0e-15 with all numbers rounded, 0.8e-15 to 1.2e-15 so,
// 0.8e-15 to 1.4e-15 where each pair of qubits is one superoperator at a time.)
bool joinChannel(FlatGate &a, const FlatGate &b) {
    typedef long double L;
    struct Maps {
        L f, g, d00, d01, d10, d11;
    };
    auto read = [](const FlatGate &c) {
        return Maps{(L)c.u[0].re + (L)c.u[3].re, c.u[0].im, (L)c.u[1].re + (L)c.u[3].im, c.u[1].im, c.u[2].re,
                    (L)c.u[2].im + (L)c.lo};
    };
    const Maps x = read(a), y = read(b);
    const Maps r{y.f * x.f + y.g * x.g,         y.f * x.g + y.g * x.f,         y.d00 * x.d00 + y.d01 * x.d10,
                 y.d00 * x.d01 + y.d01 * x.d11, y.d10 * x.d00 + y.d11 * x.d10, y.d10 * x.d01 + y.d11 * x.d11};
    const L most = 0.0625L;
    if (std::fabs(r.g) > most || std::fabs(r.d01) > most || std::fabs(r.d10) > most) return false;
    a.u[0] = Cplx{(double)r.f, (double)r.g};
    a.u[1] = Cplx{(double)r.d00, (double)r.d01};
    a.u[2] = Cplx{(double)r.d10, (double)r.d11};
    a.u[3] = Cplx{(double)(r.f - (L)a.u[0].re), (double)(r.d00 - (L)a.u[1].re)};
    a.lo = (float)(r.d11 - (L)a.u[2].im);
    return true;
}

// qubits an operation code takes (0: not a recordable QuantumLab code)
int arity(int code) {
    switch (code) {
        case QMX_OP_H: case QMX_OP_X: case QMX_OP_Y: case QMX_OP_Z: case QMX_OP_P: case QMX_OP_RX:
        case QMX_OP_RY: case QMX_OP_RZ: case QMX_OP_CC: case QMX_OP_NOISE_DAMPING: case QMX_OP_NOISE_DEPHASING:
        case QMX_OP_NOISE_DEPOLARISING: case QMX_OP_NOISE_MIX_PAULI_X: case QMX_OP_NOISE_MIX_PAULI_Y:
        case QMX_OP_NOISE_MIX_PAULI_Z: case QMX_OP_NOISE_MIX_PAULI_ALL:
            return 1;
        case QMX_OP_CX: case QMX_OP_CY: case QMX_OP_CZ: case QMX_OP_CP: case QMX_OP_CRX: case QMX_OP_CRY:
        case QMX_OP_CRZ: case QMX_OP_NOISE_TWO_QUBIT_DEPHASING: case QMX_OP_NOISE_TWO_QUBIT_DEPOLARISING:
            return 2;
        default: return 0;
    }
}

bool isNoise(int code) { return code >= QMX_OP_NOISE_DAMPING && code <= QMX_OP_NOISE_TWO_QUBIT_DEPOLARISING; }

}  // namespace

// The gates of a list in matrix form, and where the list stops for an operation
// that is not one (a collapse): ops[stops[i].second] runs before gate stops[i].first.
struct GateList {
    std::vector<FlatGate> gates;
    std::vector<int> op;                       // each gate's operation
    std::vector<std::pair<int, int>> stops;
};

// A fused circuit's sweeps for one storage precision; stops as in GateList, but
// before sweep stops[i].first.
struct CircuitSweeps {
    GateList list;
    qmx::SweepPlan plan;
    std::vector<std::pair<int, int>> stops;
    qmx::SweepProgram *program = nullptr;
};

struct qmxCircuit {
    int numQubits;
    Qureg shape;                // register of this width, for the recorders' validation
    std::vector<Op> ops;
    std::vector<Block> blocks;
    int fusedQubits = 0;
    int fusedOps = 0;           // operations the last fuse covered
    CircuitSweeps *sweeps[2] = {nullptr, nullptr};  // by storage precision, planned when first needed
    qmxNoiseAfterGate noise{};
    void releaseBlocks() {
        for (Block &b : blocks) qmx::fused5Free(b.prepared5);
        blocks.clear();
        for (CircuitSweeps *&s : sweeps) {
            if (s) qmx::sweepProgramFree(s->program);
            delete s;
            s = nullptr;
        }
    }
    ~qmxCircuit() {
        releaseBlocks();
        for (Op &o : ops)
            if (o.code == OP_MULTI_QUBIT_UNITARY) destroyComplexMatrixN(o.mN);
    }
};

namespace {

void listTargets(Block &b) {
    b.targs.clear();
    for (uint64_t m = b.mask; m; m &= m - 1) b.targs.push_back(__builtin_ctzll(m));
}

void buildBlockMatrix(const qmxCircuit &c, Block &b) {
    const size_t dim = 1ull << b.targs.size();
    b.u.assign(dim * dim, Cplx{0, 0});
    std::vector<Cplx> col(dim);
    for (size_t cidx = 0; cidx < dim; ++cidx) {
        std::fill(col.begin(), col.end(), Cplx{0, 0});
        col[cidx] = Cplx{1, 0};
        for (int gi : b.gates) applyLocal(c.ops[gi].gate, b.targs, col);
        for (size_t r = 0; r < dim; ++r) b.u[r * dim + cidx] = col[r];
    }
}

void mixNoise(const Qureg &q, int code, int a, int b, qreal p) {
    switch (code) {
        case QMX_OP_NOISE_DAMPING: mixDamping(q, a, p); break;
        case QMX_OP_NOISE_DEPHASING: mixDephasing(q, a, p); break;
        case QMX_OP_NOISE_DEPOLARISING: mixDepolarising(q, a, p); break;
        case QMX_OP_NOISE_MIX_PAULI_X: mixPauli(q, a, p, 0, 0); break;
        case QMX_OP_NOISE_MIX_PAULI_Y: mixPauli(q, a, 0, p, 0); break;
        case QMX_OP_NOISE_MIX_PAULI_Z: mixPauli(q, a, 0, 0, p); break;
        case QMX_OP_NOISE_MIX_PAULI_ALL: mixPauli(q, a, p, p, p); break;
        case QMX_OP_NOISE_TWO_QUBIT_DEPHASING: mixTwoQubitDephasing(q, a, b, p); break;
        case QMX_OP_NOISE_TWO_QUBIT_DEPOLARISING: mixTwoQubitDepolarising(q, a, b, p); break;
        default: break;
    }
}

// the QuEST call QLGate::PerformBasicOperation makes (QLGate.cpp:652-803);
// returns the collapse probability, else 1
double runOp(const Qureg &q, Op &o) {
    const int *qs = o.qubits.data();
    const qreal t = (qreal)o.param;
    const bool dm = q.isDensityMatrix != 0;
    switch (o.code) {
        case QMX_OP_H: hadamard(q, qs[0]); break;
        case QMX_OP_X: pauliX(q, qs[0]); break;
        case QMX_OP_Y: pauliY(q, qs[0]); break;
        case QMX_OP_Z: pauliZ(q, qs[0]); break;
        case QMX_OP_P: phaseShift(q, qs[0], t); break;
        case QMX_OP_RX: rotateX(q, qs[0], t); break;
        case QMX_OP_RY: rotateY(q, qs[0], t); break;
        case QMX_OP_RZ: rotateZ(q, qs[0], t); break;
        case QMX_OP_CX: controlledNot(q, qs[0], qs[1]); break;
        case QMX_OP_CY: controlledPauliY(q, qs[0], qs[1]); break;
        case QMX_OP_CZ: controlledPhaseFlip(q, qs[0], qs[1]); break;
        case QMX_OP_CP: controlledPhaseShift(q, qs[0], qs[1], t); break;
        case QMX_OP_CRX: controlledRotateX(q, qs[0], qs[1], t); break;
        case QMX_OP_CRY: controlledRotateY(q, qs[0], qs[1], t); break;
        case QMX_OP_CRZ: controlledRotateZ(q, qs[0], qs[1], t); break;
        case QMX_OP_CC: return collapseToOutcome(q, qs[0], (int)o.param);
        // noise: density registers only; a state vector ignores it, as the reference does
        case QMX_OP_NOISE_DAMPING: case QMX_OP_NOISE_DEPHASING: case QMX_OP_NOISE_DEPOLARISING:
        case QMX_OP_NOISE_MIX_PAULI_X: case QMX_OP_NOISE_MIX_PAULI_Y: case QMX_OP_NOISE_MIX_PAULI_Z:
        case QMX_OP_NOISE_MIX_PAULI_ALL: case QMX_OP_NOISE_TWO_QUBIT_DEPHASING:
        case QMX_OP_NOISE_TWO_QUBIT_DEPOLARISING:
            if (dm) mixNoise(q, o.code, qs[0], o.qubits.size() > 1 ? qs[1] : -1, t);
            break;
        case OP_COMPACT_UNITARY: compactUnitary(q, o.target, o.alpha, o.beta); break;
        case OP_UNITARY: unitary(q, o.target, o.m2); break;
        case OP_ROTATE_Z: rotateZ(q, o.target, t); break;
        case OP_MULTI_CONTROLLED_UNITARY:
            multiControlledUnitary(q, o.qubits.data(), (int)o.qubits.size(), o.target, o.m2);
            break;
        case OP_MULTI_QUBIT_UNITARY: multiQubitUnitary(q, o.qubits.data(), (int)o.qubits.size(), o.mN); break;
        default:
            // EBO_Phase and EBO_Composite: PerformBasicOperation dispatches neither
            std::printf("not supported type!\n");
            break;
    }
    return 1.0;
}

// the density simulator's noise after every operation that is neither noise
// nor a collapse, on the qubits that operation lists (QLSimulatorDensityMatrix.cpp:88-153):
// emit(code, q0, q1, p) for each channel
template <class F>
void noiseAfterGate(int code, const int *qs, int n, const qmxNoiseAfterGate &nz, F emit) {
    if (isNoise(code) || code == QMX_OP_CC) return;
    const qreal tiny = std::numeric_limits<qreal>::min();
    auto each = [&](int channel, qreal p) {
        for (int i = 0; i < n; ++i) emit(channel, qs[i], -1, p);
    };
    if (nz.damping > tiny) each(QMX_OP_NOISE_DAMPING, nz.damping);
    if (nz.dephasing > tiny && (nz.twoQubitDephasing < tiny || n == 1)) each(QMX_OP_NOISE_DEPHASING, nz.dephasing);
    if (nz.depolarising > tiny && (nz.twoQubitDepolarising < tiny || n == 1))
        each(QMX_OP_NOISE_DEPOLARISING, nz.depolarising);
    if (nz.mixPauli > tiny) each(QMX_OP_NOISE_MIX_PAULI_ALL, nz.mixPauli);
    if (nz.twoQubitDepolarising > tiny && n == 2)
        emit(QMX_OP_NOISE_TWO_QUBIT_DEPOLARISING, qs[0], qs[1], nz.twoQubitDepolarising);
    if (nz.twoQubitDephasing > tiny && n == 2)
        emit(QMX_OP_NOISE_TWO_QUBIT_DEPHASING, qs[0], qs[1], nz.twoQubitDephasing);
}

void noiseAfterGate(const Qureg &q, const Op &o, const qmxNoiseAfterGate &nz) {
    std::vector<int> qs = o.qubits;
    if (o.target >= 0) qs.push_back(o.target);
    noiseAfterGate(o.code, qs.data(), (int)qs.size(), nz,
                   [&](int channel, int a, int b, qreal p) { mixNoise(q, channel, a, b, p); });
}

bool hasNoise(const qmxNoiseAfterGate &nz) {
    return nz.damping > 0 || nz.dephasing > 0 || nz.depolarising > 0 || nz.mixPauli > 0 ||
           nz.twoQubitDephasing > 0 || nz.twoQubitDepolarising > 0;
}

// accepted and not dispatched, as in PerformBasicOperation
bool undispatched(int code) { return code == QMX_OP_PHASE || code == QMX_OP_COMPOSITE; }

void checkBasic(const Qureg &s, int code, const int *qubits, int numQubits, double param, const char *f) {
    const int need = arity(code);
    if (undispatched(code)) {
        if (numQubits < 0 || numQubits > 2) qv::raise("An operation lists at most two qubits.", f);
        for (int i = 0; i < numQubits; ++i) qv::target(s, qubits[i], f);
        return;
    }
    if (need == 0) qv::raise("Invalid operation code. Must be one of QuantumLab's basic operations (0-26).", f);
    if (numQubits != need)
        qv::raise(need == 1 ? "This operation takes exactly one qubit." : "This operation takes exactly two qubits.",
                  f);
    if (need == 1) {
        qv::target(s, qubits[0], f);
    } else if (isNoise(code)) {
        qv::uniqueTargets(s, qubits[0], qubits[1], f);
    } else {
        qv::controlTarget(s, qubits[0], qubits[1], f);
    }
    switch (code) {
        case QMX_OP_CC: qv::outcome((int)param, f); break;
        case QMX_OP_NOISE_DAMPING: qv::oneQubitDampingProb(param, f); break;
        case QMX_OP_NOISE_DEPHASING: qv::oneQubitDephaseProb(param, f); break;
        case QMX_OP_NOISE_DEPOLARISING: qv::oneQubitDepolProb(param, f); break;
        case QMX_OP_NOISE_MIX_PAULI_X: qv::oneQubitPauliProbs(param, 0, 0, f); break;
        case QMX_OP_NOISE_MIX_PAULI_Y: qv::oneQubitPauliProbs(0, param, 0, f); break;
        case QMX_OP_NOISE_MIX_PAULI_Z: qv::oneQubitPauliProbs(0, 0, param, f); break;
        case QMX_OP_NOISE_MIX_PAULI_ALL: qv::oneQubitPauliProbs(param, param, param, f); break;
        case QMX_OP_NOISE_TWO_QUBIT_DEPHASING: qv::twoQubitDephaseProb(param, f); break;
        case QMX_OP_NOISE_TWO_QUBIT_DEPOLARISING: qv::twoQubitDepolProb(param, f); break;
        default: break;
    }
}

void recordBasic(qmxCircuit *c, int code, const int *qubits, int numQubits, double param, const char *f) {
    checkBasic(c->shape, code, qubits, numQubits, param, f);
    Op o;
    o.code = code;
    o.qubits.assign(qubits, qubits + std::max(0, numQubits));
    o.param = param;
    o.barrier = code == QMX_OP_CC;
    if (!undispatched(code)) basicGate(o);
    c->ops.push_back(std::move(o));
}

void noiseParams(const qmxNoiseAfterGate &nz, const char *f) {
    qv::oneQubitDampingProb(nz.damping, f);
    qv::oneQubitDephaseProb(nz.dephasing, f);
    qv::oneQubitDepolProb(nz.depolarising, f);
    qv::oneQubitPauliProbs(nz.mixPauli, nz.mixPauli, nz.mixPauli, f);
    qv::twoQubitDephaseProb(nz.twoQubitDephasing, f);
    qv::twoQubitDepolProb(nz.twoQubitDepolarising, f);
}

void checkRegister(const qmxCircuit *c, const Qureg &q, const char *f) {
    qv::check(qmx::dev(q) != nullptr && qmx::dev(q)->magic == qmx::kMagic, qv::E_QUREG_NOT_ALLOCATED, f);
    if (q.numQubitsRepresented != c->numQubits)
        qv::raise("The circuit and the register have different numbers of qubits.", f);
}

// the first numOps operations as a state vector's gate list; `everyOp`: operations
// without a matrix form stop the list (they run as the QuEST calls they are), but for
// noise, which does nothing there; else only collapses do and the others are skipped,
// as fused application has it
GateList gateList(const qmxCircuit *c, int numOps, bool everyOp) {
    GateList l;
    l.gates.reserve(numOps);
    l.op.reserve(numOps);
    for (int i = 0; i < numOps; ++i) {
        const Op &o = c->ops[i];
        if (o.gate.kind != G_NONE) {
            l.gates.push_back(flatGate(o.gate));
            l.op.push_back(i);
        } else if ((everyOp && !isNoise(o.code)) || o.barrier) {
            l.stops.push_back({(int)l.gates.size(), i});
        }
    }
    return l;
}

// An operation list on a density register of n qubits as gates on its 2n row and
// column bits (qmx_sweep.h), noise included. Lists that hold anything but one- and
// two-qubit gates in matrix form, one-qubit channels and collapses are not taken.
struct DensityList {
    int n;
    GateList l;
    int last[64];               // per qubit: the last gate of the list on its row bit
    int operations = 0;
    explicit DensityList(int numQubits) : n(numQubits) { std::fill(last, last + 64, -1); }
    bool noise(int code, int q, double p) {
        FlatGate g;
        if (!channelGate(code, q, n, p, g)) return false;
        ++operations;
        // a run of channels on one qubit is one channel
        if (last[q] >= 0 && l.gates[last[q]].kind == FlatGate::CHANNEL && join(l.gates[last[q]], g)) return true;
        appendGate(l.gates, last, g);
        return true;
    }
    // joinChannel, whose 80-bit products (30 ns) the list's noise asks for again and again
    struct Joined {
        Cplx a[4], b[4], r[4];
        float aLo, bLo, rLo;
        bool is;
    } joined[4] = {};
    int nextJoined = 0;
    bool join(FlatGate &a, const FlatGate &b) {
        auto same = [](const Cplx *x, const Cplx *y) { return std::memcmp(x, y, 4 * sizeof(Cplx)) == 0; };
        for (const Joined &j : joined)
            if (j.is && same(j.a, a.u) && same(j.b, b.u) && j.aLo == a.lo && j.bLo == b.lo) {
                std::copy(j.r, j.r + 4, a.u);
                a.lo = j.rLo;
                return true;
            }
        Joined j;
        std::copy(a.u, a.u + 4, j.a);
        j.aLo = a.lo;
        if (!joinChannel(a, b)) return false;
        std::copy(b.u, b.u + 4, j.b);
        std::copy(a.u, a.u + 4, j.r);
        j.bLo = b.lo;
        j.rLo = a.lo;
        j.is = true;
        joined[nextJoined] = j;
        nextJoined = (nextJoined + 1) % 4;
        return true;
    }
    void gate(const FlatGate &g) {
        ++operations;
        FlatGate c = g;
        c.target += n;
        c.ctrl <<= n;
        for (Cplx &z : c.u) z.im = -z.im;
        appendGate(l.gates, last, g);
        appendGate(l.gates, last, c);
    }
    void stop(int op) {
        l.stops.push_back({(int)l.gates.size(), op});
        std::fill(last, last + 64, -1);
    }
    // false: the list holds something that has no place here
    bool add(int i, int code, const int *qs, int numQubits, double param, const qmxNoiseAfterGate *nz) {
        FlatGate g;
        if (code == QMX_OP_CC) {
            stop(i);
        } else if (isNoise(code)) {
            if (!noise(code, qs[0], param)) return false;
        } else if (!undispatched(code) && basicGate(code, qs, param, g)) {
            gate(g);
        } else {
            return false;
        }
        bool ok = true;
        if (nz)
            noiseAfterGate(code, qs, numQubits, *nz, [&](int channel, int a, int, qreal p) {
                ok = ok && noise(channel, a, p);
            });
        return ok;
    }
};

// On two qubits, every run of more than 32 gates as one matrix, formed here and kept in
// `room`: 40 ns a gate where the LDS kernel takes 0.35 us (FP32 lists of 60, 400 and 2000
// operations: 25, 35 and 81 us, gate by gate 39, 136 and 590).
void composePairs(GateList &l, std::vector<Cplx> &room) {
    static const int targs[2] = {0, 1};
    std::vector<FlatGate> out;
    const int n = (int)l.gates.size();
    room.assign(16 * (l.stops.size() + 1), Cplx{0, 0});
    int i = 0;
    for (size_t s = 0; s <= l.stops.size(); ++s) {
        const int until = s < l.stops.size() ? l.stops[s].first : n;
        if (until - i <= 32) {
            out.insert(out.end(), l.gates.begin() + i, l.gates.begin() + until);
        } else {
            Cplx *u = room.data() + 16 * s;
            for (int d = 0; d < 4; ++d) u[5 * d] = Cplx{1, 0};
            for (int g = i; g < until; ++g) {
                const FlatGate &f = l.gates[g];
                const int bit = 1 << f.target;
                for (int r = 0; r < 4; ++r) {
                    if ((r & bit) || (r & (int)f.ctrl) != (int)f.ctrl) continue;
                    Cplx *x = u + 4 * r, *y = u + 4 * (r | bit);
                    for (int c = 0; c < 4; ++c) {
                        const Cplx a = x[c], b = y[c];
                        x[c] = f.kind == FlatGate::NOT ? b : cadd(cmul(f.u[0], a), cmul(f.u[1], b));
                        y[c] = f.kind == FlatGate::NOT ? a : cadd(cmul(f.u[2], a), cmul(f.u[3], b));
                    }
                }
            }
            FlatGate m;
            m.kind = FlatGate::MATRIXN;
            m.k = 2;
            m.targs = targs;
            m.uN = u;
            out.push_back(m);
        }
        i = until;
        if (s < l.stops.size()) l.stops[s].first = (int)out.size();
    }
    l.gates = std::move(out);
}

// a gate list on a register of at most kSmallCircuitQubits qubits; stop(op)
// runs an operation that is not a gate
template <class F>
void runSmall(qmx::QuregDev *d, const GateList &l, F stop) {
    size_t s = 0;
    int i = 0;
    const int n = (int)l.gates.size();
    while (i < n || s < l.stops.size()) {
        const int until = s < l.stops.size() ? l.stops[s].first : n;
        while (i < until) {
            int j = i;
            while (j < until && l.gates[j].kind != FlatGate::MATRIXN) ++j;
            if (j > i) qmx::smallCircuit(d, l.gates.data() + i, j - i);
            if (j < until) qmx::applyFlatGate(d, l.gates[j++]);
            i = j;
        }
        if (s < l.stops.size()) stop(l.stops[s++].second);
    }
}

// sweeps for the list's gates, segment by segment: no sweep crosses a stop
void planList(const qmx::SweepShape &shape, const GateList &l, qmx::SweepPlan &plan,
              std::vector<std::pair<int, int>> &stops) {
    int i = 0;
    for (size_t s = 0; s <= l.stops.size(); ++s) {
        const int until = s < l.stops.size() ? l.stops[s].first : (int)l.gates.size();
        if (until > i) qmx::planSweeps(shape, l.gates.data() + i, until - i, i, plan);
        i = until;
        if (s < l.stops.size()) stops.push_back({(int)plan.sweeps.size(), l.stops[s].second});
    }
}

// the list in sweeps of the register, planned and run at once
template <class F>
void runSweepsOnce(qmx::QuregDev *d, const GateList &l, F stop) {
    int at = 0;
    for (size_t s = 0; s <= l.stops.size(); ++s) {
        const int until = s < l.stops.size() ? l.stops[s].first : (int)l.gates.size();
        if (until > at) {
            qmx::SweepPlan plan;
            qmx::planSweeps(qmx::sweepShape(d->numQubits, d->prec, d->isDensity), l.gates.data() + at, until - at, 0,
                            plan);
            qmx::sweepRunOnce(d, plan, l.gates.data() + at);
            if (d->isDensity) qmx::densCountSweeps((long long)plan.sweeps.size(), 0);
        }
        at = until;
        if (s < l.stops.size()) stop(l.stops[s].second);
    }
}

// The fused circuit's sweeps; nullptr where it does not run in sweeps. Small registers
// have one plan for both precisions, whatever the blocks' size: at 9 to 12 qubits and
// 20 brick layers it takes 19, 26, 35 and 63 us, where blocks of 5 at a launch each took
// 64, 104, 81 and 96 (FP32) or 780, 1070, 190 and 256 (FP64) and the gates one by one
// 123, 159, 221 and 347; 4 gates on 4 qubits 4 us, 10 one by one. A gate too wide for a
// block is a launch of its own there (4 to 9 us) and a step of 0.3 to 0.9 us one by one:
// a plan that cuts the list for fewer than 16 gates a launch is not taken.
CircuitSweeps *sweepsOf(qmxCircuit *c, int prec) {
    const bool small = c->numQubits <= qmx::kSmallCircuitQubits;
    if (c->blocks.empty() || (!small && c->fusedQubits != qmx::kSweepBlockQubits)) return nullptr;
    CircuitSweeps *&s = c->sweeps[small ? qmx::FP64 : prec];
    if (!s) {
        s = new CircuitSweeps;
        s->list = gateList(c, c->fusedOps, false);
        planList(small ? qmx::smallShape(c->numQubits) : qmx::sweepShape(c->numQubits, prec, false), s->list, s->plan,
                 s->stops);
    }
    const int cuts = (int)s->plan.sweeps.size() - (int)s->list.stops.size() - 1;
    if (small && cuts > 0 && 16 * cuts > (int)s->list.gates.size()) return nullptr;
    return s;
}

double applyCircuit(const Qureg &q, qmxCircuit *c, int fused) {
    double prob = 1.0;
    const bool noisy = q.isDensityMatrix && hasNoise(c->noise);
    qmx::QuregDev *d = qmx::dev(q);
    const bool asBlocks = fused && !c->blocks.empty() && !q.isDensityMatrix;
    if (CircuitSweeps *s = asBlocks ? sweepsOf(c, d->prec) : nullptr) {
        if (!s->program)
            s->program = qmx::sweepProgramCreate(qmx::smallStateVector(d) ? qmx::FP64 : d->prec, s->plan,
                                                 s->list.gates.data());
        int at = 0;
        for (size_t i = 0; i <= s->stops.size(); ++i) {
            const int until = i < s->stops.size() ? s->stops[i].first : (int)s->plan.sweeps.size();
            qmx::sweepProgramRun(d, s->program, s->plan, s->list.gates.data(), at, until);
            at = until;
            if (i < s->stops.size()) prob *= runOp(q, c->ops[s->stops[i].second]);
        }
        return prob;
    }
    if (qmx::smallStateVector(d)) {
        runSmall(d, asBlocks ? gateList(c, c->fusedOps, false) : gateList(c, (int)c->ops.size(), true),
                 [&](int op) { prob *= runOp(q, c->ops[op]); });
        return prob;
    }
    if (!asBlocks) {
        for (Op &o : c->ops) {
            prob *= runOp(q, o);
            if (noisy) noiseAfterGate(q, o, c->noise);
        }
        return prob;
    }
    for (Block &b : c->blocks) {
        if (b.barrierOp >= 0) {
            prob *= runOp(q, c->ops[b.barrierOp]);
            continue;
        }
        if (b.gates.size() == 1) {
            runOp(q, c->ops[b.gates[0]]);  // a lone gate keeps its cheaper kernel
            continue;
        }
        if (d->prec == qmx::FP32 && b.targs.size() == 5) {  // more than 12 qubits here
            if (!b.prepared5) b.prepared5 = qmx::fused5Prepare(b.targs.data(), b.u.data());
            qmx::fused5Apply(d, b.prepared5);
            continue;
        }
        qmx::applyMatrixN(d, 0, b.targs.data(), (int)b.targs.size(), b.u.data());
    }
    return prob;
}

// Fuse the gates of one segment (no barrier inside) into blocks of at most
// maxQubits qubits. Gates on disjoint qubits commute, so any order that keeps
// each qubit's gates in sequence is the same circuit. Each step takes the
// window of maxQubits consecutive qubits (or a ready gate's own qubits when
// they span more) that absorbs the most gates: from the window's qubits, the
// next pending gate of a qubit joins while it is next on all of its qubits
// and the block stays within maxQubits. On the 32-qubit brick periods this
// makes 18-19 steps per period where placing each gate, in list order, into the
// last block it fits made 26.
void fuseSegment(qmxCircuit *c, const std::vector<int> &seg, int maxQubits) {
    if (seg.empty()) return;
    std::vector<std::vector<int>> per(64);
    std::vector<uint64_t> maskOf(c->ops.size(), 0);
    for (int gi : seg) {
        maskOf[gi] = c->ops[gi].gate.qubitMask();
        for (uint64_t m = maskOf[gi]; m; m &= m - 1) per[__builtin_ctzll(m)].push_back(gi);
    }
    std::vector<size_t> ptr(64, 0);
    auto nextOn = [&](const std::vector<size_t> &p, int x) { return p[x] < per[x].size() ? per[x][p[x]] : -1; };
    auto readyIn = [&](const std::vector<size_t> &p, int gi) {
        for (uint64_t m = maskOf[gi]; m; m &= m - 1)
            if (nextOn(p, __builtin_ctzll(m)) != gi) return false;
        return true;
    };
    const uint64_t all = c->numQubits >= 64 ? ~0ull : (1ull << c->numQubits) - 1ull;
    size_t remaining = seg.size();
    std::vector<uint64_t> seeds;
    while (remaining) {
        seeds.clear();
        int firstReady = -1;
        for (int x = 0; x < 64; ++x) {
            const int gi = nextOn(ptr, x);
            if (gi < 0 || !readyIn(ptr, gi)) continue;
            if (firstReady < 0 || gi < firstReady) firstReady = gi;
            const uint64_t m = maskOf[gi];
            const int lo = __builtin_ctzll(m), hi = 63 - __builtin_clzll(m);
            if (hi - lo + 1 <= maxQubits) {
                for (int k = std::max(0, hi - maxQubits + 1); k <= lo; ++k) {
                    const uint64_t w = (maxQubits >= 64 ? ~0ull : ((1ull << maxQubits) - 1ull) << k) & all;
                    seeds.push_back(w);
                }
            } else if (__builtin_popcountll(m) <= maxQubits) {
                seeds.push_back(m);
            }
        }
        std::sort(seeds.begin(), seeds.end());
        seeds.erase(std::unique(seeds.begin(), seeds.end()), seeds.end());
        Block best;
        std::vector<size_t> bestPtr;
        for (uint64_t w : seeds) {
            std::vector<size_t> p = ptr;
            Block b;
            for (bool progress = true; progress;) {
                progress = false;
                for (uint64_t wm = w; wm; wm &= wm - 1) {
                    const int x = __builtin_ctzll(wm);
                    for (int gi = nextOn(p, x); gi >= 0; gi = nextOn(p, x)) {
                        if (!readyIn(p, gi) || __builtin_popcountll(b.mask | maskOf[gi]) > maxQubits) break;
                        b.mask |= maskOf[gi];
                        b.gates.push_back(gi);
                        for (uint64_t m = maskOf[gi]; m; m &= m - 1) ++p[__builtin_ctzll(m)];
                        progress = true;
                    }
                }
            }
            if (b.gates.size() > best.gates.size()) {
                best = std::move(b);
                bestPtr = std::move(p);
            }
        }
        if (best.gates.empty()) {
            // a ready gate on more than maxQubits qubits: a block of its own
            best.mask = maskOf[firstReady];
            best.gates.push_back(firstReady);
            bestPtr = ptr;
            for (uint64_t m = best.mask; m; m &= m - 1) ++bestPtr[__builtin_ctzll(m)];
        }
        remaining -= best.gates.size();
        ptr = std::move(bestPtr);
        c->blocks.push_back(std::move(best));
    }
}

int fuseCircuit(qmxCircuit *c, int maxQubits) {
    c->releaseBlocks();
    c->fusedQubits = maxQubits;
    c->fusedOps = (int)c->ops.size();
    std::vector<int> seg;  // gates since the latest barrier
    for (int gi = 0; gi < (int)c->ops.size(); ++gi) {
        const Op &o = c->ops[gi];
        if (o.barrier) {
            fuseSegment(c, seg, maxQubits);
            seg.clear();
            Block nb;
            nb.barrierOp = gi;
            c->blocks.push_back(std::move(nb));
            continue;
        }
        if (o.gate.kind == G_NONE) continue;  // noise or unsupported: nothing on a state vector
        seg.push_back(gi);
    }
    fuseSegment(c, seg, maxQubits);
    // Blocks of at most 5 qubits are the steps qmxCircuitStep reports; on registers of
    // 9 qubits and more those of several gates name exactly 5, the extra ones (identity)
    // from the top. What runs is planned anew (sweepsOf).
    if (maxQubits == 5 && c->numQubits >= 9) {
        for (Block &b : c->blocks) {
            if (b.barrierOp >= 0 || b.gates.size() < 2) continue;
            for (int qb = c->numQubits - 1; qb >= 0 && __builtin_popcountll(b.mask) < 5; --qb)
                b.mask |= 1ull << qb;
        }
    }
    // the matrices of blocks that applications read (a lone gate keeps its own kernel);
    // a step's is formed when it is asked for (qmxCircuitStep)
    const bool applied = maxQubits != qmx::kSweepBlockQubits && qmx::sweepSupported(c->numQubits);
    for (Block &b : c->blocks) {
        if (b.barrierOp >= 0) continue;
        listTargets(b);
        if (applied && b.gates.size() > 1) buildBlockMatrix(*c, b);
    }
    return (int)c->blocks.size();
}

}  // namespace

#define CIRCUIT_TRY try {
#define CIRCUIT_CATCH(ret)              \
    }                                   \
    catch (const qmx::InputError &) {   \
        return ret;                     \
    }

extern "C" {

qmxCircuit *qmxCircuitCreate(int numQubits) {
    CIRCUIT_TRY
    qv::numQubitsInQureg(numQubits, __func__);
    auto *c = new qmxCircuit;
    c->numQubits = numQubits;
    std::memset(&c->shape, 0, sizeof c->shape);
    c->shape.numQubitsRepresented = numQubits;
    c->shape.numQubitsInStateVec = numQubits;
    c->shape.numAmpsPerChunk = c->shape.numAmpsTotal = numQubits < 63 ? 1LL << numQubits : 0;
    return c;
    CIRCUIT_CATCH(nullptr)
}

void qmxCircuitDestroy(qmxCircuit *c) { delete c; }

int qmxCircuitNumGates(const qmxCircuit *c) { return (int)c->ops.size(); }

void qmxCircuitAddOperation(qmxCircuit *c, int operation, const int *qubits, int numQubits, qreal param) {
    CIRCUIT_TRY
    recordBasic(c, operation, qubits, numQubits, (double)param, __func__);
    CIRCUIT_CATCH()
}

void qmxCircuitSetNoiseAfterGate(qmxCircuit *c, qmxNoiseAfterGate noise) {
    CIRCUIT_TRY
    noiseParams(noise, __func__);
    c->noise = noise;
    CIRCUIT_CATCH()
}

void qmxCircuitCompactUnitary(qmxCircuit *c, int target, Complex a, Complex b) {
    CIRCUIT_TRY
    qv::target(c->shape, target, __func__);
    qv::unitaryComplexPair(a, b, __func__);
    Op o;
    o.code = OP_COMPACT_UNITARY;
    o.target = target;
    o.alpha = a;
    o.beta = b;
    setCompact(o.gate, target, 0, Cplx{a.real, a.imag}, Cplx{b.real, b.imag});
    c->ops.push_back(std::move(o));
    CIRCUIT_CATCH()
}

void qmxCircuitUnitary(qmxCircuit *c, int target, ComplexMatrix2 u) {
    CIRCUIT_TRY
    qv::target(c->shape, target, __func__);
    qv::oneQubitUnitary(u, __func__);
    Op o;
    o.code = OP_UNITARY;
    o.target = target;
    o.m2 = u;
    setMatrix2(o.gate, target, 0, Cplx{u.real[0][0], u.imag[0][0]}, Cplx{u.real[0][1], u.imag[0][1]},
               Cplx{u.real[1][0], u.imag[1][0]}, Cplx{u.real[1][1], u.imag[1][1]});
    c->ops.push_back(std::move(o));
    CIRCUIT_CATCH()
}

// rotateZ as QuEST applies it: compactUnitary with alpha = e^{-iθ/2}, beta = 0
void qmxCircuitRotateZ(qmxCircuit *c, int target, qreal angle) {
    CIRCUIT_TRY
    qv::target(c->shape, target, __func__);
    Op o;
    o.code = OP_ROTATE_Z;
    o.target = target;
    o.param = angle;
    setRotation(o.gate, target, 0, angle, 0, 0, 1);
    c->ops.push_back(std::move(o));
    CIRCUIT_CATCH()
}

void qmxCircuitControlledNot(qmxCircuit *c, int control, int target) {
    CIRCUIT_TRY
    const int qs[2] = {control, target};
    recordBasic(c, QMX_OP_CX, qs, 2, 0.0, __func__);
    CIRCUIT_CATCH()
}

void qmxCircuitMultiControlledUnitary(qmxCircuit *c, int *controls, int numControls, int target, ComplexMatrix2 u) {
    CIRCUIT_TRY
    qv::multiControlsTarget(c->shape, controls, numControls, target, __func__);
    qv::oneQubitUnitary(u, __func__);
    Op o;
    o.code = OP_MULTI_CONTROLLED_UNITARY;
    o.qubits.assign(controls, controls + numControls);
    o.target = target;
    o.m2 = u;
    uint64_t m = 0;
    for (int i = 0; i < numControls; ++i) m |= 1ull << controls[i];
    setMatrix2(o.gate, target, m, Cplx{u.real[0][0], u.imag[0][0]}, Cplx{u.real[0][1], u.imag[0][1]},
               Cplx{u.real[1][0], u.imag[1][0]}, Cplx{u.real[1][1], u.imag[1][1]});
    c->ops.push_back(std::move(o));
    CIRCUIT_CATCH()
}

void qmxCircuitMultiQubitUnitary(qmxCircuit *c, int *targs, int numTargs, const qreal *re, const qreal *im) {
    CIRCUIT_TRY
    qv::multiTargets(c->shape, targs, numTargs, __func__);
    qv::check(numTargs <= 10, qv::E_INVALID_NUM_TARGETS, __func__);
    Op o;
    o.code = OP_MULTI_QUBIT_UNITARY;
    o.qubits.assign(targs, targs + numTargs);
    const size_t dim = 1ull << numTargs;
    o.mN = createComplexMatrixN(numTargs);
    for (size_t r = 0; r < dim; ++r)
        for (size_t col = 0; col < dim; ++col) {
            o.mN.real[r][col] = re[r * dim + col];
            o.mN.imag[r][col] = im[r * dim + col];
        }
    try {
        qv::multiQubitUnitary(c->shape, o.mN, numTargs, __func__);
    } catch (...) {  // also a caller's throwing error hook
        destroyComplexMatrixN(o.mN);
        throw;
    }
    o.gate.kind = G_MATRIXN;
    o.gate.targs = o.qubits;
    o.gate.u.resize(dim * dim);
    for (size_t e = 0; e < dim * dim; ++e) o.gate.u[e] = Cplx{re[e], im[e]};
    c->ops.push_back(std::move(o));
    CIRCUIT_CATCH()
}

int qmxCircuitFuse(qmxCircuit *c, int maxQubits) {
    CIRCUIT_TRY
    if (maxQubits < 1 || maxQubits > 10)
        qv::raise("Invalid block size. Fused blocks span at least 1 and at most 10 qubits.", __func__);
    return fuseCircuit(c, maxQubits);
    CIRCUIT_CATCH(0)
}

int qmxCircuitStep(const qmxCircuit *c, int step, int *targs, qreal *re, qreal *im) {
    if (step < 0 || step >= (int)c->blocks.size()) return -1;
    const Block &b = c->blocks[step];
    if (b.barrierOp >= 0) return 0;
    const int k = (int)b.targs.size();
    const size_t dim = 1ull << k;
    if (targs)
        for (int j = 0; j < k; ++j) targs[j] = b.targs[j];
    if (re && im) {
        Block formed;  // of the same gates; a step that runs has its matrix already
        if (b.u.empty()) {
            formed.targs = b.targs;
            formed.gates = b.gates;
            buildBlockMatrix(*c, formed);
        }
        const std::vector<Cplx> &u = b.u.empty() ? formed.u : b.u;
        for (size_t e = 0; e < dim * dim; ++e) {
            re[e] = (qreal)u[e].re;
            im[e] = (qreal)u[e].im;
        }
    }
    return k;
}

int qmxCircuitSweepBlock(qmxCircuit *c, int precision, int sweep, int block, int *targs, qreal *re, qreal *im) {
    CIRCUIT_TRY
    if (precision != QMX_PREC_FP64 && precision != QMX_PREC_FP32) return -1;
    const CircuitSweeps *s = sweepsOf(c, precision == QMX_PREC_FP64 ? qmx::FP64 : qmx::FP32);
    if (!s) return -1;
    if (sweep < 0 || sweep >= (int)s->plan.sweeps.size()) return -1;
    const qmx::Sweep &w = s->plan.sweeps[sweep];
    if (block < 0 || block >= (w.lone >= 0 ? 1 : w.numBlocks)) return 0;
    Block b;
    if (w.lone >= 0) {
        b.gates.push_back(s->list.op[w.lone]);
        b.mask = s->list.gates[w.lone].mask();
    } else {
        const qmx::SweepBlock &sb = s->plan.blocks[w.firstBlock + block];
        for (int g = 0; g < sb.numGates; ++g) b.gates.push_back(s->list.op[s->plan.order[sb.firstGate + g]]);
        for (int j = 0; j < sb.k; ++j)
            if (sb.targs[j] < c->numQubits) b.mask |= 1ull << sb.targs[j];
    }
    listTargets(b);
    const int k = (int)b.targs.size();
    const size_t dim = 1ull << k;
    if (targs)
        for (int j = 0; j < k; ++j) targs[j] = b.targs[j];
    if (re && im) buildBlockMatrix(*c, b);
    if (re && im)
        for (size_t e = 0; e < dim * dim; ++e) {
            re[e] = (qreal)b.u[e].re;
            im[e] = (qreal)b.u[e].im;
        }
    return k;
    CIRCUIT_CATCH(-1)
}

int qmxCircuitNumBlocks(const qmxCircuit *c) {
    int n = 0;
    for (const Block &b : c->blocks) n += b.barrierOp < 0;
    return n;
}

qreal qmxCircuitApply(Qureg qureg, qmxCircuit *c, int fused) {
    CIRCUIT_TRY
    checkRegister(c, qureg, __func__);
    return (qreal)applyCircuit(qureg, c, fused);
    CIRCUIT_CATCH(0)
}

qreal qmxApplyOperations(Qureg qureg, const qmxBasicOperation *ops, int numOps, const qmxNoiseAfterGate *noise,
                         int fuseQubits) {
    CIRCUIT_TRY
    qmxCircuit c;
    c.numQubits = qureg.numQubitsRepresented;
    std::memset(&c.shape, 0, sizeof c.shape);
    c.shape.numQubitsRepresented = c.numQubits;
    c.shape.numQubitsInStateVec = c.numQubits;
    c.shape.numAmpsPerChunk = c.shape.numAmpsTotal = c.numQubits < 63 ? 1LL << c.numQubits : 0;
    checkRegister(&c, qureg, __func__);
    if (numOps < 0) qv::raise("Invalid number of operations. Must be >=0.", __func__);
    if (noise) {
        noiseParams(*noise, __func__);
        c.noise = *noise;
    }
    // Lists that need no recording (one LDS circuit, or sweeps): straight from the
    // caller's list to the kernels' gates. On density registers the list, noise
    // included, is planned as a whole over the 2n row and column bits; one pass for
    // each two composed pairs of qubits, what API calls make of it, costs 4 us of host
    // time an operation and fills a pass with two blocks: 7 qubits FP64, 60 operations
    // with noise and 8 reads, 1380 us that way and 240 in sweeps; 13 qubits FP32, 120
    // operations and 14 reads, 27 passes in 6.9 ms and 12 sweeps in 3.6.
    qmx::QuregDev *d = qmx::dev(qureg);
    const bool small = qmx::smallCircuitSupported(d);
    const bool sweeps = fuseQubits == qmx::kSweepBlockQubits && qmx::sweepSupported(d->numQubits);
    double prob = 1.0;
    auto stop = [&](int i) {
        Op o;
        o.code = ops[i].operation;
        o.qubits.assign(ops[i].qubits, ops[i].qubits + std::max(0, ops[i].numQubits));
        o.param = (double)ops[i].param;
        prob *= runOp(qureg, o);
    };
    const char *badFuse = "Invalid block size. Fused blocks span at least 1 and at most 10 qubits.";
    if (qureg.isDensityMatrix && fuseQubits >= 0 && fuseQubits <= 10) {
        for (int i = 0; i < numOps; ++i)
            checkBasic(c.shape, ops[i].operation, ops[i].qubits, ops[i].numQubits, (double)ops[i].param, __func__);
        DensityList dl(c.numQubits);
        bool taken = true;
        for (int i = 0; i < numOps && taken; ++i)
            taken = dl.add(i, ops[i].operation, ops[i].qubits, ops[i].numQubits, (double)ops[i].param,
                           hasNoise(c.noise) ? &c.noise : nullptr);
        if (taken) {
            if (small)
                runSmall(d, dl.l, stop);
            else
                runSweepsOnce(d, dl.l, stop);
            qmx::densCountSweeps(0, dl.operations);
            return (qreal)prob;
        }
    } else if (!qureg.isDensityMatrix && (small || sweeps)) {
        GateList l;
        l.gates.reserve(numOps);
        int last[64];
        std::fill(last, last + 64, -1);
        for (int i = 0; i < numOps; ++i) {
            const qmxBasicOperation &o = ops[i];
            checkBasic(c.shape, o.operation, o.qubits, o.numQubits, (double)o.param, __func__);
            FlatGate g;
            if (!undispatched(o.operation) && basicGate(o.operation, o.qubits, (double)o.param, g)) {
                appendGate(l.gates, last, g);
            } else if (o.operation == QMX_OP_CC || (fuseQubits == 0 && undispatched(o.operation))) {
                l.stops.push_back({(int)l.gates.size(), i});
                std::fill(last, last + 64, -1);
            }
        }
        if (fuseQubits < 0 || fuseQubits > 10) qv::raise(badFuse, __func__);
        // a fused list without gates and collapses goes on unfused below, where each
        // undispatched operation says so
        if (!l.gates.empty() || !l.stops.empty()) {
            std::vector<Cplx> room;
            if (c.numQubits == 2 && fuseQubits >= 2) composePairs(l, room);
            if (small)
                runSmall(d, l, stop);
            else
                runSweepsOnce(d, l, stop);
            return (qreal)prob;
        }
    }
    for (int i = 0; i < numOps; ++i)
        recordBasic(&c, ops[i].operation, ops[i].qubits, ops[i].numQubits, (double)ops[i].param, __func__);
    if (fuseQubits != 0) {
        if (fuseQubits < 1 || fuseQubits > 10) qv::raise(badFuse, __func__);
        if (!qureg.isDensityMatrix) fuseCircuit(&c, fuseQubits);
    }
    return (qreal)applyCircuit(qureg, &c, fuseQubits != 0);
    CIRCUIT_CATCH(0)
}

qreal qmxMaxAbsDiff(Qureg a, Qureg b) { return qmx::maxAbsDiff(qmx::dev(a), qmx::dev(b)); }

}  // extern "C"
