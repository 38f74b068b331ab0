// Runs of unitaries applied many to a sweep: the planner (qmx_plan.cpp, host
// only) and the kernels that carry a plan out (qmx_sweep.hip).
#pragma once

#include <vector>

#include "qmx_internal.h"

namespace qmx {

// One operation on a state vector in matrix form. A density register is the
// vector of its 2n row and column bits: a unitary is a gate on its row bits and the
// conjugate one on its column bits. CHANNEL is a one-qubit channel with real maps of
// its qubit's diagonal entries, (x00, x11) -> (d00 x00 + d01 x11, d10 x00 + d11 x11),
// and off-diagonal ones, (x01, x10) -> (f x01 + g x10, g x01 + f x10): target = the
// row bit, k = the column bit, u = {(f, g), (d00, d01), (d10, d11), (fLo, d00Lo)}, lo =
// d11Lo: what rounding f, d00 and d11 left over, where channels were joined into one.
struct FlatGate {
    enum Kind { MATRIX2 = 0, NOT = 1, MATRIXN = 2, CHANNEL = 3 };
    int kind = MATRIX2;
    int target = 0;                // MATRIX2, NOT
    uint64_t ctrl = 0;             // controls (all kinds; acts where they are 1)
    Cplx u[4] = {};                // MATRIX2, row-major
    int k = 0;                     // MATRIXN: targets (targs[0] = least significant bit), 2^k x 2^k
    const int *targs = nullptr;
    const Cplx *uN = nullptr;
    float lo = 0;                  // CHANNEL
    uint64_t mask() const {
        uint64_t m = ctrl;
        if (kind == MATRIXN)
            for (int j = 0; j < k; ++j) m |= 1ull << targs[j];
        else
            m |= 1ull << target;
        if (kind == CHANNEL) m |= 1ull << k;
        return m;
    }
};

// ---- large registers: tiles of 2^sweepTileBits amplitudes -----------------------
// A sweep reads and writes the register once. Its tile is sweepTileBits qubits:
// the lowest sweepLowBits (whole 128 B lines) and others; every gate of the sweep
// acts inside the tile, as blocks of 4 or 5 qubits applied one after another in LDS.
// 12 qubits, and 11 where tiles of 12 would leave CUs without a workgroup: up to 19
// qubits a tile of half the size takes half the time a block, for one sweep more in
// six (300 random operations on 17 qubits).
constexpr int kSweepTileBits = 12;
constexpr int sweepTileBits(int numQubits) { return numQubits < 20 ? kSweepTileBits - 1 : kSweepTileBits; }
constexpr int kSweepBlockQubits = 5;
constexpr int kSweepMaxBlocks = 64;    // blocks of one sweep
constexpr int kSweepMaxWeight = 512;   // gates of one block (a MATRIXN of more than two qubits counts as 4^k / 16)
inline int sweepLowBits(int prec) { return prec == FP64 ? 3 : 4; }
// registers the sweeps serve (smaller ones are one tile: see smallCircuit)
constexpr int kSmallCircuitQubits = 12;
inline bool sweepSupported(int numQubits) { return numQubits > kSmallCircuitQubits; }

struct SweepBlock {
    int k;                             // 4 or 5
    int targs[kSweepBlockQubits];      // qubits, ascending (targs[0] = least significant matrix bit)
    int firstGate, numGates;           // range of SweepPlan::order
};
struct Sweep {
    uint64_t tile;                     // the tile's qubits
    int firstBlock, numBlocks;
    int lone;                          // >= 0: this gate on its own kernel instead
};
struct SweepPlan {
    std::vector<int> order;            // gate indices, block by block
    std::vector<SweepBlock> blocks;
    std::vector<Sweep> sweeps;
};
// What is planned for: registers of `bits` bits, tiles of `tileBits` that always hold
// the lowest `lowBits`. density: bits b and b + bits/2 belong together (a qubit's
// row and column bit), so windows take them in pairs.
struct SweepShape {
    int bits, lowBits, tileBits;
    bool density;
    int maxBlocks;                     // of one sweep
};
inline SweepShape sweepShape(int numBits, int prec, bool density) {
    // density tiles: a qubit is two bits, so 12 hold twice the pairs of 8
    return SweepShape{numBits, sweepLowBits(prec), density ? kSweepTileBits : sweepTileBits(numBits), density,
                      kSweepMaxBlocks};
}
// Appends the sweeps of gates[0 .. count) to `plan` (gate indices offset by `base`).
void planSweeps(const SweepShape &shape, const FlatGate *gates, int count, int base, SweepPlan &plan);

// A plan's blocks on the device (matrices built there from the gates).
struct SweepProgram;
SweepProgram *sweepProgramCreate(int prec, const SweepPlan &plan, const FlatGate *gates);
void sweepProgramFree(SweepProgram *p);
// sweeps [first, last) of the plan
void sweepProgramRun(QuregDev *q, const SweepProgram *p, const SweepPlan &plan, const FlatGate *gates, int first,
                     int last);
// the whole plan once, through the library's workspace (nothing allocated per call)
void sweepRunOnce(QuregDev *q, const SweepPlan &plan, const FlatGate *gates);

// one gate on its own kernel
void applyFlatGate(QuregDev *q, const FlatGate &g);

// ---- small registers: the whole register in one workgroup's LDS -----------------
// A state vector of at most kSmallCircuitQubits is one tile, of at least 9 bits (16
// groups of a 5-qubit block; bits past the register are zeros), in FP64 for both
// storage precisions; sweeps of any number of blocks.
inline SweepShape smallShape(int numQubits) {
    const int bits = numQubits < 9 ? 9 : numQubits;
    return SweepShape{bits, sweepLowBits(FP64), bits, false, 1 << 30};
}
inline bool smallStateVector(const QuregDev *q) { return !q->isDensity && q->numQubits <= kSmallCircuitQubits; }

// Gate lists applied once run gate by gate.
// A density operation is three or four steps of the LDS kernel (rows, columns,
// channels; 0.8 us each), where a tile of 12 bits takes whole blocks of them: 6
// qubits, 82 operations with their noise and reads, FP64 379 us there and 216 in
// sweeps. In FP32 it would be 378 and 198, but the LDS kernel's FP64 arithmetic keeps
// 2.2e-7 from the 64-bit state where sweeps leave 3.5e-7 (and one pass for each pair
// of qubits 2.4e-7).
inline bool smallCircuitSupported(const QuregDev *q) {
    return q->numQubits <= (q->isDensity && q->prec == FP64 ? 10 : kSmallCircuitQubits);
}
// gates[0 .. count) in order, one launch per 4096 of them; no MATRIXN
void smallCircuit(QuregDev *q, const FlatGate *gates, int count);

}  // namespace qmx
