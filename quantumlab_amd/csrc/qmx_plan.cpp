// The sweep planner: which gates of a list share one read and write of the
// register. Gates on disjoint qubits commute, so any order that keeps each
// qubit's gates in sequence is the same circuit.
//
// Two levels, both greedy. A sweep takes the tile (the lowest qubits and a window
// of others) that absorbs the most gates; inside it, the gates become blocks of 4
// or 5 qubits, each the window with the most gates for its cost on the matrix
// cores (a 5-qubit block costs twice a 4-qubit one). On the 30-qubit brick period
// of five layers (230 gates) this makes 6 to 8 sweeps of 24 to 26 blocks, worth 12.5 to
// 15 5-qubit blocks of arithmetic, where one sweep per 5-qubit block takes 16 of each.
#include <algorithm>

#include "qmx_sweep.h"

namespace qmx {

namespace {

int popcount(uint64_t x) { return __builtin_popcountll(x); }

int weightOf(const FlatGate &g) { return g.kind == FlatGate::MATRIXN && g.k > 2 ? (1 << (2 * g.k)) / 16 : 1; }

// Planning order of a register's bits: itself, or for density registers row and
// column bit of a qubit side by side (bit q to 2q, bit q + bits/2 to 2q + 1), so that
// a window of consecutive bits is a run of whole qubits.
uint64_t toOrder(const SweepShape &s, uint64_t mask) {
    if (!s.density) return mask;
    const int half = s.bits / 2;
    uint64_t m = 0;
    for (; mask; mask &= mask - 1) {
        const int b = __builtin_ctzll(mask);
        m |= 1ull << (b < half ? 2 * b : 2 * (b - half) + 1);
    }
    return m;
}
uint64_t fromOrder(const SweepShape &s, uint64_t mask) {
    if (!s.density) return mask;
    uint64_t m = 0;
    for (; mask; mask &= mask - 1) {
        const int b = __builtin_ctzll(mask);
        m |= 1ull << (b / 2 + (b & 1 ? s.bits / 2 : 0));
    }
    return m;
}

struct Item {
    int id;          // index into the gate list
    uint64_t mask;
    int weight;
};

// Walk `rem` in order, taking every gate inside `window` that no gate left behind
// precedes on one of its qubits, up to `maxWeight`; returns how many, and their
// places in `rem` through `taken` when given.
int absorb(const std::vector<Item> &rem, uint64_t window, int maxWeight, std::vector<int> *taken) {
    uint64_t blocked = 0;
    int count = 0, weight = 0;
    for (int i = 0; i < (int)rem.size(); ++i) {
        const uint64_t m = rem[i].mask;
        if (!(m & blocked) && !(m & ~window) && weight + rem[i].weight <= maxWeight) {
            ++count;
            weight += rem[i].weight;
            if (taken) taken->push_back(i);
            continue;
        }
        blocked |= m;
        if (!(window & ~blocked)) break;
    }
    return count;
}

// the unblocked gate that adds the fewest qubits to `touched` within `maxQubits`; 0 if none
uint64_t growth(const std::vector<Item> &rem, uint64_t touched, int maxQubits, int widest) {
    uint64_t blocked = 0, best = 0;
    int bestNew = 65;
    uint64_t all = 0;
    for (const Item &it : rem) all |= it.mask;
    for (const Item &it : rem) {
        const uint64_t m = it.mask;
        if (!(m & blocked) && (m & ~touched) && popcount(m) <= widest) {
            const int add = popcount(m & ~touched);
            if (add < bestNew && popcount(touched | m) <= maxQubits) {
                bestNew = add;
                best = m;
            }
        }
        // gates inside `touched` have been taken: they block nobody
        if ((m & blocked) || (m & ~touched)) blocked |= m;
        if (!(all & ~blocked)) break;
    }
    return best;
}

// add the lowest qubits below n to `mask` until it has k
uint64_t padLow(uint64_t mask, int n, int k) {
    for (int b = 0; b < n && popcount(mask) < k; ++b) mask |= 1ull << b;
    return mask;
}

void remove(std::vector<Item> &rem, const std::vector<int> &taken) {
    size_t w = 0, t = 0;
    for (size_t i = 0; i < rem.size(); ++i) {
        if (t < taken.size() && (int)i == taken[t]) {
            ++t;
            continue;
        }
        rem[w++] = rem[i];
    }
    rem.resize(w);
}

// the gates of one tile as blocks, appended to the plan; gate ids offset by `base`
void planBlocks(std::vector<Item> rem, int base, SweepPlan &plan, std::vector<uint64_t> &blockMasks) {
    std::vector<int> taken;
    while (!rem.empty()) {
        uint64_t bits = 0;
        for (const Item &it : rem) bits |= it.mask;
        int pos[64], nb = 0;
        for (uint64_t m = bits; m; m &= m - 1) pos[nb++] = __builtin_ctzll(m);
        double best = 0;
        uint64_t window = 0;
        for (int k = kSweepBlockQubits - 1; k <= kSweepBlockQubits; ++k) {
            // matrix work 1 (4 qubits) or 2 (5), and a quarter for the LDS round trip
            const double cost = k == kSweepBlockQubits ? 2.25 : 1.25;
            for (int s = 0; s + std::min(k, nb) <= nb; ++s) {
                uint64_t w = 0;
                for (int j = s; j < s + std::min(k, nb); ++j) w |= 1ull << pos[j];
                const double value = absorb(rem, w, kSweepMaxWeight, nullptr) / cost;
                if (value > best) {
                    best = value;
                    window = w;
                }
            }
        }
        if (best == 0) window = rem[0].mask;  // its qubits are too far apart for a window
        taken.clear();
        absorb(rem, window, kSweepMaxWeight, &taken);
        uint64_t touched = 0;
        for (int i : taken) touched |= rem[i].mask;
        const int k = popcount(touched) > kSweepBlockQubits - 1 ? kSweepBlockQubits : kSweepBlockQubits - 1;
        while (uint64_t g = growth(rem, touched, k, kSweepBlockQubits)) {
            touched |= g;
            taken.clear();
            absorb(rem, touched, kSweepMaxWeight, &taken);
            if ((int)taken.size() == 0) break;
            uint64_t now = 0;
            for (int i : taken) now |= rem[i].mask;
            if ((now | touched) == touched && !(now & g)) break;  // the weight limit stopped it
        }
        SweepBlock b{};
        b.k = k;
        b.firstGate = (int)plan.order.size();
        b.numGates = (int)taken.size();
        for (int i : taken) plan.order.push_back(base + rem[i].id);
        blockMasks.push_back(touched);
        plan.blocks.push_back(b);
        remove(rem, taken);
    }
}

}  // namespace

void planSweeps(const SweepShape &shape, const FlatGate *gates, int count, int base, SweepPlan &plan) {
    const int n = shape.bits;
    std::vector<Item> rem(count);
    for (int i = 0; i < count; ++i) rem[i] = Item{i, toOrder(shape, gates[i].mask()), weightOf(gates[i])};
    const int tileBits = std::min(shape.tileBits, n), lowBits = std::min(shape.lowBits, n);
    const uint64_t low = toOrder(shape, (1ull << lowBits) - 1ull);
    const int firstStart = shape.density ? 0 : lowBits, step = shape.density ? 2 : 1;
    std::vector<int> taken;
    std::vector<Item> mine;
    std::vector<uint64_t> blockMasks;
    // gates wider than a block run on their own kernels: no tile takes them
    auto blockable = [&](const Item &it) { return popcount(it.mask) <= kSweepBlockQubits; };
    for (Item &it : rem)
        if (!blockable(it)) it.weight = 1 << 30;
    while (!rem.empty()) {
        // the lowest qubits and a window of consecutive others
        uint64_t window = 0;
        int best = 0;
        for (int s = firstStart; s == firstStart || s + tileBits - lowBits <= n; s += step) {
            uint64_t w = low;
            for (int b = s; b < n && popcount(w) < tileBits; ++b) w |= 1ull << b;
            w = padLow(w, n, tileBits);
            const int got = absorb(rem, w, 1 << 28, nullptr);
            if (got > best) {
                best = got;
                window = w;
            }
        }
        taken.clear();
        uint64_t touched = low;
        if (best == 0) {
            // the first gate left; its qubits are too far apart for a window
            if (blockable(rem[0]) && popcount(low | rem[0].mask) <= tileBits) touched |= rem[0].mask;
        } else {
            absorb(rem, window, 1 << 28, &taken);
            for (int i : taken) touched |= rem[i].mask;
        }
        // qubits the window left unused go to the gates that need the fewest
        while (uint64_t g = growth(rem, touched, tileBits, kSweepBlockQubits)) touched |= g;
        taken.clear();
        absorb(rem, touched, 1 << 28, &taken);
        if (taken.size() <= 1) {
            const int at = taken.empty() ? 0 : taken[0];
            plan.sweeps.push_back(Sweep{0, 0, 0, base + rem[at].id});
            taken.assign(1, at);
            remove(rem, taken);
            continue;
        }
        mine.clear();
        for (int i : taken) mine.push_back(rem[i]);
        remove(rem, taken);
        const uint64_t tile = padLow(touched, n, tileBits);
        const int firstBlock = (int)plan.blocks.size();
        blockMasks.clear();
        planBlocks(std::move(mine), base, plan, blockMasks);
        mine = {};
        // pad to 4 or 5 qubits from the tile's top: identity on the extra ones
        for (size_t i = 0; i < blockMasks.size(); ++i) {
            SweepBlock &b = plan.blocks[firstBlock + i];
            uint64_t m = blockMasks[i];
            for (int q = 63; q >= 0 && popcount(m) < b.k; --q)
                if ((tile >> q) & 1) m |= 1ull << q;
            m = fromOrder(shape, m);
            int j = 0;
            for (uint64_t x = m; x; x &= x - 1) b.targs[j++] = __builtin_ctzll(x);
        }
        for (int b = firstBlock, n = 0; b < (int)plan.blocks.size(); b += n) {
            n = std::min(shape.maxBlocks, (int)plan.blocks.size() - b);
            plan.sweeps.push_back(Sweep{fromOrder(shape, tile), b, n, -1});
        }
    }
}

}  // namespace qmx
