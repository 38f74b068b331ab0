// Sweeps of many gates: LDS tiles with dense 4- and 5-qubit blocks on the matrix
// cores (registers of more than kSweepTileBits qubits), and whole circuits in one
// workgroup's LDS (smaller ones).
//
// Tiles. A workgroup owns a tile of 2^12 amplitudes (32 KiB in FP32, 64 KiB in
// FP64): the sweep's 12 qubits, of which the lowest 4 (FP32) or 3 (FP64) make
// every memory run a whole 128 B line. It loads the tile into LDS, applies the
// sweep's blocks one after another there, and stores it. A block U on k = 4 or 5
// of the tile's qubits multiplies 16 groups of 2^k amplitudes at a time as three
// real products (P1 = Ur Xr, P2 = Ui Xi, P3 = (Ur + Ui)(Xr + Xi); Re = P1 - P2,
// Im = P3 - P1 - P2) of v_mfma_f32_16x16x4f32 / v_mfma_f64_16x16x4f64 steps.
//
// Why blocks share a tile: one 5-qubit block a sweep moves 16 B (FP32) for 192
// flops an amplitude, which HBM takes 1.7 times as long for as the matrix cores
// do; two or three blocks a sweep bring the two to the same time. 4-qubit blocks
// take half a 5-qubit block's arithmetic and absorb two thirds of its gates, so
// the planner prefers them. Measured per five-layer brick period: MEASURED_TABLE
//
// Operand placement (16x16x4, wave64; lane = 16 kq + col):
//   A: lane holds U[r][4 st + kq] of its row r, one fragment per step st;
//   B: lane holds amplitude (group col, combination 4 st + kq);
//   D: element v of row tile h is row 16 h + 4 kq + v in FP32, 16 h + 4 v + kq in
//      FP64. FP32 fragments hold their rows in the order that makes it 16 h + 4 v
//      + kq there too: a lane's output v of tile h is then the combination of
//      its input step st = 4 h + v, and goes back to the slot that input came from.
//
// LDS slot of tile element e: e with its higher bits folded onto the lowest 4
// (FP32: 16 slots of 8 B are one cycle of the banks) or 3 (FP64), an XOR per
// group of 4 (3) bits. A wave's 16 columns take tile bits of different residues
// modulo 4 (3) where the block leaves them, so one operand read touches all banks
// once whichever qubits the block has.
#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "qmx_device.h"
#include "qmx_sweep.h"

namespace qmx {

namespace {

typedef float f4 __attribute__((ext_vector_type(4)));
typedef double d2 __attribute__((ext_vector_type(2)));
typedef double d4 __attribute__((ext_vector_type(4)));

constexpr int kTB = kSweepTileBits;
constexpr int kWaves = kBlock / 64;

// ---- block matrices, built on the device ---------------------------------------
struct GateDev {
    int kind;            // FlatGate::Kind
    int t;               // target, a bit of the block's index
    unsigned ctrl;       // controls, bits of the block's index
    int k;               // MATRIXN
    int lt[kSweepBlockQubits];
    int mat;             // MATRIXN: its matrix (entry offset)
    Amp<double> u[4];
};
struct BuildDev {
    int firstGate, numGates, k, pad;
};

// fragments of one block: FP32 3 x 16 (k = 5) or 3 x 4 values a lane, FP64 16 or
// 4 complex ones; every block has the room of the largest
constexpr size_t kBlockBytes = 16384;

template <typename T> struct Frag;
template <> struct Frag<float> { typedef f4 V; };
template <> struct Frag<double> { typedef d2 V; };

// One workgroup per block: the product of its gates in FP64, column by column of
// the identity, in LDS; then the matrix-core fragments. The gates arrive as the
// host recorded them, so a list of any length costs one small copy instead of a
// matrix per block (on the host a block of ten gates took ~25 us).
template <typename T>
__global__ void __launch_bounds__(kBlock) kBuildBlocks(const BuildDev *__restrict__ todo,
                                                       const GateDev *__restrict__ gates,
                                                       const Amp<double> *__restrict__ mats, char *__restrict__ out) {
    __shared__ Amp<double> buf[2][32 * 32];
    const BuildDev b = todo[blockIdx.x];
    const int k = b.k, dim = 1 << k, tid = threadIdx.x;
    Amp<double> *M = buf[0], *N = buf[1];
    for (int i = tid; i < dim * dim; i += kBlock) M[i] = Amp<double>{(i >> k) == (i & (dim - 1)) ? 1.0 : 0.0, 0.0};
    __syncthreads();
    for (int g = 0; g < b.numGates; ++g) {
        const GateDev &G = gates[b.firstGate + g];
        const unsigned ctrl = G.ctrl;
        if (G.kind != FlatGate::MATRIXN) {
            const int t = G.t;
            const bool isNot = G.kind == FlatGate::NOT;
            const Amp<double> u0 = G.u[0], u1 = G.u[1], u2 = G.u[2], u3 = G.u[3];
            for (int i = tid; i < dim * dim / 2; i += kBlock) {
                const int col = i & (dim - 1);
                const unsigned r0 = (unsigned)insertZero((uint64_t)(i >> k), t), r1 = r0 | (1u << t);
                if ((r0 & ctrl) != ctrl) continue;
                const Amp<double> x = M[r0 * dim + col], y = M[r1 * dim + col];
                if (isNot) {
                    M[r0 * dim + col] = y;
                    M[r1 * dim + col] = x;
                } else {
                    M[r0 * dim + col] = Amp<double>{u0.x * x.x - u0.y * x.y + u1.x * y.x - u1.y * y.y,
                                                    u0.x * x.y + u0.y * x.x + u1.x * y.y + u1.y * y.x};
                    M[r1 * dim + col] = Amp<double>{u2.x * x.x - u2.y * x.y + u3.x * y.x - u3.y * y.y,
                                                    u2.x * x.y + u2.y * x.x + u3.x * y.y + u3.y * y.x};
                }
            }
            __syncthreads();
            continue;
        }
        const int gk = G.k, gd = 1 << gk;
        const Amp<double> *U = mats + G.mat;
        for (int i = tid; i < dim * dim; i += kBlock) {
            const int col = i & (dim - 1);
            const unsigned r = (unsigned)(i >> k);
            Amp<double> s = M[r * dim + col];
            if ((r & ctrl) == ctrl) {
                unsigned base = r;
                int row = 0;
                for (int j = 0; j < gk; ++j) {
                    row |= (int)((r >> G.lt[j]) & 1u) << j;
                    base &= ~(1u << G.lt[j]);
                }
                s = Amp<double>{0.0, 0.0};
                for (int c = 0; c < gd; ++c) {
                    unsigned rc = base;
                    for (int j = 0; j < gk; ++j) rc |= ((unsigned)(c >> j) & 1u) << G.lt[j];
                    const Amp<double> u = U[row * gd + c], x = M[rc * dim + col];
                    s.x += u.x * x.x - u.y * x.y;
                    s.y += u.x * x.y + u.y * x.x;
                }
            }
            N[r * dim + col] = s;
        }
        __syncthreads();
        Amp<double> *sw = M;
        M = N;
        N = sw;
    }
    char *dst = out + (size_t)blockIdx.x * kBlockBytes;
    const int steps = dim / 4, rowTiles = k == 5 ? 2 : 1;
    if constexpr (sizeof(T) == 4) {
        float *f = reinterpret_cast<float *>(dst);
        // vector v of lane l: fragments 4 v .. 4 v + 3, fragment (3 h + p) steps + st
        const int vecs = 3 * rowTiles * steps / 4;
        for (int i = tid; i < vecs * 64 * 4; i += kBlock) {
            const int lane = (i >> 2) & 63, fr = (i >> 8) * 4 + (i & 3);
            const int st = fr % steps, p = (fr / steps) % 3, h = fr / (3 * steps);
            const int col = lane & 15, kq = lane >> 4;
            const int row = 16 * h + 4 * (col & 3) + (col >> 2);
            const Amp<double> z = M[row * dim + 4 * st + kq];
            f[i] = (float)(p == 0 ? z.x : p == 1 ? z.y : z.x + z.y);
        }
    } else {
        Amp<double> *f = reinterpret_cast<Amp<double> *>(dst);
        for (int i = tid; i < rowTiles * steps * 64; i += kBlock) {
            const int lane = i & 63, fr = i >> 6, st = fr % steps, h = fr / steps;
            f[i] = M[(16 * h + (lane & 15)) * dim + 4 * st + (lane >> 4)];
        }
    }
}

// ---- the tile kernel ---------------------------------------------------------------
// LDS slots are linear in the tile element (see the top of the file), so a slot is
// the XOR of its bits' slots
struct BlockDev {
    int k;
    unsigned col[4];     // slot of column bit j
    unsigned kq[2];      // slot of combination bits 0, 1
    unsigned st[8];      // slot of combination 4 st
    unsigned rest[4];    // slot of the tile's other bits: 16-group chunks
};

struct TileGeom {
    int pos[kTB];        // the tile's qubits, ascending
    uint64_t jAddr[16];  // register offset of a thread's j-th transfer
    unsigned jSlot[16];
};

template <typename T>
__host__ __device__ __forceinline__ constexpr unsigned slotBit(int i) {
    constexpr int R = sizeof(T) == 4 ? 4 : 3;
    return (1u << i) | (i >= R ? 1u << (i % R) : 0u);
}

template <typename T>
__device__ __forceinline__ unsigned tileSlot(unsigned e) {
    if constexpr (sizeof(T) == 4) return e ^ ((e >> 4) & 15u) ^ ((e >> 8) & 15u);
    else return e ^ ((e >> 3) & 7u) ^ ((e >> 6) & 7u) ^ ((e >> 9) & 7u);
}

// a block of K qubits on the chunks of one wave
template <int K>
__device__ __forceinline__ void blockChunks(Amp<float> *tile, const BlockDev &B, unsigned inLane, int wave,
                                            const f4 *__restrict__ frag, int lane) {
    constexpr int S = 1 << (K - 2), H = K == 5 ? 2 : 1, NV = 3 * H * S / 4;
    f4 fv[NV];
#pragma unroll
    for (int i = 0; i < NV; ++i) fv[i] = frag[i * 64 + lane];
#pragma unroll 1
    for (int ch = wave; ch < 1 << (kTB - 4 - K); ch += kWaves) {
        unsigned s0 = inLane;
#pragma unroll
        for (int b = 0; b < kTB - 4 - K; ++b)
            if ((ch >> b) & 1) s0 ^= B.rest[b];
        f4 acc[H][3];
#pragma unroll
        for (int h = 0; h < H; ++h)
#pragma unroll
            for (int p = 0; p < 3; ++p) acc[h][p] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int st = 0; st < S; ++st) {
            const Amp<float> x = tile[s0 ^ B.st[st]];
            const float xs = x.x + x.y;
#pragma unroll
            for (int h = 0; h < H; ++h) {
                const int f0 = (3 * h) * S + st, f1 = (3 * h + 1) * S + st, f2 = (3 * h + 2) * S + st;
                acc[h][0] = __builtin_amdgcn_mfma_f32_16x16x4f32(fv[f0 >> 2][f0 & 3], x.x, acc[h][0], 0, 0, 0);
                acc[h][1] = __builtin_amdgcn_mfma_f32_16x16x4f32(fv[f1 >> 2][f1 & 3], x.y, acc[h][1], 0, 0, 0);
                acc[h][2] = __builtin_amdgcn_mfma_f32_16x16x4f32(fv[f2 >> 2][f2 & 3], xs, acc[h][2], 0, 0, 0);
            }
        }
        // the wave's reads of these 16 groups are done: results go back in place
#pragma unroll
        for (int h = 0; h < H; ++h)
#pragma unroll
            for (int v = 0; v < 4; ++v)
                tile[s0 ^ B.st[4 * h + v]] = Amp<float>{acc[h][0][v] - acc[h][1][v],
                                                        acc[h][2][v] - acc[h][0][v] - acc[h][1][v]};
    }
}

template <int K>
__device__ __forceinline__ void blockChunks(Amp<double> *tile, const BlockDev &B, unsigned inLane, int wave,
                                            const d2 *__restrict__ frag, int lane) {
    constexpr int S = 1 << (K - 2), H = K == 5 ? 2 : 1;
    d2 fv[H * S];
#pragma unroll
    for (int i = 0; i < H * S; ++i) fv[i] = frag[i * 64 + lane];
#pragma unroll 1
    for (int ch = wave; ch < 1 << (kTB - 4 - K); ch += kWaves) {
        unsigned s0 = inLane;
#pragma unroll
        for (int b = 0; b < kTB - 4 - K; ++b)
            if ((ch >> b) & 1) s0 ^= B.rest[b];
        d4 acc[H][3];
#pragma unroll
        for (int h = 0; h < H; ++h)
#pragma unroll
            for (int p = 0; p < 3; ++p) acc[h][p] = d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int st = 0; st < S; ++st) {
            const Amp<double> x = tile[s0 ^ B.st[st]];
            const double xs = x.x + x.y;
#pragma unroll
            for (int h = 0; h < H; ++h) {
                const d2 u = fv[h * S + st];
                acc[h][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(u.x, x.x, acc[h][0], 0, 0, 0);
                acc[h][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(u.y, x.y, acc[h][1], 0, 0, 0);
                acc[h][2] = __builtin_amdgcn_mfma_f64_16x16x4f64(u.x + u.y, xs, acc[h][2], 0, 0, 0);
            }
        }
#pragma unroll
        for (int h = 0; h < H; ++h)
#pragma unroll
            for (int v = 0; v < 4; ++v)
                tile[s0 ^ B.st[4 * h + v]] = Amp<double>{acc[h][0][v] - acc[h][1][v],
                                                         acc[h][2][v] - acc[h][0][v] - acc[h][1][v]};
    }
}

template <typename T, bool NT>
__global__ void __launch_bounds__(kBlock, sizeof(T) == 4 ? 4 : 2)
    kTileSweep(Amp<T> *__restrict__ a, TileGeom geo, const BlockDev *__restrict__ blocks, int numBlocks,
               const char *__restrict__ frags) {
    // a thread moves 16 B at a time: two FP32 amplitudes or one FP64
    constexpr int PAIR = sizeof(T) == 4 ? 1 : 0, J = 1 << (kTB - 8 - PAIR);
    typedef typename Frag<T>::V V;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    Amp<T> *tile = reinterpret_cast<Amp<T> *>(smem);
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    uint64_t addr = (uint64_t)flatBlock();
#pragma unroll
    for (int i = 0; i < kTB; ++i) addr = insertZero(addr, geo.pos[i]);
#pragma unroll
    for (int i = 0; i < 8; ++i)
        if ((tid >> i) & 1) addr |= 1ull << geo.pos[i + PAIR];
    Amp<T> *src = a + addr;
    const unsigned mySlot = tileSlot<T>((unsigned)tid << PAIR);
    {
        V r[J];
#pragma unroll
        for (int j = 0; j < J; ++j) {
            const V *p = reinterpret_cast<const V *>(src + geo.jAddr[j]);
            r[j] = NT ? __builtin_nontemporal_load(p) : *p;
        }
#pragma unroll
        for (int j = 0; j < J; ++j) {
            tile[mySlot ^ geo.jSlot[j]] = Amp<T>{r[j][0], r[j][1]};
            if constexpr (PAIR) tile[mySlot ^ geo.jSlot[j] ^ 1u] = Amp<T>{r[j][2], r[j][3]};
        }
    }
    __syncthreads();
    for (int b = 0; b < numBlocks; ++b) {
        const BlockDev &B = blocks[b];
        const V *frag = reinterpret_cast<const V *>(frags + (size_t)b * kBlockBytes);
        unsigned inLane = 0;
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if ((lane >> j) & 1) inLane ^= B.col[j];
#pragma unroll
        for (int j = 0; j < 2; ++j)
            if ((lane >> (4 + j)) & 1) inLane ^= B.kq[j];
        if (B.k == 5) blockChunks<5>(tile, B, inLane, wave, frag, lane);
        else blockChunks<4>(tile, B, inLane, wave, frag, lane);
        __syncthreads();
    }
#pragma unroll
    for (int j = 0; j < J; ++j) {
        V r;
        const Amp<T> lo = tile[mySlot ^ geo.jSlot[j]];
        r[0] = lo.x;
        r[1] = lo.y;
        if constexpr (PAIR) {
            const Amp<T> hi = tile[mySlot ^ geo.jSlot[j] ^ 1u];
            r[2] = hi.x;
            r[3] = hi.y;
        }
        V *p = reinterpret_cast<V *>(src + geo.jAddr[j]);
        if (NT) __builtin_nontemporal_store(r, p);
        else *p = r;
    }
}

// ---- small registers -----------------------------------------------------------------
struct SmallGate {
    int kind;                    // FlatGate::MATRIX2 or NOT
    int target;
    int numFixed;                // target and controls
    unsigned set;                // the controls' mask
    unsigned char fixed[16];     // their positions, ascending
    Amp<double> u[4];
};

// The register (2^n amplitudes, n <= 12) stays in one workgroup's LDS while every
// gate of the list is applied, so a circuit is one launch: a launch per gate costs
// 2 us on the device and more on the host, a gate here SMALL_GATE_US us (a barrier
// and an LDS round trip; nothing bounds it but that chain).
template <typename T>
__global__ void __launch_bounds__(512) kSmallCircuit(Amp<T> *__restrict__ a, int n,
                                                     const SmallGate *__restrict__ gates, int numGates) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    Amp<T> *s = reinterpret_cast<Amp<T> *>(smem);
    const unsigned dim = 1u << n, step = blockDim.x;
    for (unsigned i = threadIdx.x; i < dim; i += step) s[i] = a[i];
    __syncthreads();
    for (int g = 0; g < numGates; ++g) {
        const SmallGate &G = gates[g];
        const unsigned work = dim >> G.numFixed, bit = 1u << G.target, set = G.set;
        if (G.kind == FlatGate::NOT) {
            for (unsigned w = threadIdx.x; w < work; w += step) {
                unsigned i = w;
                for (int j = 0; j < G.numFixed; ++j) i = ((i >> G.fixed[j]) << (G.fixed[j] + 1)) | (i & ((1u << G.fixed[j]) - 1u));
                i |= set;
                const Amp<T> x = s[i], y = s[i | bit];
                s[i] = y;
                s[i | bit] = x;
            }
        } else {
            const T ar = (T)G.u[0].x, ai = (T)G.u[0].y, br = (T)G.u[1].x, bi = (T)G.u[1].y;
            const T cr = (T)G.u[2].x, ci = (T)G.u[2].y, dr = (T)G.u[3].x, di = (T)G.u[3].y;
            for (unsigned w = threadIdx.x; w < work; w += step) {
                unsigned i = w;
                for (int j = 0; j < G.numFixed; ++j) i = ((i >> G.fixed[j]) << (G.fixed[j] + 1)) | (i & ((1u << G.fixed[j]) - 1u));
                i |= set;
                const Amp<T> x = s[i], y = s[i | bit];
                s[i] = Amp<T>{ar * x.x - ai * x.y + br * y.x - bi * y.y, ar * x.y + ai * x.x + br * y.y + bi * y.x};
                s[i | bit] = Amp<T>{cr * x.x - ci * x.y + dr * y.x - di * y.y,
                                    cr * x.y + ci * x.x + dr * y.y + di * y.x};
            }
        }
        __syncthreads();
    }
    for (unsigned i = threadIdx.x; i < dim; i += step) a[i] = s[i];
}

// ---- host side -----------------------------------------------------------------------
size_t align16(size_t x) { return (x + 15) & ~(size_t)15; }

// One upload holds the build list, the gates and their matrices, then the blocks'
// kernel descriptions.
struct Upload {
    size_t todo, gates, mats, blocks, bytes;
};

int numMats(const FlatGate *gates, const SweepPlan &plan, int firstBlock, int numBlocks, size_t *entries) {
    int count = 0;
    *entries = 0;
    for (int b = firstBlock; b < firstBlock + numBlocks; ++b)
        for (int g = 0; g < plan.blocks[b].numGates; ++g) {
            const FlatGate &f = gates[plan.order[plan.blocks[b].firstGate + g]];
            if (f.kind != FlatGate::MATRIXN) continue;
            ++count;
            *entries += (size_t)1 << (2 * f.k);
        }
    return count;
}

int gateCount(const SweepPlan &plan, int firstBlock, int numBlocks) {
    int n = 0;
    for (int b = firstBlock; b < firstBlock + numBlocks; ++b) n += plan.blocks[b].numGates;
    return n;
}

Upload layoutOf(const SweepPlan &plan, const FlatGate *gates, int firstBlock, int numBlocks) {
    size_t entries = 0;
    numMats(gates, plan, firstBlock, numBlocks, &entries);
    Upload u;
    u.todo = 0;
    u.gates = align16(numBlocks * sizeof(BuildDev));
    u.mats = u.gates + align16((size_t)gateCount(plan, firstBlock, numBlocks) * sizeof(GateDev));
    u.blocks = u.mats + entries * sizeof(Amp<double>);
    u.bytes = align16(u.blocks + numBlocks * sizeof(BlockDev));
    return u;
}

void fillBuild(const SweepPlan &plan, const FlatGate *gates, int firstBlock, int numBlocks, const Upload &u,
               char *host) {
    BuildDev *todo = reinterpret_cast<BuildDev *>(host + u.todo);
    GateDev *gd = reinterpret_cast<GateDev *>(host + u.gates);
    Amp<double> *mats = reinterpret_cast<Amp<double> *>(host + u.mats);
    int at = 0, mat = 0;
    for (int i = 0; i < numBlocks; ++i) {
        const SweepBlock &b = plan.blocks[firstBlock + i];
        todo[i] = BuildDev{at, b.numGates, b.k, 0};
        auto local = [&](int qubit) {
            for (int j = 0; j < b.k; ++j)
                if (b.targs[j] == qubit) return j;
            std::fprintf(stderr, "libquest_mi355x: a planned block does not hold qubit %d\n", qubit);
            std::abort();
        };
        for (int g = 0; g < b.numGates; ++g) {
            const FlatGate &f = gates[plan.order[b.firstGate + g]];
            GateDev &d = gd[at++];
            d = GateDev{};
            d.kind = f.kind;
            for (uint64_t m = f.ctrl; m; m &= m - 1) d.ctrl |= 1u << local(__builtin_ctzll(m));
            if (f.kind == FlatGate::MATRIXN) {
                d.k = f.k;
                for (int j = 0; j < f.k; ++j) d.lt[j] = local(f.targs[j]);
                d.mat = mat;
                const int entries = 1 << (2 * f.k);
                for (int e = 0; e < entries; ++e) mats[mat + e] = Amp<double>{f.uN[e].re, f.uN[e].im};
                mat += entries;
            } else {
                d.t = local(f.target);
                for (int e = 0; e < 4; ++e) d.u[e] = Amp<double>{f.u[e].re, f.u[e].im};
            }
        }
    }
}

void tilePositions(uint64_t tile, int pos[kTB]) {
    int n = 0;
    for (uint64_t m = tile; m && n < kTB; m &= m - 1) pos[n++] = __builtin_ctzll(m);
    if (n != kTB || __builtin_popcountll(tile) != kTB) {
        std::fprintf(stderr, "libquest_mi355x: a planned tile has %d qubits\n", __builtin_popcountll(tile));
        std::abort();
    }
}

template <typename T>
BlockDev blockDev(const SweepBlock &b, const int pos[kTB]) {
    constexpr int R = sizeof(T) == 4 ? 4 : 3;   // columns per bank cycle: 2^R lanes
    BlockDev d{};
    d.k = b.k;
    int t[kSweepBlockQubits];
    bool used[kTB] = {};
    for (int j = 0; j < b.k; ++j) {
        t[j] = -1;
        for (int i = 0; i < kTB; ++i)
            if (pos[i] == b.targs[j]) t[j] = i;
        if (t[j] < 0) {
            std::fprintf(stderr, "libquest_mi355x: a planned block leaves its tile\n");
            std::abort();
        }
        used[t[j]] = true;
    }
    // columns: the first R take tile bits of different residues modulo R
    int cols[4], nc = 0;
    bool residue[4] = {};
    for (int i = 0; i < kTB && nc < R; ++i)
        if (!used[i] && !residue[i % R]) {
            residue[i % R] = used[i] = true;
            cols[nc++] = i;
        }
    for (int i = 0; i < kTB && nc < 4; ++i)
        if (!used[i]) {
            used[i] = true;
            cols[nc++] = i;
        }
    for (int j = 0; j < 4; ++j) d.col[j] = slotBit<T>(cols[j]);
    for (int j = 0; j < 2; ++j) d.kq[j] = slotBit<T>(t[j]);
    for (int st = 0; st < 1 << (b.k - 2); ++st)
        for (int j = 2; j < b.k; ++j)
            if ((st >> (j - 2)) & 1) d.st[st] ^= slotBit<T>(t[j]);
    for (int i = 0, r = 0; i < kTB; ++i)
        if (!used[i]) d.rest[r++] = slotBit<T>(i);
    return d;
}

// descriptions of the blocks that sweeps [first, last) hold
void fillBlocks(int prec, const SweepPlan &plan, int first, int last, int firstBlock, BlockDev *out) {
    for (int s = first; s < last; ++s) {
        const Sweep &w = plan.sweeps[s];
        if (w.lone >= 0) continue;
        int pos[kTB];
        tilePositions(w.tile, pos);
        for (int b = w.firstBlock; b < w.firstBlock + w.numBlocks; ++b)
            out[b - firstBlock] = prec == FP64 ? blockDev<double>(plan.blocks[b], pos)
                                               : blockDev<float>(plan.blocks[b], pos);
    }
}

void launchBuild(int prec, int numBlocks, const Upload &u, char *dev, char *frags) {
    const BuildDev *todo = reinterpret_cast<const BuildDev *>(dev + u.todo);
    const GateDev *gd = reinterpret_cast<const GateDev *>(dev + u.gates);
    const Amp<double> *mats = reinterpret_cast<const Amp<double> *>(dev + u.mats);
    QMX_DISPATCH(prec, T, {
        hipLaunchKernelGGL(kBuildBlocks<T>, dim3(numBlocks), dim3(kBlock), 0, hstream(), todo, gd, mats, frags);
    });
    checkLaunch("sweep block matrices");
}

template <typename T>
void launchSweep(QuregDev *q, const Sweep &w, const BlockDev *blocks, const char *frags) {
    constexpr int PAIR = sizeof(T) == 4 ? 1 : 0, J = 1 << (kTB - 8 - PAIR);
    constexpr size_t lds = sizeof(Amp<T>) << kTB;
    TileGeom geo{};
    tilePositions(w.tile, geo.pos);
    for (int j = 0; j < J; ++j)
        for (int i = 0; i < 4; ++i)
            if ((j >> i) & 1) {
                geo.jAddr[j] |= 1ull << geo.pos[8 + PAIR + i];
                geo.jSlot[j] ^= slotBit<T>(8 + PAIR + i);
            }
    // streaming accesses where the register outgrows the last-level cache
    const bool nt = q->numAmps * (long long)sizeof(Amp<T>) > (256ll << 20);
    const dim3 grid = gridOf(q->numAmps >> kTB);
    if (nt)
        hipLaunchKernelGGL((kTileSweep<T, true>), grid, dim3(kBlock), lds, hstream(), (Amp<T> *)q->amps, geo, blocks,
                           w.numBlocks, frags);
    else
        hipLaunchKernelGGL((kTileSweep<T, false>), grid, dim3(kBlock), lds, hstream(), (Amp<T> *)q->amps, geo, blocks,
                           w.numBlocks, frags);
    checkLaunch("tile sweep");
}

void runSweeps(QuregDev *q, const SweepPlan &plan, const FlatGate *gates, int first, int last, int firstBlock,
               const BlockDev *blocks, const char *frags) {
    for (int s = first; s < last; ++s) {
        const Sweep &w = plan.sweeps[s];
        if (w.lone >= 0) {
            applyFlatGate(q, gates[w.lone]);
            continue;
        }
        const BlockDev *b = blocks + (w.firstBlock - firstBlock);
        const char *f = frags + (size_t)(w.firstBlock - firstBlock) * kBlockBytes;
        QMX_DISPATCH(q->prec, T, { launchSweep<T>(q, w, b, f); });
    }
}

// The library's workspace for lists applied once: the upload (pinned and on the
// device) and the fragments of a batch of blocks. It grows to what a batch
// needs and no further; the host copy is rewritten after its last copy's event,
// the device side by work queued behind everything that read it.
constexpr int kBatchBlocks = 256;
struct Workspace {
    char *host = nullptr, *dev = nullptr, *frags = nullptr;
    size_t bytes = 0;
    int fragBlocks = 0;
    hipEvent_t ev = nullptr;
    bool used = false;

    char *hostRoom(size_t need) {
        if (!ev) QMX_HIP_CHECK(hipEventCreateWithFlags(&ev, hipEventDisableTiming));
        if (need > bytes) {
            deviceSync();  // the old buffers may still be in use
            if (dev) QMX_HIP_CHECK(hipFree(dev));
            if (host) QMX_HIP_CHECK(hipHostFree(host));
            bytes = std::max(need, (size_t)1 << 18);
            QMX_HIP_CHECK(hipMalloc(reinterpret_cast<void **>(&dev), bytes));
            QMX_HIP_CHECK(hipHostMalloc(reinterpret_cast<void **>(&host), bytes, hipHostMallocDefault));
            used = false;
        }
        if (used) QMX_HIP_CHECK(hipEventSynchronize(ev));
        return host;
    }
    void commit(size_t n) {
        QMX_HIP_CHECK(hipMemcpyAsync(dev, host, n, hipMemcpyHostToDevice, hstream()));
        QMX_HIP_CHECK(hipEventRecord(ev, hstream()));
        used = true;
    }
    char *fragRoom(int blocks) {
        if (blocks > fragBlocks) {
            if (frags) devFree(frags);
            fragBlocks = std::max(blocks, 32);
            frags = static_cast<char *>(devAlloc((size_t)fragBlocks * kBlockBytes));
        }
        return frags;
    }
} g_ws;

}  // namespace

struct SweepProgram {
    int prec;
    char *upload = nullptr, *frags = nullptr;
    const BlockDev *blocks = nullptr;
};

SweepProgram *sweepProgramCreate(int prec, const SweepPlan &plan, const FlatGate *gates) {
    auto *p = new SweepProgram;
    p->prec = prec;
    const int n = (int)plan.blocks.size();
    if (n == 0) return p;
    const Upload u = layoutOf(plan, gates, 0, n);
    std::vector<char> host(u.bytes);
    fillBuild(plan, gates, 0, n, u, host.data());
    fillBlocks(prec, plan, 0, (int)plan.sweeps.size(), 0, reinterpret_cast<BlockDev *>(host.data() + u.blocks));
    p->upload = static_cast<char *>(devAlloc(u.bytes));
    hostToDevice(p->upload, host.data(), u.bytes);
    p->frags = static_cast<char *>(devAlloc((size_t)n * kBlockBytes));
    p->blocks = reinterpret_cast<const BlockDev *>(p->upload + u.blocks);
    launchBuild(prec, n, u, p->upload, p->frags);
    return p;
}

void sweepProgramFree(SweepProgram *p) {
    if (!p) return;
    devFree(p->upload);
    devFree(p->frags);
    delete p;
}

void sweepProgramRun(QuregDev *q, const SweepProgram *p, const SweepPlan &plan, const FlatGate *gates, int first,
                     int last) {
    runSweeps(q, plan, gates, first, last, 0, p->blocks, p->frags);
}

void sweepRunOnce(QuregDev *q, const SweepPlan &plan, const FlatGate *gates) {
    runtimeInit();
    const int total = (int)plan.sweeps.size();
    for (int first = 0; first < total;) {
        // a batch: whole sweeps of at most kBatchBlocks blocks (one sweep has at most kSweepMaxBlocks)
        int last = first, firstBlock = -1, n = 0;
        while (last < total) {
            const Sweep &w = plan.sweeps[last];
            if (w.lone < 0) {
                if (n + w.numBlocks > kBatchBlocks) break;
                if (firstBlock < 0) firstBlock = w.firstBlock;
                n += w.numBlocks;
            }
            ++last;
        }
        if (n == 0) {
            runSweeps(q, plan, gates, first, last, 0, nullptr, nullptr);
            first = last;
            continue;
        }
        const Upload u = layoutOf(plan, gates, firstBlock, n);
        char *host = g_ws.hostRoom(u.bytes);
        fillBuild(plan, gates, firstBlock, n, u, host);
        fillBlocks(q->prec, plan, first, last, firstBlock, reinterpret_cast<BlockDev *>(host + u.blocks));
        char *frags = g_ws.fragRoom(n);
        g_ws.commit(u.bytes);
        launchBuild(q->prec, n, u, g_ws.dev, frags);
        runSweeps(q, plan, gates, first, last, firstBlock, reinterpret_cast<const BlockDev *>(g_ws.dev + u.blocks),
                  frags);
        first = last;
    }
}

void applyFlatGate(QuregDev *q, const FlatGate &g) {
    if (g.kind == FlatGate::MATRIXN) {
        applyMatrixN(q, g.ctrl, g.targs, g.k, g.uN);
        return;
    }
    if (g.kind == FlatGate::NOT) {
        applyNot(q, g.ctrl, 1ull << g.target);
        return;
    }
    auto is = [](const Cplx &z, double re) { return z.re == re && z.im == 0; };
    if (is(g.u[0], 1) && is(g.u[1], 0) && is(g.u[2], 0)) {
        applyPhaseOnAllOnes(q, g.ctrl | (1ull << g.target), g.u[3]);
        return;
    }
    applyMatrix2(q, g.target, g.ctrl, 0, g.u);
}

void smallCircuit(QuregDev *q, const FlatGate *gates, int count) {
    runtimeInit();
    // gates per launch: bounds the upload
    constexpr int kPerLaunch = 4096;
    const int n = q->numQubits;
    // two pairs a thread where there are that many; whole waves
    const unsigned threads = std::min(512u, std::max(64u, 1u << std::max(0, n - 2)));
    for (int first = 0; first < count; first += kPerLaunch) {
        const int num = std::min(kPerLaunch, count - first);
        SmallGate *h = reinterpret_cast<SmallGate *>(g_ws.hostRoom((size_t)num * sizeof(SmallGate)));
        for (int i = 0; i < num; ++i) {
            const FlatGate &f = gates[first + i];
            SmallGate &d = h[i];
            d.kind = f.kind;
            d.target = f.target;
            d.set = (unsigned)f.ctrl;
            d.numFixed = 0;
            for (uint64_t m = f.mask(); m; m &= m - 1) d.fixed[d.numFixed++] = (unsigned char)__builtin_ctzll(m);
            for (int e = 0; e < 4; ++e) d.u[e] = Amp<double>{f.u[e].re, f.u[e].im};
        }
        g_ws.commit((size_t)num * sizeof(SmallGate));
        const SmallGate *dg = reinterpret_cast<const SmallGate *>(g_ws.dev);
        QMX_DISPATCH(q->prec, T, {
            hipLaunchKernelGGL(kSmallCircuit<T>, dim3(1), dim3(threads), sizeof(Amp<T>) << n, hstream(),
                               (Amp<T> *)q->amps, n, dg, num);
        });
        checkLaunch("smallCircuit");
    }
}

}  // namespace qmx
