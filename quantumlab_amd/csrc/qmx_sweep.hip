// Sweeps of many gates: LDS tiles with dense 4- and 5-qubit blocks on the matrix
// cores (registers of more than kSweepTileBits qubits), and whole circuits in one
// workgroup's LDS (smaller ones).
//
// Tiles. A workgroup owns a tile of 2^12 amplitudes (32 KiB in FP32, 64 KiB in
// FP64): the sweep's 12 qubits, of which the lowest 4 (FP32) or 3 (FP64) make
// every memory run a whole 128 B line. It loads the tile into LDS, applies the
// sweep's blocks one after another there, and stores it. A block U on k = 4 or 5
// of the tile's qubits multiplies 16 groups of 2^k amplitudes at a time as three
// real products of v_mfma_f32_16x16x4f32 / v_mfma_f64_16x16x4f64 steps:
//   FP32: P = Ur Xr, Q = Ui Xi, R = (Ur + Ui)(Xr + Xi); Re = P - Q, Im = R - P - Q;
//   FP64: T = Ur (Xr + Xi); Re = T - (Ur + Ui) Xi, Im = T + (Ui - Ur) Xr, where T is
//         the start value of the other two sums, so nothing is left to subtract.
// (In FP32 the second form took 2 % off a sweep, but its real parts then share
// the rounding of the larger product: 5.9e-7 from the 64-bit state after a 30-qubit
// brick period, where the first form is at 5.4e-7.)
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
static_assert(sizeof(GateDev) == 112, "no uninitialised tail");
struct BuildDev {
    int firstGate, numGates, k, pad;
    // byte offsets of the LDS slots: column bits, combination bits 0 and 1,
    // combinations 4 st
    unsigned col[4], kq[2], st[8];
};

// What a lane needs of a block, in 16 B vectors (vector i of all lanes, then i + 1):
// its operands' LDS slots, one for each step (1 vector for k = 4, 2 for k = 5), then
// its 3 x 4 or 3 x 16 matrix fragments. Every block has the room of the largest.
constexpr size_t kBlockBytes = (2 * 16 + 3 * 16 * sizeof(double)) * 64;
template <typename T> constexpr int blockVecs(int k) { return (k == 5 ? 2 : 1) + 3 * (k == 5 ? 16 : 4) * (int)sizeof(T) / 16; }
static_assert(blockVecs<double>(5) * 1024 <= (int)kBlockBytes, "a block's vectors fit its room");

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
    // gates staged in LDS at a time (a scalar load of each on the critical path
    // made a block of 15 gates 23 us)
    constexpr int kStage = 32;
    static_assert(sizeof(GateDev) % 16 == 0, "gates move in 16 B pieces");
    __shared__ Amp<double> buf[2][32 * 32];
    __shared__ GateDev stage[kStage];
    const BuildDev b = todo[blockIdx.x];
    const int k = b.k, dim = 1 << k, tid = threadIdx.x;
    Amp<double> *M = buf[0], *N = buf[1];
    for (int i = tid; i < dim * dim; i += kBlock) M[i] = Amp<double>{(i >> k) == (i & (dim - 1)) ? 1.0 : 0.0, 0.0};
    __syncthreads();
    for (int g = 0; g < b.numGates; ++g) {
        if (g % kStage == 0) {
            const int words = min(kStage, b.numGates - g) * (int)(sizeof(GateDev) / 16);
            const uint4 *src = reinterpret_cast<const uint4 *>(gates + b.firstGate + g);
            for (int i = tid; i < words; i += kBlock) reinterpret_cast<uint4 *>(stage)[i] = src[i];
            __syncthreads();
        }
        const GateDev &G = stage[g % kStage];
        const unsigned ctrl = (unsigned)__builtin_amdgcn_readfirstlane((int)G.ctrl);
        const int kind = __builtin_amdgcn_readfirstlane(G.kind);
        if (kind != FlatGate::MATRIXN) {
            const int t = __builtin_amdgcn_readfirstlane(G.t);
            const bool isNot = kind == FlatGate::NOT;
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
    // fragment (h steps + st) of each of the three matrices: Ur, Ui, Ur + Ui in FP32,
    // Ur, -(Ur + Ui), Ui - Ur in FP64
    char *dst = out + (size_t)blockIdx.x * kBlockBytes;
    const int steps = dim / 4, frags = (k == 5 ? 2 : 1) * steps;
    unsigned *slots = reinterpret_cast<unsigned *>(dst);
    for (int i = tid; i < steps * 64; i += kBlock) {
        const int lane = (i >> 2) & 63, st = (i >> 8) * 4 + (i & 3);
        unsigned o = b.st[st];
        for (int j = 0; j < 4; ++j) o ^= ((lane >> j) & 1) ? b.col[j] : 0u;
        for (int j = 0; j < 2; ++j) o ^= ((lane >> (4 + j)) & 1) ? b.kq[j] : 0u;
        slots[i] = o;
    }
    dst += (size_t)steps * 64 * sizeof(unsigned);
    if constexpr (sizeof(T) == 4) {
        float *f = reinterpret_cast<float *>(dst);
        // matrix p: vectors p frags/4 ..., vector v of lane l: fragments 4 v .. 4 v + 3
        for (int i = tid; i < 3 * frags * 64; i += kBlock) {
            const int lane = (i >> 2) & 63, v = i >> 8;
            const int p = v / (frags / 4), fr = (v % (frags / 4)) * 4 + (i & 3);
            const int st = fr % steps, h = fr / steps;
            const int col = lane & 15, kq = lane >> 4;
            const int row = 16 * h + 4 * (col & 3) + (col >> 2);
            const Amp<double> z = M[row * dim + 4 * st + kq];
            f[i] = (float)(p == 0 ? z.x : p == 1 ? z.y : z.x + z.y);
        }
    } else {
        double *f = reinterpret_cast<double *>(dst);
        // matrix p: vectors p frags/2 ..., vector v of lane l: fragments 2 v, 2 v + 1
        for (int i = tid; i < 3 * frags * 64; i += kBlock) {
            const int lane = (i >> 1) & 63, v = i >> 7;
            const int p = v / (frags / 2), fr = (v % (frags / 2)) * 2 + (i & 1);
            const int st = fr % steps, h = fr / steps;
            const Amp<double> z = M[(16 * h + (lane & 15)) * dim + 4 * st + (lane >> 4)];
            f[i] = p == 0 ? z.x : p == 1 ? -(z.x + z.y) : z.y - z.x;
        }
    }
}

// ---- the tile kernel ---------------------------------------------------------------
// LDS slots are linear in the tile element (see the top of the file), so a slot is
// the XOR of its bits' slots; here as byte offsets
struct BlockDev {
    int k;
    unsigned rest[4];    // slots of the tile's bits beyond columns and targets: 16-group chunks
};

struct TileGeom {
    int pos[kTB];        // the tile's qubits, ascending
    uint64_t jAddr[16];  // register offset of a thread's j-th transfer
    unsigned jSlot[16];  // its slot's part from j (bytes)
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

__device__ __forceinline__ f4 mfma(float a, float b, f4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ d4 mfma(double a, double b, d4 c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
template <typename T> struct Acc4;
template <> struct Acc4<float> { typedef f4 type; };
template <> struct Acc4<double> { typedef d4 type; };

// A block of K qubits on the chunks of one wave, IL chunks at a time: v holds the
// block's vectors, s0 the slot of each chunk of the wave.
template <typename T, int K, int WAVES>
__device__ __forceinline__ void blockChunks(char *tile, const typename Frag<T>::V *v, const BlockDev &B, int wave) {
    typedef typename Acc4<T>::type A;
    constexpr int S = 1 << (K - 2), H = K == 5 ? 2 : 1, PV = 16 / sizeof(T), NV = H * S / PV, SV = S / 4;
    constexpr int CH = (1 << (kTB - 4 - K)) / WAVES, IL = K == 5 ? 1 : 2;
    unsigned slot[S];
#pragma unroll
    for (int i = 0; i < SV; ++i) {
        union {
            typename Frag<T>::V f;
            unsigned u[4];
        } c;
        c.f = v[i];
#pragma unroll
        for (int j = 0; j < 4; ++j) slot[4 * i + j] = c.u[j];
    }
#pragma unroll 1
    for (int c0 = 0; c0 < CH; c0 += IL) {
        unsigned s0[IL];  // the same for the whole wave
#pragma unroll
        for (int l = 0; l < IL; ++l) {
            const int ch = wave + WAVES * (c0 + l);
            s0[l] = 0;
#pragma unroll
            for (int b = 0; b < kTB - 4 - K; ++b) s0[l] ^= ((ch >> b) & 1) ? B.rest[b] : 0u;
        }
        Amp<T> x[IL][S];
#pragma unroll
        for (int l = 0; l < IL; ++l)
#pragma unroll
            for (int st = 0; st < S; ++st) x[l][st] = *reinterpret_cast<const Amp<T> *>(tile + (slot[st] ^ s0[l]));
        A t[IL][H], re[IL][H], im[IL][H];
        const A zero = {0, 0, 0, 0};
#pragma unroll
        for (int l = 0; l < IL; ++l)
#pragma unroll
            for (int h = 0; h < H; ++h) t[l][h] = re[l][h] = im[l][h] = zero;
        if constexpr (sizeof(T) == 4) {
            // P, Q, R in re, im, t
#pragma unroll
            for (int st = 0; st < S; ++st)
#pragma unroll
                for (int l = 0; l < IL; ++l) {
                    const T xs = x[l][st].x + x[l][st].y;
#pragma unroll
                    for (int h = 0; h < H; ++h) {
                        const int i = h * S + st;
                        re[l][h] = mfma(v[SV + i / PV][i % PV], x[l][st].x, re[l][h]);
                        im[l][h] = mfma(v[SV + NV + i / PV][i % PV], x[l][st].y, im[l][h]);
                        t[l][h] = mfma(v[SV + 2 * NV + i / PV][i % PV], xs, t[l][h]);
                    }
                }
#pragma unroll
            for (int l = 0; l < IL; ++l)
#pragma unroll
                for (int h = 0; h < H; ++h) {
                    const A p = re[l][h], q = im[l][h];
                    re[l][h] = p - q;
                    im[l][h] = t[l][h] - p - q;
                }
        } else {
#pragma unroll
            for (int st = 0; st < S; ++st)
#pragma unroll
                for (int l = 0; l < IL; ++l) {
                    const T xs = x[l][st].x + x[l][st].y;
#pragma unroll
                    for (int h = 0; h < H; ++h) {
                        const int i = h * S + st;
                        t[l][h] = mfma(v[SV + i / PV][i % PV], xs, t[l][h]);
                    }
                }
#pragma unroll
            for (int l = 0; l < IL; ++l)
#pragma unroll
                for (int h = 0; h < H; ++h) re[l][h] = im[l][h] = t[l][h];
#pragma unroll
            for (int st = 0; st < S; ++st)
#pragma unroll
                for (int l = 0; l < IL; ++l)
#pragma unroll
                    for (int h = 0; h < H; ++h) {
                        const int i = h * S + st;
                        re[l][h] = mfma(v[SV + NV + i / PV][i % PV], x[l][st].y, re[l][h]);
                        im[l][h] = mfma(v[SV + 2 * NV + i / PV][i % PV], x[l][st].x, im[l][h]);
                    }
        }
        // the wave's reads of these groups are done: results go back in place
#pragma unroll
        for (int l = 0; l < IL; ++l)
#pragma unroll
            for (int h = 0; h < H; ++h)
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    *reinterpret_cast<Amp<T> *>(tile + (slot[4 * h + e] ^ s0[l])) = Amp<T>{re[l][h][e], im[l][h][e]};
    }
}

template <typename T, bool NT, int WAVES>
__global__ void __launch_bounds__(64 * WAVES, sizeof(T) == 4 ? 4 : 2)
    kTileSweep(Amp<T> *__restrict__ a, TileGeom geo, const BlockDev *__restrict__ blocks, int numBlocks,
               const char *__restrict__ frags) {
    // a thread moves 16 B at a time: two FP32 amplitudes or one FP64
    constexpr int PAIR = sizeof(T) == 4 ? 1 : 0, THREADS = 6 + (WAVES == 8 ? 3 : 2), J = 1 << (kTB - THREADS - PAIR);
    typedef typename Frag<T>::V V;
    __shared__ __attribute__((aligned(16))) char tile[sizeof(Amp<T>) << kTB];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    uint64_t addr = (uint64_t)flatBlock();
#pragma unroll
    for (int i = 0; i < kTB; ++i) addr = insertZero(addr, geo.pos[i]);
#pragma unroll
    for (int i = 0; i < THREADS; ++i)
        if ((tid >> i) & 1) addr |= 1ull << geo.pos[i + PAIR];
    Amp<T> *src = a + addr;
    const unsigned mySlot = tileSlot<T>((unsigned)tid << PAIR) * (unsigned)sizeof(Amp<T>);
    auto at = [&](unsigned slot) -> Amp<T> & { return *reinterpret_cast<Amp<T> *>(tile + slot); };
    {
        V r[J];
#pragma unroll
        for (int j = 0; j < J; ++j) {
            const V *p = reinterpret_cast<const V *>(src + geo.jAddr[j]);
            r[j] = NT ? __builtin_nontemporal_load(p) : *p;
        }
#pragma unroll
        for (int j = 0; j < J; ++j) {
            at(mySlot ^ geo.jSlot[j]) = Amp<T>{r[j][0], r[j][1]};
            if constexpr (PAIR) at(mySlot ^ geo.jSlot[j] ^ (unsigned)sizeof(Amp<T>)) = Amp<T>{r[j][2], r[j][3]};
        }
    }
    __syncthreads();
    // a 4-qubit block's vectors are loaded while the block before it multiplies
    constexpr int V4 = blockVecs<T>(4), V5 = blockVecs<T>(5);
    const V *next = reinterpret_cast<const V *>(frags) + lane;
    BlockDev B = blocks[0], nB = B;
    V v[V5], pre[V4];
#pragma unroll
    for (int i = 0; i < V4; ++i) pre[i] = next[i * 64];
    for (int b = 0; b < numBlocks; ++b) {
        const V *mineB = next;
        next += kBlockBytes / sizeof(V);
#pragma unroll
        for (int i = 0; i < V4; ++i) v[i] = pre[i];
        if (b + 1 < numBlocks) {  // the same for the whole workgroup
            nB = blocks[b + 1];
#pragma unroll
            for (int i = 0; i < V4; ++i) pre[i] = next[i * 64];
        }
        if (B.k == 5) {
#pragma unroll
            for (int i = V4; i < V5; ++i) v[i] = mineB[i * 64];
            blockChunks<T, 5, WAVES>(tile, v, B, wave);
        } else {
            blockChunks<T, 4, WAVES>(tile, v, B, wave);
        }
        B = nB;
        __syncthreads();
    }
#pragma unroll
    for (int j = 0; j < J; ++j) {
        V r;
        const Amp<T> lo = at(mySlot ^ geo.jSlot[j]);
        r[0] = lo.x;
        r[1] = lo.y;
        if constexpr (PAIR) {
            const Amp<T> hi = at(mySlot ^ geo.jSlot[j] ^ (unsigned)sizeof(Amp<T>));
            r[2] = hi.x;
            r[3] = hi.y;
        }
        V *p = reinterpret_cast<V *>(src + geo.jAddr[j]);
        if (NT) __builtin_nontemporal_store(r, p);
        else *p = r;
    }
}

// ---- small registers -----------------------------------------------------------------
// The register (2^n amplitudes, n <= 12) stays in one workgroup's LDS, in FP64 for
// both storage precisions, while every gate of the list is applied: a circuit is
// one launch, rounded to FP32 once at its end. Gates run in groups whose targets
// are at most two qubits: a thread holds the four amplitudes of those two (a
// "quad"), applies the group's gates in registers and writes them back, so a
// group costs one LDS round trip and one barrier. Controls may be any qubits.
// Nothing but that chain bounds it (one workgroup): SMALL_MEASURED
struct SmallGate {
    int group;                   // > 0: opens a group with this many gates on qubits (t0, t1)
    int t0, t1;                  // the group's qubits, ascending
    int target;                  // 0: t0, 1: t1
    int kind;                    // SG_*
    unsigned ctrl;               // controls, bits of the register index
    Amp<double> u[4];
};
enum { SG_GENERAL = 0, SG_NOT = 1, SG_DIAGONAL = 2, SG_REAL = 3 };

// gates staged in LDS at a time (coalesced loads once, instead of a scalar load
// of each gate on the critical path)
constexpr int kSmallStage = 64;
constexpr int kSmallThreads = 512;

__device__ __forceinline__ void smallPair(const SmallGate &G, int kind, Amp<double> &x, Amp<double> &y) {
    const Amp<double> p = x, q = y;
    switch (kind) {
    case SG_NOT:
        x = q;
        y = p;
        break;
    case SG_DIAGONAL: {
        const Amp<double> a = G.u[0], d = G.u[3];
        if (a.x != 1.0 || a.y != 0.0) x = Amp<double>{a.x * p.x - a.y * p.y, a.x * p.y + a.y * p.x};
        y = Amp<double>{d.x * q.x - d.y * q.y, d.x * q.y + d.y * q.x};
        break;
    }
    case SG_REAL:
        x = Amp<double>{G.u[0].x * p.x + G.u[1].x * q.x, G.u[0].x * p.y + G.u[1].x * q.y};
        y = Amp<double>{G.u[2].x * p.x + G.u[3].x * q.x, G.u[2].x * p.y + G.u[3].x * q.y};
        break;
    default: {
        const Amp<double> a = G.u[0], b = G.u[1], c = G.u[2], d = G.u[3];
        x = Amp<double>{a.x * p.x - a.y * p.y + b.x * q.x - b.y * q.y, a.x * p.y + a.y * p.x + b.x * q.y + b.y * q.x};
        y = Amp<double>{c.x * p.x - c.y * p.y + d.x * q.x - d.y * q.y, c.x * p.y + c.y * p.x + d.x * q.y + d.y * q.x};
    }
    }
}

template <typename T>
__global__ void __launch_bounds__(kSmallThreads) kSmallCircuit(Amp<T> *__restrict__ a, int n,
                                                               const SmallGate *__restrict__ gates, int numGates) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    // n = 1 runs as two qubits whose upper half stays zero
    const int nn = n < 2 ? 2 : n;
    const unsigned dim = 1u << n, step = blockDim.x, quads = 1u << (nn - 2);
    Amp<double> *s = reinterpret_cast<Amp<double> *>(smem);
    SmallGate *stage = reinterpret_cast<SmallGate *>(smem + (sizeof(Amp<double>) << nn));
    for (unsigned i = threadIdx.x; i < 1u << nn; i += step)
        s[i] = i < dim ? Amp<double>{(double)a[i].x, (double)a[i].y} : Amp<double>{0, 0};
    for (int g0 = 0; g0 < numGates;) {
        // whole groups only: the host cuts groups at multiples of the stage
        const int num = min(kSmallStage, numGates - g0);
        const unsigned words = num * sizeof(SmallGate) / 16;
        const uint4 *src = reinterpret_cast<const uint4 *>(gates + g0);
        uint4 *dst = reinterpret_cast<uint4 *>(stage);
        for (unsigned i = threadIdx.x; i < words; i += step) dst[i] = src[i];
        __syncthreads();
        for (int g = 0; g < num;) {
            // the same in every lane: read into scalar registers
            const int count = __builtin_amdgcn_readfirstlane(stage[g].group);
            const int t0 = __builtin_amdgcn_readfirstlane(stage[g].t0), t1 = __builtin_amdgcn_readfirstlane(stage[g].t1);
            const unsigned b0 = 1u << t0, b1 = 1u << t1;
            for (unsigned w = threadIdx.x; w < quads; w += step) {
                unsigned i = ((w >> t0) << (t0 + 1)) | (w & (b0 - 1u));
                i = ((i >> t1) << (t1 + 1)) | (i & (b1 - 1u));
                Amp<double> x00 = s[i], x01 = s[i | b0], x10 = s[i | b1], x11 = s[i | b0 | b1];
                for (int e = 0; e < count; ++e) {
                    const SmallGate &G = stage[g + e];
                    const unsigned c = (unsigned)__builtin_amdgcn_readfirstlane((int)G.ctrl);
                    const int kind = __builtin_amdgcn_readfirstlane(G.kind);
                    if (__builtin_amdgcn_readfirstlane(G.target) == 0) {
                        if ((i & c) == c) smallPair(G, kind, x00, x01);
                        if (((i | b1) & c) == c) smallPair(G, kind, x10, x11);
                    } else {
                        if ((i & c) == c) smallPair(G, kind, x00, x10);
                        if (((i | b0) & c) == c) smallPair(G, kind, x01, x11);
                    }
                }
                s[i] = x00;
                s[i | b0] = x01;
                s[i | b1] = x10;
                s[i | b0 | b1] = x11;
            }
            g += count;
            __syncthreads();
        }
        g0 += num;
    }
    for (unsigned i = threadIdx.x; i < dim; i += step) a[i] = Amp<T>{(T)s[i].x, (T)s[i].y};
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
        todo[i] = BuildDev{at, b.numGates, b.k, 0, {}, {}, {}};
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
void blockSlots(const SweepBlock &b, const int pos[kTB], BuildDev &todo, BlockDev &d) {
    constexpr int R = sizeof(T) == 4 ? 4 : 3;   // columns per bank cycle: 2^R lanes
    d = BlockDev{};
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
    auto slot = [](int i) { return slotBit<T>(i) * (unsigned)sizeof(Amp<T>); };
    for (int j = 0; j < 4; ++j) todo.col[j] = slot(cols[j]);
    for (int j = 0; j < 2; ++j) todo.kq[j] = slot(t[j]);
    for (int st = 0; st < 1 << (b.k - 2); ++st)
        for (int j = 2; j < b.k; ++j)
            if ((st >> (j - 2)) & 1) todo.st[st] ^= slot(t[j]);
    for (int i = 0, r = 0; i < kTB; ++i)
        if (!used[i]) d.rest[r++] = slot(i);
}

// LDS slots and descriptions of the blocks that sweeps [first, last) hold
void fillBlocks(int prec, const SweepPlan &plan, int first, int last, int firstBlock, const Upload &u, char *host) {
    BuildDev *todo = reinterpret_cast<BuildDev *>(host + u.todo);
    BlockDev *out = reinterpret_cast<BlockDev *>(host + u.blocks);
    for (int s = first; s < last; ++s) {
        const Sweep &w = plan.sweeps[s];
        if (w.lone >= 0) continue;
        int pos[kTB];
        tilePositions(w.tile, pos);
        for (int b = w.firstBlock; b < w.firstBlock + w.numBlocks; ++b)
            QMX_DISPATCH(prec, T, { blockSlots<T>(plan.blocks[b], pos, todo[b - firstBlock], out[b - firstBlock]); });
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

template <typename T, int WAVES>
void launchSweepWaves(QuregDev *q, const Sweep &w, const BlockDev *blocks, const char *frags) {
    constexpr int PAIR = sizeof(T) == 4 ? 1 : 0, THREADS = 6 + (WAVES == 8 ? 3 : 2), J = 1 << (kTB - THREADS - PAIR);
    TileGeom geo{};
    tilePositions(w.tile, geo.pos);
    for (int j = 0; j < J; ++j)
        for (int i = 0; THREADS + PAIR + i < kTB; ++i)
            if ((j >> i) & 1) {
                geo.jAddr[j] |= 1ull << geo.pos[THREADS + PAIR + i];
                geo.jSlot[j] ^= slotBit<T>(THREADS + PAIR + i) * (unsigned)sizeof(Amp<T>);
            }
    // streaming accesses where the register outgrows the last-level cache
    const bool nt = q->numAmps * (long long)sizeof(Amp<T>) > (256ll << 20);
    const dim3 grid = gridOf(q->numAmps >> kTB);
    if (nt)
        hipLaunchKernelGGL((kTileSweep<T, true, WAVES>), grid, dim3(64 * WAVES), 0, hstream(), (Amp<T> *)q->amps, geo,
                           blocks, w.numBlocks, frags);
    else
        hipLaunchKernelGGL((kTileSweep<T, false, WAVES>), grid, dim3(64 * WAVES), 0, hstream(), (Amp<T> *)q->amps,
                           geo, blocks, w.numBlocks, frags);
    checkLaunch("tile sweep");
}

// Eight waves a tile where the register has too few tiles to fill the CUs with
// four (4 workgroups of 32 KiB, or 2 of 64, fit a CU): WAVES_MEASURED
template <typename T>
void launchSweep(QuregDev *q, const Sweep &w, const BlockDev *blocks, const char *frags) {
    constexpr int perCU = sizeof(T) == 4 ? 4 : 2;
    if ((q->numAmps >> kTB) < (long long)perCU * numCUs()) launchSweepWaves<T, 8>(q, w, blocks, frags);
    else launchSweepWaves<T, 4>(q, w, blocks, frags);
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
    fillBlocks(prec, plan, 0, (int)plan.sweeps.size(), 0, u, host.data());
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
        fillBlocks(q->prec, plan, first, last, firstBlock, u, host);
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

// a gate's arithmetic, by the entries of its matrix
static int smallKind(const FlatGate &f) {
    if (f.kind == FlatGate::NOT) return SG_NOT;
    auto zero = [](const Cplx &z) { return z.re == 0 && z.im == 0; };
    if (zero(f.u[1]) && zero(f.u[2])) return SG_DIAGONAL;
    for (const Cplx &z : f.u)
        if (z.im != 0) return SG_GENERAL;
    return SG_REAL;
}

// the SmallGates of gates[0 .. count): greedy runs of consecutive gates on at most
// two targets, no run across a multiple of kSmallStage
static void smallGroups(int n, const FlatGate *gates, int count, SmallGate *out) {
    for (int i = 0; i < count;) {
        int t0 = gates[i].target, t1 = -1, j = i;
        for (; j < count && (j == i || j % kSmallStage); ++j) {
            const int t = gates[j].target;
            if (t == t0 || t == t1) continue;
            if (t1 >= 0) break;
            t1 = t;
        }
        if (t1 < 0) t1 = t0 == 0 ? 1 : 0;  // any other qubit (n = 1: the one that stays zero)
        if (t0 > t1) std::swap(t0, t1);
        for (int k = i; k < j; ++k) {
            const FlatGate &f = gates[k];
            SmallGate &d = out[k];
            d.group = k == i ? j - i : 0;
            d.t0 = t0;
            d.t1 = t1;
            d.target = f.target == t0 ? 0 : 1;
            d.kind = smallKind(f);
            d.ctrl = (unsigned)f.ctrl;
            for (int e = 0; e < 4; ++e) d.u[e] = Amp<double>{f.u[e].re, f.u[e].im};
        }
        i = j;
    }
}

void smallCircuit(QuregDev *q, const FlatGate *gates, int count) {
    runtimeInit();
    static_assert(sizeof(SmallGate) % 16 == 0, "gates move in 16 B pieces");
    // gates per launch: bounds the upload
    constexpr int kPerLaunch = 64 * kSmallStage;
    const int n = q->numQubits, nn = std::max(n, 2);
    const unsigned threads = std::min((unsigned)kSmallThreads, std::max(64u, 1u << (nn - 2)));
    const size_t lds = (sizeof(Amp<double>) << nn) + kSmallStage * sizeof(SmallGate);
    for (int first = 0; first < count; first += kPerLaunch) {
        const int num = std::min(kPerLaunch, count - first);
        SmallGate *h = reinterpret_cast<SmallGate *>(g_ws.hostRoom((size_t)num * sizeof(SmallGate)));
        smallGroups(n, gates + first, num, h);
        g_ws.commit((size_t)num * sizeof(SmallGate));
        const SmallGate *dg = reinterpret_cast<const SmallGate *>(g_ws.dev);
        QMX_DISPATCH(q->prec, T, {
            static bool ldsAllowed = false;
            if (!ldsAllowed) {
                if (!allowDynamicLds(reinterpret_cast<const void *>(&kSmallCircuit<T>),
                                     (sizeof(Amp<double>) << kSmallCircuitQubits) + kSmallStage * sizeof(SmallGate),
                                     "a small register's circuit"))
                    std::abort();
                ldsAllowed = true;
            }
            hipLaunchKernelGGL(kSmallCircuit<T>, dim3(1), dim3(threads), lds, hstream(), (Amp<T> *)q->amps, n, dg,
                               num);
        });
        checkLaunch("smallCircuit");
    }
}

}  // namespace qmx
