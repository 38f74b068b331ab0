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
// the planner prefers them. Five-layer brick period, one block a sweep before and
// now: 30 qubits FP32 50.7 -> 30.1 ms (16 sweeps -> 6 to 8, of 24 to 26 blocks), 27
// qubits FP64 12.6 -> 7.0 ms. Seven blocks a sweep keep the matrix cores busy 70 % of the
// time, two leave it to HBM (3.1 ms for 16 GiB).
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

constexpr int kMaxTB = kSweepTileBits;

// ---- block matrices, built on the device ---------------------------------------
typedef double d8 __attribute__((ext_vector_type(8)));

struct GateDev {
    int kind;            // FlatGate::Kind
    unsigned t;          // target, a bit of the block's index; MATRIXN: its targets, 4 bits each;
                         // CHANNEL: row bit | column bit << 4
    unsigned ctrl;       // controls, bits of the block's index
    int k;               // MATRIXN
    int mat;             // MATRIXN: its matrix (entry offset)
    float lo;            // CHANNEL: d11Lo
    int pad[2];
    alignas(16) double u[8];  // the matrix, (re, im) by rows; CHANNEL: f, g, d00, d01, d10, d11, fLo, d00Lo
};

// gates staged in LDS at a time (whole coalesced loads; one entry more is read)
constexpr int kStage = 64;
template <typename G>
__device__ __forceinline__ void stageGates(G *stage, const G *__restrict__ src, int num, int tid, int threads) {
    static_assert(sizeof(G) % 16 == 0, "gates move in 16 B pieces");
    const uint4 *from = reinterpret_cast<const uint4 *>(src);
    for (int i = tid; i < num * (int)(sizeof(G) / 16); i += threads) reinterpret_cast<uint4 *>(stage)[i] = from[i];
}

// a staged gate's matrix as one vector value (indexed as an array, entries that
// differ between branches end up in scratch memory)
__device__ __forceinline__ d8 matrixOf(const double *u) {
    const d2 *v = reinterpret_cast<const d2 *>(u);
    const d2 a = v[0], b = v[1], c = v[2], d = v[3];
    return d8{a.x, a.y, b.x, b.y, c.x, c.y, d.x, d.y};
}

__device__ __forceinline__ unsigned uniform(unsigned x) { return (unsigned)__builtin_amdgcn_readfirstlane((int)x); }

// the gate with its integers in scalar registers (every lane holds the same gate)
__device__ __forceinline__ GateDev uniformGate(const GateDev &g) {
    GateDev r = g;
    r.kind = (int)uniform((unsigned)g.kind);
    r.t = uniform(g.t);
    r.ctrl = uniform(g.ctrl);
    r.k = (int)uniform((unsigned)g.k);
    r.mat = (int)uniform((unsigned)g.mat);
    return r;
}

// u0 p + u1 q of a gate's row (u0, u1) = (u[0] + i u[1], u[2] + i u[3])
__device__ __forceinline__ Amp<double> rowTimes(double a, double b, double c, double d, const Amp<double> &p,
                                                const Amp<double> &q) {
    return Amp<double>{a * p.x - b * p.y + c * q.x - d * q.y, a * p.y + b * p.x + c * q.y + d * q.x};
}
// (a + aLo) p + b q, b small beside a where aLo counts; the low part goes in before the
// sum is rounded to the size of a p, beside which it would be lost
__device__ __forceinline__ Amp<double> realTimes(double a, double aLo, double b, const Amp<double> &p,
                                                 const Amp<double> &q) {
    return Amp<double>{fma(a, p.x, fma(b, q.x, aLo * p.x)), fma(a, p.y, fma(b, q.y, aLo * p.y))};
}
// what a tile sweep needs of a block besides its vectors
struct BlockDev {
    int k;
    unsigned rest[4];    // slots of the tile's bits beyond columns and targets: 16-group chunks
};
struct BuildDev {
    int firstGate, numGates, k;
    unsigned at;         // its vectors' place, in KiB
    // byte offsets of the LDS slots: column bits, combination bits 0 and 1,
    // combinations 4 st
    unsigned col[4], kq[2], st[8];
    BlockDev tile;
};

// What a lane needs of a block, in 16 B vectors (vector i of all lanes, then i + 1):
// its operands' LDS slots, one for each step (1 vector for k = 4, 2 for k = 5), then
// its 3 x 4 or 3 x 16 matrix fragments; the next block's follow. A vector of all lanes
// is 1 KiB: a block takes 4 (4 qubits, FP32) to 26 of them.
template <typename T> constexpr int blockVecs(int k) { return (k == 5 ? 2 : 1) + 3 * (k == 5 ? 16 : 4) * (int)sizeof(T) / 16; }
constexpr size_t kMaxBlockBytes = (size_t)blockVecs<double>(5) * 1024;

template <typename T> struct Frag;
template <> struct Frag<float> { typedef f4 V; };
template <> struct Frag<double> { typedef d2 V; };

// One workgroup per block: the product of its gates in FP64, in LDS, then the
// block's vectors. The gates arrive as the host recorded them, so a list of any
// length costs one small copy instead of a matrix per block (on the host a block
// of ten gates took ~25 us). A wave owns a quarter of the matrix's columns, which no
// other wave touches, so gates follow one another without barriers (but for those with a
// matrix of their own, which is staged first); each gate is read from LDS while the one
// before it is applied (scalar loads straight from memory arrive a line at a time, 0.65
// us a gate). todo, gates and mats lie in pinned host memory: each is read once, whole,
// into LDS.
template <typename T>
__global__ void __launch_bounds__(kBlock) kBuildBlocks(const BuildDev *__restrict__ todo,
                                                       const GateDev *__restrict__ gates,
                                                       const Amp<double> *__restrict__ mats, char *__restrict__ out,
                                                       BlockDev *__restrict__ blocks) {
    __shared__ Amp<double> buf[2][32 * 32];
    __shared__ GateDev stage[kStage + 1];
    __shared__ Amp<double> U[32 * 32];
    __shared__ BuildDev b;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    static_assert(sizeof(BuildDev) / 4 <= 64, "one load a lane");
    if (tid < (int)(sizeof(BuildDev) / 4))
        reinterpret_cast<unsigned *>(&b)[tid] = reinterpret_cast<const unsigned *>(todo + blockIdx.x)[tid];
    __syncthreads();
    if (tid == 0) blocks[blockIdx.x] = b.tile;
    const int k = (int)uniform((unsigned)b.k), dim = 1 << k, numGates = (int)uniform((unsigned)b.numGates);
    Amp<double> *M = buf[0], *N = buf[1];
    for (int i = tid; i < dim * dim; i += kBlock) M[i] = Amp<double>{(i >> k) == (i & (dim - 1)) ? 1.0 : 0.0, 0.0};
    // pairs of a wave: dim/4 columns x dim/2 row pairs, 32 (k = 4) or 128 (k = 5)
    const int cb = k - 2, col = wave * (dim / 4) + (lane & ((1 << cb) - 1)), pairs = dim / 2;
    GateDev next{};
    for (int g = 0; g < numGates; ++g) {
        if (g % kStage == 0) {
            __syncthreads();
            stageGates(stage, gates + b.firstGate + g, min(kStage, numGates - g), tid, kBlock);
            __syncthreads();
            next = stage[0];
        }
        const GateDev G = uniformGate(next);
        next = stage[g % kStage + 1];  // past a stage's last one: unused
        if (G.kind == FlatGate::CHANNEL) {
            const unsigned b0 = 1u << (G.t & 15u), b1 = 1u << (G.t >> 4);
            const unsigned lo = ~(min(b0, b1) - 1u), hi = ~(max(b0, b1) - 1u);
            for (unsigned p = lane >> cb; p < (unsigned)pairs / 2; p += 64 >> cb) {
                unsigned r = p + (p & lo);
                r += r & hi;
                Amp<double> *p00 = M + (r << k) + col, *p11 = p00 + ((b0 | b1) << k);
                Amp<double> *p01 = p00 + (b0 << k), *p10 = p00 + (b1 << k);
                const Amp<double> x = *p00, y = *p11, v = *p01, w = *p10;
                *p00 = realTimes(G.u[2], G.u[7], G.u[3], x, y);
                *p11 = realTimes(G.u[5], G.lo, G.u[4], y, x);
                *p01 = realTimes(G.u[0], G.u[6], G.u[1], v, w);
                *p10 = realTimes(G.u[0], G.u[6], G.u[1], w, v);
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
            continue;
        }
        if (G.kind != FlatGate::MATRIXN) {
            // row r0 of pair p: p with a zero inserted at the target
            const unsigned bit = 1u << G.t, high = ~(bit - 1u);
            for (unsigned p = lane >> cb; p < (unsigned)pairs; p += 64 >> cb) {
                const unsigned r0 = p + (p & high);
                if ((r0 & G.ctrl) != G.ctrl) continue;
                Amp<double> *px = M + (r0 << k) + col, *py = px + (bit << k);
                const Amp<double> x = *px, y = *py;
                if (G.kind == FlatGate::NOT) {
                    *px = y;
                    *py = x;
                } else {
                    *px = rowTimes(G.u[0], G.u[1], G.u[2], G.u[3], x, y);
                    *py = rowTimes(G.u[4], G.u[5], G.u[6], G.u[7], x, y);
                }
            }
            // LDS accesses of one wave complete in order; keep the compiler's too
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
            continue;
        }
        const int gk = G.k, gd = 1 << gk;
        __syncthreads();  // the last matrix has been read
        for (int i = tid; i < gd * gd; i += kBlock) U[i] = mats[G.mat + i];
        __syncthreads();
        for (int r = lane >> cb; r < dim; r += 64 >> cb) {
            Amp<double> s = M[r * dim + col];
            if (((unsigned)r & G.ctrl) == G.ctrl) {
                unsigned base = (unsigned)r;
                int row = 0;
                for (int j = 0; j < gk; ++j) {
                    const unsigned q = (G.t >> (4 * j)) & 15u;
                    row |= ((r >> q) & 1) << j;
                    base &= ~(1u << q);
                }
                s = Amp<double>{0.0, 0.0};
                for (int c = 0; c < gd; ++c) {
                    unsigned rc = base;
                    for (int j = 0; j < gk; ++j) rc |= ((unsigned)(c >> j) & 1u) << ((G.t >> (4 * j)) & 15u);
                    const Amp<double> u = U[row * gd + c], x = M[rc * dim + col];
                    s.x += u.x * x.x - u.y * x.y;
                    s.y += u.x * x.y + u.y * x.x;
                }
            }
            N[r * dim + col] = s;
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        Amp<double> *sw = M;
        M = N;
        N = sw;
    }
    __syncthreads();
    // fragment (h steps + st) of each of the three matrices: Ur, Ui, Ur + Ui in FP32,
    // Ur, -(Ur + Ui), Ui - Ur in FP64
    char *dst = out + ((size_t)b.at << 10);
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
struct TileGeom {
    int pos[kMaxTB];     // the tile's qubits, ascending
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
// waves of a small register's workgroup: one chunk of a 4-qubit block each, two at 12
// bits (16 waves would leave a lane 128 registers, and two a SIMD keep it busy)
constexpr int smallWaves(int tileBits) { return tileBits >= 11 ? 8 : 1 << (tileBits - 8); }

template <typename T> struct Acc4;
template <> struct Acc4<float> { typedef f4 type; };
template <> struct Acc4<double> { typedef d4 type; };

// A block of K qubits on the chunks of one wave, IL chunks at a time: v holds the
// block's vectors, s0 the slot of each chunk of the wave.
template <typename T, int K, int WAVES, int TB>
__device__ __forceinline__ void blockChunks(char *tile, const typename Frag<T>::V *v, const BlockDev &B, int wave) {
    typedef typename Acc4<T>::type A;
    constexpr int S = 1 << (K - 2), H = K == 5 ? 2 : 1, PV = 16 / sizeof(T), NV = H * S / PV, SV = S / 4;
    constexpr int CH = (1 << (TB - 4 - K)) / WAVES, IL = K == 5 || CH < 2 ? 1 : 2;
    static_assert(CH > 0 && CH % IL == 0, "every wave has whole runs of chunks");
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
            for (int b = 0; b < TB - 4 - K; ++b) s0[l] ^= ((ch >> b) & 1) ? B.rest[b] : 0u;
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

// The blocks on a tile in LDS, one after another; a barrier behind each.
template <typename T, int WAVES, int TB>
__device__ __forceinline__ void tileBlocks(char *tile, const BlockDev *__restrict__ blocks, int numBlocks,
                                           const char *__restrict__ frags, int lane, int wave) {
    typedef typename Frag<T>::V V;
    // a 4-qubit block's vectors are loaded while the block before it multiplies
    constexpr int V4 = blockVecs<T>(4), V5 = blockVecs<T>(5);
    // waves of a 5-qubit block: small tiles have fewer chunks of it than waves
    constexpr int W5 = (1 << (TB - 9)) < WAVES ? 1 << (TB - 9) : WAVES;
    const V *next = reinterpret_cast<const V *>(frags) + lane;
    BlockDev B = blocks[0], nB = B;
    V v[V5], pre[V4];
#pragma unroll
    for (int i = 0; i < V4; ++i) pre[i] = next[i * 64];
    for (int b = 0; b < numBlocks; ++b) {
        const V *mineB = next;
        next += (B.k == 5 ? V5 : V4) * 64;
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
            if (W5 == WAVES || wave < W5) blockChunks<T, 5, W5, TB>(tile, v, B, wave);
        } else {
            blockChunks<T, 4, WAVES, TB>(tile, v, B, wave);
        }
        B = nB;
        __syncthreads();
    }
}

template <typename T, bool NT, int WAVES, int TB>
__global__ void __launch_bounds__(64 * WAVES, sizeof(T) == 4 ? 4 : 2)
    kTileSweep(Amp<T> *__restrict__ a, TileGeom geo, const BlockDev *__restrict__ blocks, int numBlocks,
               const char *__restrict__ frags) {
    // a thread moves 16 B at a time: two FP32 amplitudes or one FP64
    constexpr int PAIR = sizeof(T) == 4 ? 1 : 0, THREADS = 6 + (WAVES == 8 ? 3 : 2), J = 1 << (TB - THREADS - PAIR);
    typedef typename Frag<T>::V V;
    __shared__ __attribute__((aligned(16))) char tile[sizeof(Amp<T>) << TB];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    uint64_t addr = (uint64_t)flatBlock();
#pragma unroll
    for (int i = 0; i < TB; ++i) addr = insertZero(addr, geo.pos[i]);
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
    tileBlocks<T, WAVES, TB>(tile, blocks, numBlocks, frags, lane, wave);
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
// one launch, rounded to FP32 once at its end. One pair of amplitudes a thread (two
// at 12 qubits), one barrier a gate. Nothing but a gate's own chain bounds it (one
// workgroup): its constants, read from LDS while the gate before it runs, the
// pair's LDS reads, the products, the writes, the barrier; so the code of a gate is
// kept short: 0.4 us a gate up to 9 qubits, 0.45 at 10, 0.6 at 11, 0.9 at 12 (2x2s and
// CNOTs). 80 operations on 10 qubits, 53 gates after joins, take 26 us here; as 10 fused
// blocks of a launch each they took 45 us on the device and 340 us with the host's part
// of each block.
struct SmallGate {
    unsigned what;               // SG_*
    unsigned bit;                // the target's bit, as a byte offset of the LDS register (16 B an amplitude)
    unsigned ctrl;               // the controls' bits, likewise; SG_CHANNEL: the column bit
    float lo;                    // SG_CHANNEL: d11Lo
    alignas(16) double u[8];     // the matrix, (re, im) by rows; SG_CHANNEL: f, g, d00, d01, d10, d11, fLo, d00Lo
};
enum { SG_GENERAL = 0, SG_NOT = 1, SG_PHASE = 2, SG_REAL = 3, SG_CHANNEL = 4 };  // SG_PHASE: diag(1, u)
constexpr int kSmallStage = 256;
constexpr int kSmallThreads = 1024;

template <typename T>
__global__ void __launch_bounds__(kSmallThreads) kSmallCircuit(Amp<T> *__restrict__ a, int n,
                                                               const SmallGate *__restrict__ gates, int numGates) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    const unsigned dim = 1u << n, step = blockDim.x, tid = threadIdx.x;
    SmallGate *stage = reinterpret_cast<SmallGate *>(smem + (sizeof(Amp<double>) << n));
    auto at = [&](unsigned off) -> Amp<double> & { return *reinterpret_cast<Amp<double> *>(smem + off); };
    for (unsigned i = tid; i < dim; i += step) at(16u * i) = Amp<double>{(double)a[i].x, (double)a[i].y};
    uint4 nextHead{};
    d8 nextU = {0, 0, 0, 0, 0, 0, 0, 0};
    for (int g = 0; g < numGates; ++g) {
        if (g % kSmallStage == 0) {
            __syncthreads();
            stageGates(stage, gates + g, min(kSmallStage, numGates - g), (int)tid, (int)step);
            __syncthreads();
            nextHead = *reinterpret_cast<const uint4 *>(stage);
            nextU = matrixOf(stage[0].u);
        }
        const unsigned what = uniform(nextHead.x), bit = uniform(nextHead.y), ctrl = uniform(nextHead.z);
        const unsigned high = ~(bit - 1u);
        const float lo = __uint_as_float(nextHead.w);
        const d8 u = nextU;
        // past a stage's last one: unused
        nextHead = *reinterpret_cast<const uint4 *>(stage + g % kSmallStage + 1);
        nextU = matrixOf(stage[g % kSmallStage + 1].u);
        if (what == SG_CHANNEL) {
            const unsigned low = ~(min(bit, ctrl) - 1u), top = ~(max(bit, ctrl) - 1u);
            // FP32 amplitudes hold nothing of the low parts, 3 % of a 3-qubit list's time
            for (unsigned w = 16u * tid; w < 4u * dim; w += 16u * step) {
                unsigned i = w + (w & low);
                i += i & top;
                Amp<double> &A = at(i), &B = at(i + bit), &C = at(i + ctrl), &D = at(i + bit + ctrl);
                const Amp<double> x = A, y = D, v = B, z = C;
                if constexpr (sizeof(T) == 4) {
                    A = Amp<double>{u[2] * x.x + u[3] * y.x, u[2] * x.y + u[3] * y.y};
                    D = Amp<double>{u[4] * x.x + u[5] * y.x, u[4] * x.y + u[5] * y.y};
                    B = Amp<double>{u[0] * v.x + u[1] * z.x, u[0] * v.y + u[1] * z.y};
                    C = Amp<double>{u[1] * v.x + u[0] * z.x, u[1] * v.y + u[0] * z.y};
                } else {
                    A = realTimes(u[2], u[7], u[3], x, y);
                    D = realTimes(u[5], lo, u[4], y, x);
                    B = realTimes(u[0], u[6], u[1], v, z);
                    C = realTimes(u[0], u[6], u[1], z, v);
                }
            }
            __syncthreads();
            continue;
        }
        for (unsigned w = 16u * tid; w < 8u * dim; w += 16u * step) {
            const unsigned i = w + (w & high);  // the pair's index with a zero inserted at the target
            if ((i & ctrl) != ctrl) continue;
            Amp<double> &X = at(i), &Y = at(i + bit);
            if (what == SG_NOT) {
                const Amp<double> x = X, y = Y;
                X = y;
                Y = x;
            } else if (what == SG_PHASE) {
                const Amp<double> y = Y;
                Y = Amp<double>{u[6] * y.x - u[7] * y.y, u[6] * y.y + u[7] * y.x};
            } else if (what == SG_REAL) {
                const Amp<double> x = X, y = Y;
                X = Amp<double>{u[0] * x.x + u[2] * y.x, u[0] * x.y + u[2] * y.y};
                Y = Amp<double>{u[4] * x.x + u[6] * y.x, u[4] * x.y + u[6] * y.y};
            } else {
                const Amp<double> x = X, y = Y;
                X = rowTimes(u[0], u[1], u[2], u[3], x, y);
                Y = rowTimes(u[4], u[5], u[6], u[7], x, y);
            }
        }
        __syncthreads();
    }
    for (unsigned i = tid; i < dim; i += step) a[i] = Amp<T>{(T)at(16u * i).x, (T)at(16u * i).y};
}

// A planned list on a small register: the whole register is one workgroup's tile, in
// FP64 for both storage precisions (FP32 results are rounded once: 1.4e-7 from the
// 64-bit state after 400 gates on 12 qubits, 6.1e-7 with FP32 blocks). Up to 10 qubits a
// 4-qubit block is one chain of LDS reads, 12 products and writes, 0.6 us; at 12 the
// products of 16 chunks on one CU are 1.3 us of its 2. 400 random gates make 41 to 47
// blocks, 20 brick layers 19 to 28.
template <typename S, int TB>
__global__ void __launch_bounds__(64 * smallWaves(TB)) kSmallBlocks(Amp<S> *__restrict__ a, int n,
                                                                   const BlockDev *__restrict__ blocks, int numBlocks,
                                                                   const char *__restrict__ frags) {
    constexpr int WAVES = smallWaves(TB);
    __shared__ __attribute__((aligned(16))) char tile[sizeof(Amp<double>) << TB];
    const unsigned tid = threadIdx.x, dim = 1u << n;
    auto at = [&](unsigned i) -> Amp<double> & {
        return *reinterpret_cast<Amp<double> *>(tile + tileSlot<double>(i) * sizeof(Amp<double>));
    };
    for (unsigned i = tid; i < 1u << TB; i += 64 * WAVES)
        at(i) = i < dim ? Amp<double>{(double)a[i].x, (double)a[i].y} : Amp<double>{0.0, 0.0};
    __syncthreads();
    tileBlocks<double, WAVES, TB>(tile, blocks, numBlocks, frags, tid & 63,
                                  __builtin_amdgcn_readfirstlane((int)tid >> 6));
    for (unsigned i = tid; i < dim; i += 64 * WAVES) a[i] = Amp<S>{(S)at(i).x, (S)at(i).y};
}

// ---- host side -----------------------------------------------------------------------
size_t align16(size_t x) { return (x + 15) & ~(size_t)15; }

// One upload holds the build list, the gates and their matrices.
struct Upload {
    size_t todo, gates, mats, bytes;
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
    u.bytes = u.mats + entries * sizeof(Amp<double>);
    return u;
}

void fillBuild(const SweepPlan &plan, const FlatGate *gates, int firstBlock, int numBlocks, const Upload &u,
               const unsigned *place, char *host) {
    BuildDev *todo = reinterpret_cast<BuildDev *>(host + u.todo);
    GateDev *gd = reinterpret_cast<GateDev *>(host + u.gates);
    Amp<double> *mats = reinterpret_cast<Amp<double> *>(host + u.mats);
    int at = 0, mat = 0;
    for (int i = 0; i < numBlocks; ++i) {
        const SweepBlock &b = plan.blocks[firstBlock + i];
        todo[i] = BuildDev{};
        todo[i].firstGate = at;
        todo[i].numGates = b.numGates;
        todo[i].k = b.k;
        todo[i].at = place[i];
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
                for (int j = 0; j < f.k; ++j) d.t |= (unsigned)local(f.targs[j]) << (4 * j);
                d.mat = mat;
                const int entries = 1 << (2 * f.k);
                for (int e = 0; e < entries; ++e) mats[mat + e] = Amp<double>{f.uN[e].re, f.uN[e].im};
                mat += entries;
            } else if (f.kind == FlatGate::CHANNEL) {
                d.t = (unsigned)local(f.target) | (unsigned)local(f.k) << 4;
                for (int e = 0; e < 4; ++e) {
                    d.u[2 * e] = f.u[e].re;
                    d.u[2 * e + 1] = f.u[e].im;
                }
                d.lo = f.lo;
            } else {
                d.t = (unsigned)local(f.target);
                for (int e = 0; e < 4; ++e) {
                    d.u[2 * e] = f.u[e].re;
                    d.u[2 * e + 1] = f.u[e].im;
                }
            }
        }
    }
}

// the tile's qubits, ascending; returns how many
int tilePositions(uint64_t tile, int pos[kMaxTB]) {
    const int bits = __builtin_popcountll(tile);
    if (bits > kMaxTB || bits < 9) {
        std::fprintf(stderr, "libquest_mi355x: a planned tile has %d qubits\n", bits);
        std::abort();
    }
    int n = 0;
    for (uint64_t m = tile; m; m &= m - 1) pos[n++] = __builtin_ctzll(m);
    return n;
}

template <typename T>
void blockSlots(const SweepBlock &b, const int *pos, int tb, BuildDev &todo) {
    constexpr int R = sizeof(T) == 4 ? 4 : 3;   // columns per bank cycle: 2^R lanes
    todo.tile.k = b.k;
    int t[kSweepBlockQubits];
    bool used[kMaxTB] = {};
    for (int j = 0; j < b.k; ++j) {
        t[j] = -1;
        for (int i = 0; i < tb; ++i)
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
    for (int i = 0; i < tb && nc < R; ++i)
        if (!used[i] && !residue[i % R]) {
            residue[i % R] = used[i] = true;
            cols[nc++] = i;
        }
    for (int i = 0; i < tb && nc < 4; ++i)
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
    for (int i = 0, r = 0; i < tb; ++i)
        if (!used[i]) todo.tile.rest[r++] = slot(i);
}

// LDS slots of blocks [firstBlock, firstBlock + num)
void fillBlocks(int prec, const SweepPlan &plan, int firstBlock, int num, const Upload &u, char *host) {
    BuildDev *todo = reinterpret_cast<BuildDev *>(host + u.todo);
    for (const Sweep &w : plan.sweeps) {
        const int from = std::max(w.firstBlock, firstBlock);
        const int to = std::min(w.firstBlock + w.numBlocks, firstBlock + num);
        if (w.lone >= 0 || from >= to) continue;
        int pos[kMaxTB];
        const int tb = tilePositions(w.tile, pos);
        for (int b = from; b < to; ++b)
            QMX_DISPATCH(prec, T, { blockSlots<T>(plan.blocks[b], pos, tb, todo[b - firstBlock]); });
    }
}

// where the vectors of blocks [firstBlock, firstBlock + num) lie, in KiB, and their end
void placeBlocks(int prec, const SweepPlan &plan, int firstBlock, int num, std::vector<unsigned> &at) {
    at.resize(num + 1);
    at[0] = 0;
    QMX_DISPATCH(prec, T, {
        for (int i = 0; i < num; ++i) at[i + 1] = at[i] + (unsigned)blockVecs<T>(plan.blocks[firstBlock + i].k);
    });
}

// from `src`, an upload that the device can read
void launchBuild(int prec, int numBlocks, const Upload &u, const char *src, char *frags, BlockDev *blocks) {
    const BuildDev *todo = reinterpret_cast<const BuildDev *>(src + u.todo);
    const GateDev *gd = reinterpret_cast<const GateDev *>(src + u.gates);
    const Amp<double> *mats = reinterpret_cast<const Amp<double> *>(src + u.mats);
    QMX_DISPATCH(prec, T, {
        hipLaunchKernelGGL(kBuildBlocks<T>, dim3(numBlocks), dim3(kBlock), 0, hstream(), todo, gd, mats, frags,
                           blocks);
    });
    checkLaunch("sweep block matrices");
}

template <typename T, bool NT, int WAVES, int TB>
void launchTiles(QuregDev *q, const Sweep &w, const BlockDev *blocks, const char *frags) {
    constexpr int PAIR = sizeof(T) == 4 ? 1 : 0, THREADS = 6 + (WAVES == 8 ? 3 : 2), J = 1 << (TB - THREADS - PAIR);
    TileGeom geo{};
    if (tilePositions(w.tile, geo.pos) != TB) {
        std::fprintf(stderr, "libquest_mi355x: a sweep's tile does not have %d qubits\n", TB);
        std::abort();
    }
    for (int j = 0; j < J; ++j)
        for (int i = 0; THREADS + PAIR + i < TB; ++i)
            if ((j >> i) & 1) {
                geo.jAddr[j] |= 1ull << geo.pos[THREADS + PAIR + i];
                geo.jSlot[j] ^= slotBit<T>(THREADS + PAIR + i) * (unsigned)sizeof(Amp<T>);
            }
    hipLaunchKernelGGL((kTileSweep<T, NT, WAVES, TB>), gridOf(q->numAmps >> TB), dim3(64 * WAVES), 0, hstream(),
                       (Amp<T> *)q->amps, geo, blocks, w.numBlocks, frags);
    checkLaunch("tile sweep");
}

// Four waves a tile; eight where tiles of 12 qubits are too few to fill the CUs with
// workgroups of four (4 of 32 KiB or 2 of 64 KiB fit a CU; eight waves on large
// registers: 33.6 instead of 30.8 ms for the 30-qubit FP32 period, 9.8 instead of
// 7.7 for the 27-qubit FP64 one). Nontemporal accesses where the register outgrows
// the last-level cache.
template <typename T>
void launchSweep(QuregDev *q, const Sweep &w, const BlockDev *blocks, const char *frags) {
    constexpr int perCU = sizeof(T) == 4 ? 4 : 2;
    if (__builtin_popcountll(w.tile) < kSweepTileBits)
        launchTiles<T, false, 4, kSweepTileBits - 1>(q, w, blocks, frags);
    else if ((q->numAmps >> kSweepTileBits) < (long long)perCU * numCUs())
        launchTiles<T, false, 8, kSweepTileBits>(q, w, blocks, frags);
    else if (q->numAmps * (long long)sizeof(Amp<T>) > (256ll << 20))
        launchTiles<T, true, 4, kSweepTileBits>(q, w, blocks, frags);
    else
        launchTiles<T, false, 4, kSweepTileBits>(q, w, blocks, frags);
}

void launchSmallBlocks(QuregDev *q, const Sweep &w, const BlockDev *blocks, const char *frags) {
    QMX_DISPATCH(q->prec, S, {
        auto launch = [&](auto kernel, int tb) {
            hipLaunchKernelGGL(kernel, dim3(1), dim3(64 * smallWaves(tb)), 0, hstream(), (Amp<S> *)q->amps,
                               q->numQubits, blocks, w.numBlocks, frags);
        };
        switch (__builtin_popcountll(w.tile)) {
            case 9: launch(kSmallBlocks<S, 9>, 9); break;
            case 10: launch(kSmallBlocks<S, 10>, 10); break;
            case 11: launch(kSmallBlocks<S, 11>, 11); break;
            default: launch(kSmallBlocks<S, 12>, 12); break;
        }
    });
    checkLaunch("small register's blocks");
}

void runSweeps(QuregDev *q, const SweepPlan &plan, const FlatGate *gates, int first, int last, int firstBlock,
               const BlockDev *blocks, const std::vector<unsigned> &place, const char *frags) {
    for (int s = first; s < last; ++s) {
        const Sweep &w = plan.sweeps[s];
        const bool small = smallStateVector(q);
        if (w.lone >= 0) {
            if (small && gates[w.lone].kind != FlatGate::MATRIXN) smallCircuit(q, gates + w.lone, 1);
            else applyFlatGate(q, gates[w.lone]);
            continue;
        }
        const BlockDev *b = blocks + (w.firstBlock - firstBlock);
        const char *f = frags + ((size_t)place[w.firstBlock - firstBlock] << 10);
        if (small) launchSmallBlocks(q, w, b, f);
        else QMX_DISPATCH(q->prec, T, { launchSweep<T>(q, w, b, f); });
    }
}

// The library's workspace for lists applied once. The gates lie in pinned host memory,
// where the one kernel that wants them reads them (17 qubits FP64, 300 gates: 148 us,
// 178 with a copy to the device before it and one of the results): two buffers in
// turn, each rewritten after the event behind its last reader. The fragments and
// descriptions of a batch of blocks are on the device, rewritten by work queued
// behind everything that read them. All grow to what a batch needs and no further.
constexpr int kBatchBlocks = 256;
struct Workspace {
    struct Host {
        char *p = nullptr;
        size_t bytes = 0;
        hipEvent_t ev = nullptr;
        bool used = false;
    } host[2];
    int at = 0;
    char *frags = nullptr;
    int fragBlocks = 0;
    std::vector<unsigned> place;

    char *hostRoom(size_t need) {
        at ^= 1;
        Host &h = host[at];
        if (!h.ev) QMX_HIP_CHECK(hipEventCreateWithFlags(&h.ev, hipEventDisableTiming));
        if (h.used) QMX_HIP_CHECK(hipEventSynchronize(h.ev));
        if (need > h.bytes) {
            if (h.p) QMX_HIP_CHECK(hipHostFree(h.p));
            h.bytes = std::max(need, (size_t)1 << 17);
            QMX_HIP_CHECK(hipHostMalloc(reinterpret_cast<void **>(&h.p), h.bytes, hipHostMallocDefault));
            h.used = false;
        }
        return h.p;
    }
    // after the launch that reads the host buffer
    void launched() {
        QMX_HIP_CHECK(hipEventRecord(host[at].ev, hstream()));
        host[at].used = true;
    }
    char *fragRoom(int blocks) {
        if (blocks > fragBlocks) {
            if (frags) devFree(frags);
            fragBlocks = std::max(blocks, 32);
            frags = static_cast<char *>(devAlloc((size_t)fragBlocks * (kMaxBlockBytes + sizeof(BlockDev))));
        }
        return frags;
    }
    BlockDev *blocks() const { return reinterpret_cast<BlockDev *>(frags + (size_t)fragBlocks * kMaxBlockBytes); }
} g_ws;

// Blocks [firstBlock, firstBlock + num) on the device: their vectors where `place` says,
// their descriptions at blocks.
void buildBatch(int prec, const SweepPlan &plan, const FlatGate *gates, int firstBlock, int num,
                const unsigned *place, char *frags, BlockDev *blocks) {
    const Upload u = layoutOf(plan, gates, firstBlock, num);
    char *host = g_ws.hostRoom(u.bytes);
    fillBuild(plan, gates, firstBlock, num, u, place, host);
    fillBlocks(prec, plan, firstBlock, num, u, host);
    launchBuild(prec, num, u, host, frags, blocks);
    g_ws.launched();
}

}  // namespace

struct SweepProgram {
    int prec;
    char *frags = nullptr;
    size_t bytes = 0;
    BlockDev *blocks = nullptr;
    std::vector<unsigned> place;
};

SweepProgram *sweepProgramCreate(int prec, const SweepPlan &plan, const FlatGate *gates) {
    auto *p = new SweepProgram;
    p->prec = prec;
    const int n = (int)plan.blocks.size();
    if (n == 0) return p;
    runtimeInit();
    placeBlocks(prec, plan, 0, n, p->place);
    const size_t fragBytes = (size_t)p->place[n] << 10;
    p->bytes = fragBytes + (size_t)n * sizeof(BlockDev);
    p->frags = static_cast<char *>(poolAlloc(p->bytes));
    if (!p->frags) {
        std::fprintf(stderr, "libquest_mi355x: no device memory for a circuit's blocks (%zu bytes)\n", p->bytes);
        std::abort();
    }
    p->blocks = reinterpret_cast<BlockDev *>(p->frags + fragBytes);
    for (int b = 0; b < n; b += kBatchBlocks)
        buildBatch(prec, plan, gates, b, std::min(kBatchBlocks, n - b), p->place.data() + b, p->frags, p->blocks + b);
    return p;
}

void sweepProgramFree(SweepProgram *p) {
    if (!p) return;
    poolFree(p->frags, p->bytes);
    delete p;
}

void sweepProgramRun(QuregDev *q, const SweepProgram *p, const SweepPlan &plan, const FlatGate *gates, int first,
                     int last) {
    runSweeps(q, plan, gates, first, last, 0, p->blocks, p->place, p->frags);
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
            runSweeps(q, plan, gates, first, last, 0, nullptr, g_ws.place, nullptr);
            first = last;
            continue;
        }
        char *frags = g_ws.fragRoom(n);
        placeBlocks(q->prec, plan, firstBlock, n, g_ws.place);
        buildBatch(q->prec, plan, gates, firstBlock, n, g_ws.place.data(), frags, g_ws.blocks());
        runSweeps(q, plan, gates, first, last, firstBlock, g_ws.blocks(), g_ws.place, frags);
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
    if (g.kind == FlatGate::CHANNEL) {
        // entry e = row bit + 2 * column bit
        const int bits[2] = {g.target, g.k};
        Cplx S[16] = {};
        S[0] = {g.u[1].re, 0};
        S[3] = {g.u[1].im, 0};
        S[12] = {g.u[2].re, 0};
        S[15] = {g.u[2].im, 0};
        S[5] = S[10] = {g.u[0].re, 0};
        S[6] = S[9] = {g.u[0].im, 0};
        applyDense(q, bits, 2, S);
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
    if (f.kind == FlatGate::CHANNEL) return SG_CHANNEL;
    auto is = [](const Cplx &z, double re) { return z.re == re && z.im == 0; };
    if (is(f.u[0], 1) && is(f.u[1], 0) && is(f.u[2], 0)) return SG_PHASE;
    for (const Cplx &z : f.u)
        if (z.im != 0) return SG_GENERAL;
    return SG_REAL;
}

void smallCircuit(QuregDev *q, const FlatGate *gates, int count) {
    runtimeInit();
    // gates per launch: bounds the upload
    constexpr int kPerLaunch = 4096;
    const int n = q->numQubits;
    const unsigned threads = std::min((unsigned)kSmallThreads, std::max(64u, 1u << (n - 1)));
    constexpr size_t stageBytes = (kSmallStage + 1) * sizeof(SmallGate);
    const size_t lds = (sizeof(Amp<double>) << n) + stageBytes;
    for (int first = 0; first < count; first += kPerLaunch) {
        const int num = std::min(kPerLaunch, count - first);
        SmallGate *h = reinterpret_cast<SmallGate *>(g_ws.hostRoom((size_t)num * sizeof(SmallGate)));
        for (int i = 0; i < num; ++i) {
            const FlatGate &f = gates[first + i];
            SmallGate &d = h[i];
            d.what = (unsigned)smallKind(f);
            d.bit = 16u << f.target;
            d.ctrl = f.kind == FlatGate::CHANNEL ? 16u << f.k : 16u * (unsigned)f.ctrl;
            d.lo = f.lo;
            for (int e = 0; e < 4; ++e) {
                d.u[2 * e] = f.u[e].re;
                d.u[2 * e + 1] = f.u[e].im;
            }
        }
        QMX_DISPATCH(q->prec, T, {
            static bool ldsAllowed = false;
            if (!ldsAllowed) {
                if (!allowDynamicLds(reinterpret_cast<const void *>(&kSmallCircuit<T>),
                                     (sizeof(Amp<double>) << kSmallCircuitQubits) + stageBytes,
                                     "a small register's circuit"))
                    std::abort();
                ldsAllowed = true;
            }
            hipLaunchKernelGGL(kSmallCircuit<T>, dim3(1), dim3(threads), lds, hstream(), (Amp<T> *)q->amps, n, h,
                               num);
        });
        checkLaunch("smallCircuit");
        g_ws.launched();
    }
}

}  // namespace qmx
