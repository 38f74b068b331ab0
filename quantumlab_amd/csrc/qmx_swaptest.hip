// Batched swap tests for quantum k-means (QKMeans): thousands of registers of
// uneven size in one launch.
//
// Reference construction (QuantumLab): a point v1 and a centroid v2 of length
// 2^q are amplitude-encoded into q-qubit registers by a tree of uniformly
// controlled Ry rotations (AmplitudeEncodeCuda.cu:61-150 angles,
// :498-533 ExchangeToYGate, FRGate.cu:154-252 FRy), and swap-tested on a
// (2q+1)-qubit register: H(anc); AE(v1) on qubits 1..q; AE(v2) on q+1..2q;
// q controlled-SWAPs (anc, i, i+q); H(anc) (SwapTest.cpp:70-123). P(anc = 0)
// gives the overlap.
//
// MI355X form:
//  * kAEState: the encoding tree applied to |0...0> for every vector at once,
//    one workgroup per vector: level-by-level angles theta = 2 atan2(right,
//    left) (the reference's recursion), then each amplitude as the product of
//    cos/sin(theta/2) along its path — the state the Ry tree prepares, in
//    O(2^q) instead of 2^q gates of O(2^(2q+1)) each.
//  * kOverlap: after H and the two encodings the register is |+>|a>|b>; the
//    CSWAP ladder and the final H leave ancilla-0 amplitudes
//    (a_x b_y + a_y b_x)/2, so P(anc = 0) = 1/4 sum_xy (a_x b_y + a_y b_x)^2.
//    The registers are real, and the double sum factors exactly into
//    (|a|^2 |b|^2 + <a, b>^2)/2: three sums of 2^q products instead of one of
//    2^(2q) squares. The inner products of 16 points with 16 centroids are one
//    FP64 matrix product over the registers' rows.
//  * one k-means iteration = inner products, P0 and argmax assignment in one
//    launch -> partial centroid sums -> centroid means, normalised and
//    re-encoded at every size; three launches, captured once as a hipGraph and
//    replayed.
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <limits>
#include <vector>

#include "qmx_device.h"
#include "quest_mi355x.h"

namespace qmx {

namespace {

constexpr int kMinQ = 1, kMaxQ = 12;

// one workgroup's points: up to 16 * (4 / split) consecutive entries of the
// size-ordered point list, all of register size q; `split` waves share a
// register's rows
struct Tile {
    int first, count;
    int q;
    int split;
};

// ---- amplitude encoding -----------------------------------------------------
// cos and sin of half the reference's angle 2 atan2(s, c): c/h and s/h with
// h = hypot(c, s). The quotients replace an atan2, a cosine and a sine per node
// (the levels of the tree are a serial chain, so their latency is the kernel's
// time: 54 us for one 1024-entry vector before). Where h is zero, not finite or
// so small that it has lost digits, the angle itself is used.
__device__ __forceinline__ void angleFactors(double c, double s, double &cs, double &sn) {
    const double h = hypot(c, s);
    if (h > 1e-280 && h < std::numeric_limits<double>::infinity()) {
        cs = c / h;
        sn = s / h;
    } else {
        const double theta = 2.0 * atan2(s, c);
        cs = cos(theta / 2.0);
        sn = sin(theta / 2.0);
    }
}

// The encoding tree over mag[0 .. 2^q) (LDS, overwritten), one workgroup; cs, sn:
// 2^q doubles each in LDS. Writes the encoded state to o (storage precision)
// and its squared norm as stored to *norm2 (nullptr: not wanted).
template <typename T>
__device__ __forceinline__ void encodeTree(double *mag, double *cs, double *sn, int q, T *__restrict__ o,
                                           double *norm2) {
    const int D = 1 << q;
    // level l: pairs (left = k 2^(l+1), right = left + 2^l) of the running
    // magnitudes; angle index = D - 2^(q-l) + k (AmplitudeEncodeCuda.cu:126-129)
    for (int l = 0; l < q; ++l) {
        const int pairs = D >> (l + 1);
        const int base = D - (D >> l);
        for (int k = threadIdx.x; k < pairs; k += kBlock) {
            const int left = k << (l + 1), right = left + (1 << l);
            const double c = mag[left], s = mag[right];
            angleFactors(c, s, cs[base + k], sn[base + k]);
            if (pairs != 1) {
                // magnitudes at or below the arithmetic's epsilon are zeroed, as
                // the reference does with _QL_FLT_EPSILON (QLFloat.h:120,139: the
                // epsilon of the precision the angles are computed in)
                const double m2 = c * c + s * s;
                mag[left] = m2 > std::numeric_limits<double>::epsilon() ? sqrt(m2) : 0.0;
            }
        }
        __syncthreads();
    }
    // amplitude of basis state x: product over levels of cos (bit 0) / sin (bit 1)
    Acc acc[1];
    for (int x = threadIdx.x; x < D; x += kBlock) {
        double amp = 1.0;
        for (int l = 0; l < q; ++l) {
            const int idx = D - (D >> l) + (x >> (l + 1));
            amp *= ((x >> l) & 1) ? sn[idx] : cs[idx];
        }
        o[x] = (T)amp;
        const double stored = (double)(T)amp;
        acc[0].add(stored * stored);
    }
    if (!norm2) return;  // the same for every thread
    double tot[1];
    blockReduce<1>(acc, tot);
    if (threadIdx.x == 0) *norm2 = tot[0];
}

// vectors: packed real FP64 inputs (length 2^q each, offsets in off[]); out:
// the encoded states in the storage precision T (same packing), norm2 (may be
// nullptr) their squared norms. The encoding is O(2^q) per vector, so it is
// computed in FP64 for both storage precisions and each amplitude is rounded
// once when stored. One workgroup per vector; LDS holds the magnitudes and the
// cos/sin factors of the 2^q - 1 angles.
template <typename T>
__global__ void __launch_bounds__(kBlock) kAEState(const double *__restrict__ vecs, const long long *__restrict__ off,
                                                   const int *__restrict__ qs, T *__restrict__ out,
                                                   double *__restrict__ norm2, int count) {
    extern __shared__ unsigned char smem[];
    const int v = blockIdx.x;
    if (v >= count) return;
    const int q = qs[v];
    const int D = 1 << q;
    double *mag = reinterpret_cast<double *>(smem);
    const double *in = vecs + off[v];
    for (int i = threadIdx.x; i < D; i += kBlock) mag[i] = in[i];
    __syncthreads();
    encodeTree<T>(mag, mag + D, mag + 2 * D, q, out + off[v], norm2 ? norm2 + v : nullptr);
}

// ---- inner products, P0 and assignment ----------------------------------------
// P0[p][c] = (|a|^2 |b|^2 + <a, b>^2)/2 and each point's best centroid (largest
// P0, ties to the lowest index). A wave takes 16 points of one size and 16
// centroids at a time on v_mfma_f64_16x16x4f64: lane l holds point l%16 and
// centroid l%16 at row 4 (l/16) + k of each run of 16 rows, k = 0..3 in four
// products, so a lane reads four consecutive rows at once (the order of the
// rows in the sum is free). FP32 registers are widened first: every product and
// sum is FP64. The result's lane l holds points l/16 + 4v, centroid l%16.
//
// What bounds it: the registers are read once per iteration (FP32, 4096 points
// of 16..1024 amplitudes: 4.8 MB, from the caches) and the products take ~1 us
// of the matrix cores, so it is the latency of a wave's serial chain of loads
// and products; `split` waves divide a register's rows (4 from 256 rows, 2 from
// 64) and their sums meet in LDS. Replaces 4^q amplitudes formed on the matrix
// cores and squared on the VALU (490 us a launch at that size; bound there by
// the squares).
constexpr int kWaves = kBlock / 64;
typedef double d4v __attribute__((ext_vector_type(4)));

// rows i .. i+3 of a register of D rows, zeros past its end. `vec`: registers
// start at multiples of 4 rows, so four rows are one aligned access
template <typename T>
__device__ __forceinline__ d4v rows4(const T *__restrict__ a, int i, int D, bool vec) {
    typedef T V __attribute__((ext_vector_type(4)));
    if (vec) {
        if (i >= D) return d4v{0, 0, 0, 0};
        // 16 B units: FP64 offsets of 4 rows are 32 B apart
        const V v = *reinterpret_cast<const V *>(a + i);
        return d4v{(double)v.x, (double)v.y, (double)v.z, (double)v.w};
    }
    d4v r;
#pragma unroll
    for (int k = 0; k < 4; ++k) r[k] = i + k < D ? (double)a[i + k] : 0.0;
    return r;
}

template <typename T>
__global__ void __launch_bounds__(kBlock) kOverlap(const Tile *__restrict__ tiles, const int *__restrict__ order,
                                                   const T *__restrict__ pointAE, const long long *__restrict__ pOff,
                                                   const double *__restrict__ pNorm, const T *__restrict__ centAE,
                                                   const long long *__restrict__ cOff,
                                                   const double *__restrict__ cNorm, int C, int qLo, int vec,
                                                   double *__restrict__ p0, int *__restrict__ assign) {
    __shared__ d4v part[kWaves][64];
    const Tile t = tiles[blockIdx.x];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int col = lane & 15, kq = lane >> 4;
    const int D = 1 << t.q;
    const int mine = wave / t.split, share = wave % t.split;   // point group, part of the rows
    const int count = min(16, t.count - 16 * mine);            // may be <= 0: a wave without points
    const int nx = D / t.split < 16 ? 16 : D / t.split;        // split > 1 only from 64 rows
    const int *ids = order + t.first + 16 * mine;
    const int pm = col < count ? ids[col] : -1;
    const T *a = pm >= 0 ? pointAE + pOff[pm] : pointAE;
    // best centroid so far of points l/16 + 4v (every lane of the 16 alike)
    double best[4];
    int bestC[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        best[v] = -std::numeric_limits<double>::infinity();
        bestC[v] = 0;
    }
    for (int c0 = 0; c0 < C; c0 += 16) {
        const int c = c0 + col;
        const T *b = centAE + cOff[(t.q - qLo) * C + (c < C ? c : C - 1)];
        d4v acc = {0, 0, 0, 0};
        if (count > 0)
            for (int s = share * nx; s < (share + 1) * nx; s += 16) {
                const int i = s + 4 * kq;
                const d4v x = pm >= 0 ? rows4<T>(a, i, D, vec) : d4v{0, 0, 0, 0};
                const d4v y = rows4<T>(b, i, D, vec);
#pragma unroll
                for (int k = 0; k < 4; ++k) acc = __builtin_amdgcn_mfma_f64_16x16x4f64(x[k], y[k], acc, 0, 0, 0);
            }
        if (t.split > 1) {  // the same for the whole workgroup
            part[wave][lane] = acc;
            __syncthreads();
            if (share == 0)
                for (int k = 1; k < t.split; ++k) acc += part[wave + k][lane];
            __syncthreads();
        }
        if (share != 0 || count <= 0) continue;
        const double bb = c < C ? cNorm[(t.q - qLo) * C + c] : 0.0;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int row = kq + 4 * v;
            const int p = row < count ? ids[row] : -1;
            double val = -std::numeric_limits<double>::infinity();
            int at = c;
            if (p >= 0 && c < C) {
                val = 0.5 * (pNorm[p] * bb + acc[v] * acc[v]);
                p0[(size_t)p * C + c] = val;
                // a P0 that is not a number is never larger than another, and as
                // the first one it stays
                if (!(val == val)) val = c == 0 ? std::numeric_limits<double>::infinity()
                                                : -std::numeric_limits<double>::infinity();
            }
#pragma unroll
            for (int off = 1; off < 16; off <<= 1) {
                const double ov = __shfl_xor(val, off, 64);
                const int oc = __shfl_xor(at, off, 64);
                if (ov > val || (ov == val && oc < at)) {
                    val = ov;
                    at = oc;
                }
            }
            if (val > best[v]) {
                best[v] = val;
                bestC[v] = at;
            }
        }
    }
    if (share != 0 || col != 0) return;
#pragma unroll
    for (int v = 0; v < 4; ++v)
        if (kq + 4 * v < count) assign[ids[kq + 4 * v]] = bestC[v];
}

// ---- centroid means --------------------------------------------------------------
// means over assigned points, coordinate by coordinate (points only contribute
// their own 2^q coordinates); empty clusters keep their centroid. Stage 1
// (kCentroidPartial): one workgroup per (centroid, 256-coordinate slice, chunk
// of points) writes the chunk's sum and count; stage 2 (kCentroidUpdate) adds
// the chunks in order. FP64, deterministic.
// The chunk's members are first listed in LDS, 256 assignments at a time, so
// their coordinates are loads that do not wait for one another (a loop over all
// points that loaded each member's coordinates in turn took 30 us at 4096
// points and 16 centroids).
constexpr int kMeanChunks = 16;

__global__ void __launch_bounds__(kBlock) kCentroidPartial(const double *__restrict__ pointsV,
                                                           const long long *__restrict__ pOff,
                                                           const int *__restrict__ pQ, const int *__restrict__ assign,
                                                           int P, int C, int maxQ, double *__restrict__ sums,
                                                           int *__restrict__ counts, int *__restrict__ members) {
    __shared__ long long listOff[kBlock];
    __shared__ int listD[kBlock];
    __shared__ int waveHits[kWaves], waveMembers[kWaves];
    const int dim = 1 << maxQ;
    const int slices = dim / kBlock > 0 ? dim / kBlock : 1;
    const int chunk = blockIdx.x % kMeanChunks;
    const int cs = blockIdx.x / kMeanChunks;
    const int c = cs / slices;
    const int j0 = (cs % slices) * kBlock, j = j0 + threadIdx.x;
    const int per = (P + kMeanChunks - 1) / kMeanChunks;
    const int p0 = chunk * per, p1 = p0 + per < P ? p0 + per : P;
    if (c >= C) return;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    double sum = 0.0;
    int cnt = 0, mem = 0;
    for (int base = p0; base < p1; base += kBlock) {
        const int p = base + threadIdx.x;
        const bool in = p < p1 && assign[p] == c;
        const int D = in ? 1 << pQ[p] : 0;
        const bool hit = D > j0;  // has coordinates in this slice
        const unsigned long long hits = __ballot(hit);
        const unsigned long long ins = __ballot(in);
        if (lane == 0) {
            waveHits[wave] = __popcll(hits);
            waveMembers[wave] = __popcll(ins);
        }
        __syncthreads();
        int at = __popcll(hits & ((1ull << lane) - 1ull)), total = 0;
        for (int w = 0; w < kWaves; ++w) {
            if (w < wave) at += waveHits[w];
            total += waveHits[w];
            mem += waveMembers[w];
        }
        if (hit) {
            listOff[at] = pOff[p];
            listD[at] = D;
        }
        __syncthreads();
        for (int i = 0; i < total; i += 8) {
            double v[8];
            bool ok[8];
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                ok[k] = i + k < total && j < listD[i + k < total ? i + k : 0];
                v[k] = ok[k] ? pointsV[listOff[i + k] + j] : 0.0;
            }
#pragma unroll
            for (int k = 0; k < 8; ++k)
                if (ok[k]) {
                    sum += v[k];
                    ++cnt;
                }
        }
        __syncthreads();
    }
    if (j < dim) {
        const size_t o = ((size_t)chunk * C + c) * dim + j;
        sums[o] = sum;
        counts[o] = cnt;
    }
    if (threadIdx.x == 0 && (cs % slices) == 0) members[chunk * C + c] = mem;
}

// One workgroup per (register size q, centroid c): the new centroid's first 2^q
// coordinates (the mean where points were assigned, else the old coordinate;
// chunks = 0: the centroids as they are), L2-normalised and encoded at size q,
// with the squared norm of the stored register. The workgroup of the largest
// size also writes the new coordinates to `cent`: only coordinates that have
// members, which the other sizes' workgroups do not read from there.
template <typename T>
__global__ void __launch_bounds__(kBlock) kCentroidUpdate(const double *__restrict__ sums,
                                                          const int *__restrict__ counts,
                                                          const int *__restrict__ members, int chunks, int maxQ, int C,
                                                          int qLo, int qHi, const long long *__restrict__ cOff,
                                                          double *cent, T *__restrict__ centAE,
                                                          double *__restrict__ cNorm) {
    extern __shared__ unsigned char smem[];
    __shared__ double norm;
    const int q = qLo + blockIdx.x / C, c = blockIdx.x % C;
    const int D = 1 << q;
    const size_t dim = (size_t)1 << maxQ;
    double *mag = reinterpret_cast<double *>(smem);
    double *cc = cent + (size_t)c * dim;
    // whether the cluster has members: one load a lane, not a chain of them
    const int lane = threadIdx.x & 63;
    const bool mem = __ballot(lane < chunks && members[lane * C + c] > 0) != 0;
    Acc acc[1];
    for (int i = threadIdx.x; i < D; i += kBlock) {
        double sum = 0.0;
        int cnt = 0;
        if (mem) {
            // all chunks' loads in flight, then the sum in order (4096 points, 16
            // centroids up to 10 qubits: the kernel takes 16 us, 22 with four at a time)
            double part[kMeanChunks];
            int num[kMeanChunks];
#pragma unroll
            for (int k = 0; k < kMeanChunks; ++k) {
                const size_t o = ((size_t)k * C + c) * dim + i;
                part[k] = sums[o];
                num[k] = counts[o];
            }
#pragma unroll
            for (int k = 0; k < kMeanChunks; ++k) {
                sum += part[k];
                cnt += num[k];
            }
        }
        double v;
        if (cnt > 0) {
            v = sum / cnt;
            if (q == qHi) cc[i] = v;
        } else {
            v = cc[i];
        }
        mag[i] = v;
        acc[0].add(v * v);
    }
    double tot[1];
    blockReduce<1>(acc, tot);
    if (threadIdx.x == 0) norm = tot[0] > 0 ? 1.0 / sqrt(tot[0]) : 0.0;
    __syncthreads();
    for (int i = threadIdx.x; i < D; i += kBlock) mag[i] *= norm;
    __syncthreads();
    encodeTree<T>(mag, mag + D, mag + 2 * D, q, centAE + cOff[blockIdx.x], cNorm + blockIdx.x);
}

}  // namespace

// ---- the plan ------------------------------------------------------------------

struct SwapPlanImpl {
    int prec;
    int P, C, maxQ, qLo, qHi;
    std::vector<int> hQ;
    int sizeCount[kMaxQ + 1] = {0};    // points of each register size
    std::vector<long long> hPOff, hCOff;
    void *pointsV = nullptr, *pointAE = nullptr, *cent = nullptr, *centAE = nullptr;
    long long *pOff = nullptr, *cOff = nullptr;
    int *pQ = nullptr, *assign = nullptr;
    int *order = nullptr;      // points by register size, largest first
    Tile *tiles = nullptr;     // room for every choice of rowsPerTile
    double *pNorm = nullptr, *cNorm = nullptr, *p0 = nullptr;
    double *meanSums = nullptr;
    int *meanCounts = nullptr, *meanMembers = nullptr;
    int numTiles = 0;
    int rowsPerTile[kMaxQ + 1] = {0};  // register rows one wave sums: 2^q, or a half or quarter of it
    hipGraph_t graph = nullptr;
    hipGraphExec_t graphExec = nullptr;
    size_t aeSmem = 0;
};

namespace {

// results to p0 and assign (the plan's, or scratch where only the time counts)
template <typename T>
void launchOverlap(SwapPlanImpl *s, double *p0, int *assign) {
    hipLaunchKernelGGL(kOverlap<T>, dim3(s->numTiles), dim3(kBlock), 0, hstream(), s->tiles, s->order,
                       (const T *)s->pointAE, s->pOff, s->pNorm, (const T *)s->centAE, s->cOff, s->cNorm, s->C, s->qLo,
                       s->qLo >= 2 ? 1 : 0, p0, assign);
}

// the centroids at every register size: new means from the partial sums
// (chunks = kMeanChunks) or the current centroids (chunks = 0)
template <typename T>
void launchCentroids(SwapPlanImpl *s, int chunks) {
    const int numCent = (s->qHi - s->qLo + 1) * s->C;
    hipLaunchKernelGGL(kCentroidUpdate<T>, dim3(numCent), dim3(kBlock), s->aeSmem, hstream(), s->meanSums,
                       s->meanCounts, s->meanMembers, chunks, s->maxQ, s->C, s->qLo, s->qHi, s->cOff,
                       (double *)s->cent, (T *)s->centAE, s->cNorm);
}

template <typename T>
void launchIteration(SwapPlanImpl *s) {
    launchOverlap<T>(s, s->p0, s->assign);
    const int slices = std::max(1, (1 << s->maxQ) / kBlock);
    hipLaunchKernelGGL(kCentroidPartial, dim3(s->C * slices * kMeanChunks), dim3(kBlock), 0, hstream(),
                       (const double *)s->pointsV, s->pOff, s->pQ, s->assign, s->P, s->C, s->maxQ, s->meanSums,
                       s->meanCounts, s->meanMembers);
    launchCentroids<T>(s, kMeanChunks);
}

// waves that share a register's rows, from the rows one of them takes
int splitOf(const SwapPlanImpl *s, int q) {
    const int split = (1 << q) / s->rowsPerTile[q];
    return split >= 4 ? 4 : split >= 2 ? 2 : 1;
}

// the tile list for the current rows-per-tile choice (per q), largest registers
// first: the last workgroups to start are the short ones
void buildTiles(SwapPlanImpl *s) {
    std::vector<Tile> tl;
    for (int first = 0, q = s->qHi; q >= s->qLo; --q) {
        const int split = splitOf(s, q), per = 16 * (kWaves / split);
        for (int left = s->sizeCount[q]; left > 0; left -= per) {
            const int n = std::min(left, per);
            tl.push_back(Tile{first, n, q, split});
            first += n;
        }
    }
    s->numTiles = (int)tl.size();
    hostToDevice(s->tiles, tl.data(), tl.size() * sizeof(Tile));
}

// outputs of launches that are only timed: the plan keeps its last results
struct TimingScratch {
    double *p0;
    int *assign;
    explicit TimingScratch(const SwapPlanImpl *s)
        : p0(static_cast<double *>(devAlloc((size_t)s->P * s->C * sizeof(double)))),
          assign(static_cast<int *>(devAlloc((size_t)s->P * sizeof(int)))) {}
    TimingScratch(const TimingScratch &) = delete;
    ~TimingScratch() {
        devFree(p0);
        devFree(assign);
    }
};

void dropGraph(SwapPlanImpl *s) {
    if (s->graphExec) QMX_HIP_CHECK(hipGraphExecDestroy(s->graphExec));
    if (s->graph) QMX_HIP_CHECK(hipGraphDestroy(s->graph));
    s->graphExec = nullptr;
    s->graph = nullptr;
}

}  // namespace

}  // namespace qmx

using qmx::SwapPlanImpl;

struct qmxSwapPlan {
    SwapPlanImpl impl;
};

namespace qmx {
namespace {
template <typename T>
__global__ void __launch_bounds__(kBlock) kAEWrite(Amp<T> *__restrict__ a, const double *__restrict__ v, int D) {
    const int x = blockIdx.x * kBlock + threadIdx.x;
    if (x < D) a[x] = Amp<T>{(T)v[x], (T)0};
}

// AmplitudeEncodeOneVector without its global phase gate (AmplitudeEncodeCuda.cu:
// 691-724, angles :20-30 and :61-109, circuit :452-496 with FRyz): the Y tree
// of the real encoder over |v_i|, plus a phase tree over arg v_i (Z = left
// phase - right phase, running phase = their mean). Each level's FRyz applies
// Ry(Y) and then Rz(-Z) uniformly controlled by the higher qubits, so basis
// state x ends with the product of cos / sin(Y/2) along its path and the phase
// sum of +Z/2 (bit clear) / -Z/2 (bit set). One workgroup; LDS holds the
// running magnitudes and phases and the Y and Z lists (4 x 2^q doubles).
__global__ void __launch_bounds__(kBlock) kAEComplex(const double *__restrict__ vre, const double *__restrict__ vim,
                                                     int q, double *__restrict__ ore, double *__restrict__ oim) {
    extern __shared__ unsigned char smem[];
    const int D = 1 << q;
    double *mag = reinterpret_cast<double *>(smem), *ph = mag + D, *Y = ph + D, *Z = Y + D;
    for (int i = threadIdx.x; i < D; i += kBlock) {
        mag[i] = hypot(vre[i], vim[i]);
        ph[i] = atan2(vim[i], vre[i]);
    }
    __syncthreads();
    for (int l = 0; l < q; ++l) {
        const int pairs = D >> (l + 1);
        const int base = D - (D >> l);
        for (int k = threadIdx.x; k < pairs; k += kBlock) {
            const int left = k << (l + 1), right = left + (1 << l);
            const double c = mag[left], s = mag[right];
            Y[base + k] = 2.0 * atan2(s, c);
            if (pairs != 1) {
                const double m2 = c * c + s * s;
                mag[left] = m2 > std::numeric_limits<double>::epsilon() ? sqrt(m2) : 0.0;
            }
            Z[base + k] = ph[left] - ph[right];
            ph[left] = 0.5 * (ph[left] + ph[right]);
        }
        __syncthreads();
    }
    for (int x = threadIdx.x; x < D; x += kBlock) {
        double amp = 1.0, phase = 0.0;
        for (int l = 0; l < q; ++l) {
            const int idx = D - (D >> l) + (x >> (l + 1));
            const bool bit = (x >> l) & 1;
            amp *= bit ? sin(0.5 * Y[idx]) : cos(0.5 * Y[idx]);
            phase += bit ? -0.5 * Z[idx] : 0.5 * Z[idx];
        }
        ore[x] = amp * cos(phase);
        oim[x] = amp * sin(phase);
    }
}

template <typename T>
__global__ void __launch_bounds__(kBlock) kAEWriteComplex(Amp<T> *__restrict__ a, const double *__restrict__ re,
                                                          const double *__restrict__ im, int D) {
    const int x = blockIdx.x * kBlock + threadIdx.x;
    if (x < D) a[x] = Amp<T>{(T)re[x], (T)im[x]};
}
}  // namespace

// qubits 0..q-1 take the encoded complex vector, the others stay |0>
void amplitudeEncodeComplex(QuregDev *q, const double *re, const double *im, int qbits) {
    const int D = 1 << qbits;
    const size_t smem = (size_t)4 * D * sizeof(double);
    if (smem > 65536 && !allowDynamicLds(reinterpret_cast<const void *>(kAEComplex), smem,
                                         "qmxAmplitudeEncodeComplex"))
        return;
    double *buf = static_cast<double *>(devAlloc((size_t)4 * D * sizeof(double)));
    hostToDevice(buf, re, (size_t)D * sizeof(double));
    hostToDevice(buf + D, im, (size_t)D * sizeof(double));
    hipLaunchKernelGGL(kAEComplex, dim3(1), dim3(kBlock), smem, hstream(), buf, buf + D, qbits, buf + 2 * D,
                       buf + 3 * D);
    initBlank(q);
    QMX_DISPATCH(q->prec, T, {
        hipLaunchKernelGGL(kAEWriteComplex<T>, dim3(gridFor(D, 1)), dim3(kBlock), 0, hstream(), (Amp<T> *)q->amps,
                           buf + 2 * D, buf + 3 * D, D);
    });
    checkLaunch("qmxAmplitudeEncodeComplex");
    devFree(buf);
}

// the reference's amplitude-encoding circuit (AmplitudeEncodeCuda.cu:112-150 angles,
// Ry + uniformly controlled Ry ladder, FRGate.cu:181-252) applied to |0...0>:
// qubits 0..q-1 take the encoded vector, the others stay |0>
void amplitudeEncode(QuregDev *q, const double *vec, int qbits) {
    const int D = 1 << qbits;
    const size_t smem = (size_t)3 * D * sizeof(double);
    if (smem > 65536 && !allowDynamicLds(reinterpret_cast<const void *>(kAEState<double>), smem,
                                         "qmxAmplitudeEncodeReal"))
        return;
    struct Hdr {
        long long off;
        int q;
    };
    char *buf = static_cast<char *>(devAlloc((size_t)2 * D * sizeof(double) + 64));
    double *dIn = reinterpret_cast<double *>(buf), *dOut = dIn + D;
    long long *dOff = reinterpret_cast<long long *>(dOut + D);
    int *dQ = reinterpret_cast<int *>(dOff + 1);
    const Hdr h{0, qbits};
    hostToDevice(dIn, vec, (size_t)D * sizeof(double));
    hostToDevice(dOff, &h.off, sizeof(long long));
    hostToDevice(dQ, &h.q, sizeof(int));
    hipLaunchKernelGGL(kAEState<double>, dim3(1), dim3(kBlock), smem, hstream(), dIn, dOff, dQ, dOut,
                       (double *)nullptr, 1);
    initBlank(q);
    QMX_DISPATCH(q->prec, T, {
        hipLaunchKernelGGL(kAEWrite<T>, dim3(gridFor(D, 1)), dim3(kBlock), 0, hstream(), (Amp<T> *)q->amps, dOut, D);
    });
    checkLaunch("qmxAmplitudeEncodeReal");
    devFree(buf);
}
}  // namespace qmx

extern "C" {

qmxSwapPlan *qmxSwapPlanCreate(int numPoints, const int *pointQubits, const double *points, int numCentroids,
                               int maxQubits, const double *centroids, int precision) {
    using namespace qmx;
    runtimeInit();
    if (numPoints < 1 || numCentroids < 1 || maxQubits < kMinQ || maxQubits > kMaxQ || (precision != 0 && precision != 1)) {
        std::fprintf(stderr, "libquest_mi355x: qmxSwapPlanCreate: invalid sizes or precision\n");
        return nullptr;
    }
    auto *plan = new qmxSwapPlan;
    SwapPlanImpl *s = &plan->impl;
    s->prec = precision;
    s->P = numPoints;
    s->C = numCentroids;
    s->maxQ = maxQubits;
    s->qLo = maxQubits;
    s->qHi = 1;
    s->hQ.assign(pointQubits, pointQubits + numPoints);
    for (int q : s->hQ) {
        if (q < kMinQ || q > maxQubits) {
            std::fprintf(stderr, "libquest_mi355x: qmxSwapPlanCreate: point register size %d outside [1, %d]\n", q,
                         maxQubits);
            delete plan;
            return nullptr;
        }
        s->qLo = std::min(s->qLo, q);
        s->qHi = std::max(s->qHi, q);
        ++s->sizeCount[q];
    }
    s->hPOff.resize(numPoints);
    long long tot = 0;
    for (int p = 0; p < numPoints; ++p) {
        s->hPOff[p] = tot;
        tot += 1ll << s->hQ[p];
    }
    const int nq = s->qHi - s->qLo + 1;
    s->hCOff.resize((size_t)nq * numCentroids);
    long long ctot = 0;
    for (int qi = 0; qi < nq; ++qi)
        for (int c = 0; c < numCentroids; ++c) {
            s->hCOff[(size_t)qi * numCentroids + c] = ctot;
            ctot += 1ll << (s->qLo + qi);
        }
    // encoded registers in the storage precision; inputs, centroids and the
    // encoding arithmetic in FP64
    const size_t eb = precision == FP64 ? 8 : 4;
    std::vector<double> pts(points, points + tot);
    for (int p = 0; p < numPoints; ++p) {
        double n2 = 0;
        const long long D = 1ll << s->hQ[p];
        for (long long i = 0; i < D; ++i) n2 += pts[s->hPOff[p] + i] * pts[s->hPOff[p] + i];
        const double f = n2 > 0 ? 1.0 / std::sqrt(n2) : 0.0;
        for (long long i = 0; i < D; ++i) pts[s->hPOff[p] + i] *= f;
    }
    s->pointsV = devAlloc((size_t)tot * 8);
    hostToDevice(s->pointsV, pts.data(), (size_t)tot * 8);
    s->pointAE = devAlloc((size_t)tot * eb);
    const size_t centCount = (size_t)numCentroids * (1ull << maxQubits);
    s->cent = devAlloc(centCount * 8);
    hostToDevice(s->cent, centroids, centCount * 8);
    s->centAE = devAlloc((size_t)ctot * eb);
    s->pOff = static_cast<long long *>(devAlloc(numPoints * sizeof(long long)));
    s->cOff = static_cast<long long *>(devAlloc(s->hCOff.size() * sizeof(long long)));
    s->pQ = static_cast<int *>(devAlloc(numPoints * sizeof(int)));
    s->assign = static_cast<int *>(devAlloc(numPoints * sizeof(int)));
    s->order = static_cast<int *>(devAlloc(numPoints * sizeof(int)));
    s->tiles = static_cast<Tile *>(devAlloc((size_t)(numPoints / 16 + kMaxQ + 1) * sizeof(Tile)));
    s->pNorm = static_cast<double *>(devAlloc(numPoints * sizeof(double)));
    s->cNorm = static_cast<double *>(devAlloc((size_t)nq * numCentroids * sizeof(double)));
    s->p0 = static_cast<double *>(devAlloc((size_t)numPoints * numCentroids * sizeof(double)));
    const size_t meanSlots = (size_t)kMeanChunks * numCentroids * (1ull << maxQubits);
    s->meanSums = static_cast<double *>(devAlloc(meanSlots * sizeof(double)));
    s->meanCounts = static_cast<int *>(devAlloc(meanSlots * sizeof(int)));
    s->meanMembers = static_cast<int *>(devAlloc((size_t)kMeanChunks * numCentroids * sizeof(int)));
    hostToDevice(s->pOff, s->hPOff.data(), numPoints * sizeof(long long));
    hostToDevice(s->cOff, s->hCOff.data(), s->hCOff.size() * sizeof(long long));
    hostToDevice(s->pQ, s->hQ.data(), numPoints * sizeof(int));
    std::vector<int> order(numPoints);
    for (int p = 0; p < numPoints; ++p) order[p] = p;
    std::stable_sort(order.begin(), order.end(), [&](int x, int y) { return s->hQ[x] > s->hQ[y]; });
    hostToDevice(s->order, order.data(), numPoints * sizeof(int));
    s->aeSmem = (size_t)3 * (1u << s->qHi) * sizeof(double);
    // 11- and 12-qubit registers need more than the 64 KiB default of dynamic LDS
    bool ldsOk = true;
    QMX_DISPATCH(precision, T, {
        if (s->aeSmem > 65536)
            ldsOk = allowDynamicLds(reinterpret_cast<const void *>(kAEState<T>), s->aeSmem, "qmxSwapPlanCreate") &&
                    allowDynamicLds(reinterpret_cast<const void *>(kCentroidUpdate<T>), s->aeSmem, "qmxSwapPlanCreate");
    });
    if (!ldsOk) {
        qmxSwapPlanDestroy(plan);
        return nullptr;
    }
    // default rows per wave: a register's rows split over four waves from 256
    // rows, over two from 64 (see kOverlap); smaller ones are one wave's
    for (int q = 0; q <= kMaxQ; ++q) s->rowsPerTile[q] = (1 << q) / (q >= 8 ? 4 : q >= 6 ? 2 : 1);
    QMX_DISPATCH(precision, T, {
        hipLaunchKernelGGL(kAEState<T>, dim3(numPoints), dim3(kBlock), s->aeSmem, hstream(),
                           (const double *)s->pointsV, s->pOff, s->pQ, (T *)s->pointAE,
                           s->pNorm, numPoints);
        launchCentroids<T>(s, 0);
    });
    checkLaunch("qmxSwapPlanCreate");
    buildTiles(s);
    deviceSync();
    return plan;
}

void qmxSwapPlanDestroy(qmxSwapPlan *plan) {
    using namespace qmx;
    if (!plan) return;
    SwapPlanImpl *s = &plan->impl;
    dropGraph(s);
    for (void *p : {s->pointsV, s->pointAE, s->cent, s->centAE, (void *)s->pOff, (void *)s->cOff, (void *)s->pQ,
                    (void *)s->assign, (void *)s->order, (void *)s->tiles, (void *)s->pNorm, (void *)s->cNorm,
                    (void *)s->p0, (void *)s->meanSums, (void *)s->meanCounts, (void *)s->meanMembers})
        devFree(p);
    delete plan;
}

// time candidate rows-per-tile for each register size on the device (the rows
// whole, halved or quartered over a workgroup's waves) and keep the fastest;
// returns the number of (size, candidate) timings made
int qmxSwapPlanAutotune(qmxSwapPlan *plan) {
    using namespace qmx;
    SwapPlanImpl *s = &plan->impl;
    dropGraph(s);
    TimingScratch scratch(s);
    int timings = 0;
    for (int q = s->qLo; q <= s->qHi; ++q) {
        if (!s->sizeCount[q]) continue;
        double best = 1e30;
        int bestRows = s->rowsPerTile[q];
        for (int split = 1; split <= kWaves; split *= 2) {
            if (split > 1 && (1 << q) / split < 16) break;  // a product step takes 16 rows
            s->rowsPerTile[q] = (1 << q) / split;
            buildTiles(s);
            timerBegin();
            QMX_DISPATCH(s->prec, T, { launchOverlap<T>(s, scratch.p0, scratch.assign); });
            checkLaunch("autotune");
            const double ms = timerEndMs();
            ++timings;
            if (ms < best) {
                best = ms;
                bestRows = s->rowsPerTile[q];
            }
        }
        s->rowsPerTile[q] = bestRows;
    }
    buildTiles(s);
    deviceSync();
    return timings;
}

int qmxSwapPlanRowsPerTile(const qmxSwapPlan *plan, int q) {
    return (q >= 0 && q <= qmx::kMaxQ) ? plan->impl.rowsPerTile[q] : 0;
}

int qmxSwapPlanNumTiles(const qmxSwapPlan *plan) { return plan->impl.numTiles; }

// 16 x 16 x 4 matrix-core products one iteration makes
long long qmxSwapPlanMfmaBlocks(const qmxSwapPlan *plan) {
    using namespace qmx;
    const SwapPlanImpl *s = &plan->impl;
    long long products = 0;
    for (int q = s->qLo; q <= s->qHi; ++q)
        products += (long long)((s->sizeCount[q] + 15) / 16) * (std::max(16, 1 << q) / 4);
    return products * ((s->C + 15) / 16);
}

// device time of one swap-test launch (inner products, P0, assignment; ms, HIP events on the
// library stream), averaged over `launches`
double qmxSwapPlanTimeTiles(qmxSwapPlan *plan, int launches) {
    using namespace qmx;
    SwapPlanImpl *s = &plan->impl;
    if (launches < 1) return 0.0;
    TimingScratch scratch(s);
    deviceSync();
    timerBegin();
    for (int i = 0; i < launches; ++i)
        QMX_DISPATCH(s->prec, T, { launchOverlap<T>(s, scratch.p0, scratch.assign); });
    checkLaunch("qmxSwapPlanTimeTiles");
    return timerEndMs() / launches;
}

// run `iterations` k-means iterations; useGraph != 0 replays one captured
// iteration graph (captured on first use)
void qmxSwapPlanRun(qmxSwapPlan *plan, int iterations, int useGraph) {
    using namespace qmx;
    SwapPlanImpl *s = &plan->impl;
    if (useGraph) {
        if (!s->graphExec) {
            QMX_HIP_CHECK(hipStreamBeginCapture(hstream(), hipStreamCaptureModeThreadLocal));
            QMX_DISPATCH(s->prec, T, { launchIteration<T>(s); });
            QMX_HIP_CHECK(hipStreamEndCapture(hstream(), &s->graph));
            QMX_HIP_CHECK(hipGraphInstantiate(&s->graphExec, s->graph, nullptr, nullptr, 0));
        }
        for (int i = 0; i < iterations; ++i) QMX_HIP_CHECK(hipGraphLaunch(s->graphExec, hstream()));
    } else {
        for (int i = 0; i < iterations; ++i) {
            QMX_DISPATCH(s->prec, T, { launchIteration<T>(s); });
            checkLaunch("qmxSwapPlanRun");
        }
    }
}

// P(ancilla = 0) of every test of the last iteration, [point][centroid]
void qmxSwapPlanP0(qmxSwapPlan *plan, double *out) {
    qmx::deviceToHost(out, plan->impl.p0, (size_t)plan->impl.P * plan->impl.C * sizeof(double));
}

void qmxSwapPlanAssignments(qmxSwapPlan *plan, int *out) {
    qmx::deviceToHost(out, plan->impl.assign, (size_t)plan->impl.P * sizeof(int));
}

// current centroids (numCentroids x 2^maxQubits), as doubles
void qmxSwapPlanCentroids(qmxSwapPlan *plan, double *out) {
    using namespace qmx;
    SwapPlanImpl *s = &plan->impl;
    deviceToHost(out, s->cent, (size_t)s->C * (1ull << s->maxQ) * sizeof(double));
}

// replace the centroids (numCentroids x 2^maxQubits doubles) and re-encode
// them; the point registers, tiles, tuned shapes and a captured graph stay
void qmxSwapPlanSetCentroids(qmxSwapPlan *plan, const double *centroids) {
    using namespace qmx;
    SwapPlanImpl *s = &plan->impl;
    deviceSync();
    hostToDevice(s->cent, centroids, (size_t)s->C * (1ull << s->maxQ) * sizeof(double));
    QMX_DISPATCH(s->prec, T, { launchCentroids<T>(s, 0); });
    checkLaunch("qmxSwapPlanSetCentroids");
    deviceSync();
}

// encoded state of point p (its 2^q amplitudes), for checking the encoder
void qmxSwapPlanPointState(qmxSwapPlan *plan, int p, double *out) {
    using namespace qmx;
    SwapPlanImpl *s = &plan->impl;
    const size_t D = 1ull << s->hQ[p];
    if (s->prec == FP64) {
        deviceToHost(out, (double *)s->pointAE + s->hPOff[p], D * 8);
    } else {
        std::vector<float> f(D);
        deviceToHost(f.data(), (float *)s->pointAE + s->hPOff[p], D * 4);
        for (size_t i = 0; i < D; ++i) out[i] = f[i];
    }
}

}  // extern "C"
