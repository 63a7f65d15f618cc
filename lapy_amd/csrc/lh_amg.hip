// Smoothed-aggregation multigrid for the linear solves' operator K
// (symmetric, sparse, Laplacian-like: stiffness, Dirichlet-masked stiffness,
// mass + t stiffness).
//
// Setup (once per solve, all on the device, deterministic), level by level:
//  * lambda_max of D^-1 K from ten power steps, bmax = 1.1 times it and 2 at
//    most, and D raised in the rows whose Gershgorin sum exceeds 1.16 bmax, so
//    that no eigenvalue does;
//  * aggregates around the roots of a maximal independent set of distance 2
//    in the graph of strong connections (k_ij^2 > theta^2 k_ii k_jj), found
//    with hashed keys in a fixed number of rounds; the roots are numbered in
//    row order, so the coarse rows keep the fine rows' locality;
//  * P = (I - w D^-1 K) P_0, P_0 the aggregates' indicator, w = 4 / (3
//    bmax): the smoothing that makes the interpolated coarse functions
//    continuous, without which the cycle's quality decays with every level;
//  * K_c = P^T (K P): two sparse products, one wave per output row, the
//    row's entries gathered in a hash table in LDS whose values are summed
//    in the order of the first factor's entries (so the result does not
//    depend on scheduling).
//
// Cycle: V(1,1) with the Chebyshev polynomial of degree 2 on [bmax / 6, bmax]
// as the smoother before and after.  Its error polynomial is at most 1 in
// magnitude on [0, 7/6 bmax], which holds the spectrum, hence a symmetric
// positive definite preconditioner, as conjugate gradients need.  (Power steps
// alone miss the mode of one bad element among good ones: a vertex of an
// icosphere of 40,962 moved to 0.08 of its height has lambda_max 2.01, the
// steps find 1.50, and the cycle was indefinite.  Raising D where the
// row asks for it leaves the other rows' smoothing as it is, and takes bad
// elements' modes out of bmax: CG on 4,913 tet vertices jittered by a quarter
// of the spacing took 35 iterations with bmax 4.1, 28 now.)  A level is six launches; all
// levels of at most kTailRows rows run in one workgroup per column with
// their vectors in LDS (one launch instead of six a level, which at these
// sizes are nothing but launch latency), and the last level (at most 128
// rows) multiplies with its inverse.
//
// The coarsest matrix of a pure Neumann operator is singular (constants), and
// that of A - sigma B nearly so where sigma is small against the eigenvalues
// (a mesh in small units): its unit diagonal is raised by 1e-9 in FP64, which
// leaves the other components unchanged to that accuracy and bounds the
// constant one, which the right-hand sides of such systems have only to
// rounding.  The eigensolver's blocks are raised by 1e-5 (the other components'
// eigenvalues are (pi / 128)^2 / 2 = 3e-4 and more, a chain's; about 0.04 on a
// sphere): its first residuals hold the constant components in full, and
// columns that are the same to 1e-6 after the cycle fail in the Cholesky-QR,
// whose pivots are squares (with 1e-6 at radius 1e-8, with 1e-9 at 0.01).  The
// inverse and its sums stay in FP64 there too.
#include "lh_amg.hpp"

#include <cmath>

namespace lh {

namespace {

constexpr double kTheta = 0.05;      // strength threshold of the finest level, halved on each coarser one
constexpr int kPowerSteps = 10;
constexpr int kMisRounds = 8;
constexpr int kMaxLevels = 12;
constexpr int kCoarsest = 128;       // rows of the inverted level at most (kCholMax)
constexpr int kTailRows = 2048;      // rows of a one-workgroup level at most
constexpr int kTailNnz = 24576;      // and its entries: one CU reads them from L2 for every product
constexpr int kTailSum = 2560;       // rows of all of them together at most
constexpr int kLongRow = 20;         // mean row length from which a wave forms a row of P,
constexpr int kLongestRow = 128;     // and the longest from which it does whatever the mean
constexpr double kSmoothRatio = 6.0; // the smoother's interval is [bmax / ratio, bmax]
constexpr double kSmoothTop = 2.0;   // bmax at most (good elements: 1.5 to 1.9 on the finest level, 1.3 to 1.5 below)
constexpr double kGuard = 1.16;      // rows' Gershgorin sums are held to this many bmax (7/6: the smoother's limit)

static_assert(kCoarsest <= kCholMax, "the coarsest level is factorised by cholinv");

// coefficients of the degree-2 Chebyshev smoother on [bmax / ratio, bmax]:
// y = x + s D^-1 (b - K x), x' = y + c1 (y - x) + c2 D^-1 (b - K y)
struct Cheb2 {
    double s, c1, c2;
};
__host__ __device__ inline Cheb2 cheb2(double bmax) {
    const double amin = bmax / kSmoothRatio;
    const double th = 0.5 * (bmax + amin), de = 0.5 * (bmax - amin), sig = th / de;
    const double rho0 = 1.0 / sig, rho1 = 1.0 / (2.0 * sig - rho0);
    return Cheb2{1.0 / th, rho1 * rho0, 2.0 * rho1 / de};
}

template <int V>
struct IntC {
    static constexpr int v = V;
};
// lanes for a row of the mean length: about four entries a lane
int lanes_for(int64_t nnz, int64_t n) {
    const int64_t avg = n > 0 ? nnz / n : 0;
    return avg >= 40 ? 16 : avg >= 20 ? 8 : avg >= 8 ? 4 : 1;
}
template <typename F>
void with_lanes(int g, F&& f) {
    switch (g) {
        case 1: f(IntC<1>{}); break;
        case 4: f(IntC<4>{}); break;
        case 8: f(IntC<8>{}); break;
        default: f(IntC<16>{}); break;
    }
}

// C. Wellons' "lowbias32" (hash prospector, 2018), a 32-bit integer mixer
__device__ __forceinline__ uint32_t mix32(uint32_t x) {
    x ^= x >> 16;
    x *= 0x7feb352du;
    x ^= x >> 15;
    x *= 0x846ca68bu;
    x ^= x >> 16;
    return x;
}

// ---- setup ------------------------------------------------------------------
// The kernels over the rows of a level's matrix take G lanes a row (about the
// row's entries): with a thread a row a wave's loads are scattered over 64 rows
// and the longest row sets its time.  118k tet vertices (15 entries a row; 50 on
// the next level): power step 26 -> 5.4 us, averaged over the levels, and the
// spreading step 35 -> 4.4, which also stopped testing every entry's strength
// again in each round.

// dinv and the row sums of |D^-1 K|; bad[0] set when a row's diagonal is negative, missing or zero beside
// non-zero entries; start vector of the power iteration (0 on zero rows);
// longest: raised to the length of the rows above kLongestRow, if any
template <int G>
__global__ void __launch_bounds__(256)
k_amg_diag(int64_t n, const int32_t* __restrict__ rp, const int32_t* __restrict__ cl, const double* __restrict__ kv,
           double* __restrict__ dinv, double* __restrict__ gersh, double* __restrict__ x, int* __restrict__ bad,
           int* __restrict__ longest) {
    const int64_t i = (xcd_block() * 256 + threadIdx.x) / G;
    if (i >= n) return;
    double d = 0.0, other = 0.0;  // other: sum of the magnitudes beside the diagonal
    for (int32_t s = rp[i] + (int32_t)(threadIdx.x % G); s < rp[i + 1]; s += G) {
        if (cl[s] == (int32_t)i) d = kv[s];
        else other += fabs(kv[s]);
    }
#pragma unroll
    for (int o = G / 2; o > 0; o >>= 1) {
        d += __shfl_xor(d, o, 64);  // zero in all lanes but one
        other += __shfl_xor(other, o, 64);
    }
    if (threadIdx.x % G) return;
    if (!(d >= 0.0) || (d == 0.0 && other != 0.0)) bad[0] = 1;  // every writer stores the same value
    const bool pos = d > 0.0;
    if (rp[i + 1] - rp[i] > kLongestRow) atomicMax(longest, rp[i + 1] - rp[i]);
    dinv[i] = pos ? 1.0 / d : 0.0;
    gersh[i] = pos ? 1.0 + other / d : 0.0;
    x[i] = pos ? (double)(mix32((uint32_t)i * 2654435761u + 12345u) >> 8) * (1.0 / 8388608.0) - 1.0 : 0.0;
}
// D raised where the row's sum exceeds the limit: by Gershgorin's theorem no
// eigenvalue of the new D^-1 K does
__global__ void k_amg_guard(int64_t n, const double* __restrict__ gersh, double limit, double* __restrict__ dinv) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n && gersh[i] > limit) dinv[i] *= limit / gersh[i];
}
// y = D^-1 K x
template <int G>
__global__ void __launch_bounds__(256)
k_amg_power(int64_t n, const int32_t* __restrict__ rp, const int32_t* __restrict__ cl, const double* __restrict__ kv,
            const double* __restrict__ dinv, const double* __restrict__ x, double* __restrict__ y) {
    const int64_t i = (xcd_block() * 256 + threadIdx.x) / G;
    if (i >= n) return;
    double a = 0.0;
    for (int32_t s = rp[i] + (int32_t)(threadIdx.x % G); s < rp[i + 1]; s += G) a += kv[s] * x[cl[s]];
#pragma unroll
    for (int o = G / 2; o > 0; o >>= 1) a += __shfl_xor(a, o, 64);
    if (threadIdx.x % G == 0) y[i] = dinv[i] * a;
}
// block partials of x^T D x and x^T D y (y = D^-1 K x): 2 doubles a block
__global__ void __launch_bounds__(256)
k_amg_rayleigh(int64_t n, const double* __restrict__ dinv, const double* __restrict__ x, const double* __restrict__ y,
               double* __restrict__ part) {
    __shared__ double sh[2][4];
    double a = 0.0, b = 0.0;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
        if (dinv[i] > 0.0) {
            const double d = 1.0 / dinv[i];
            a += x[i] * d * x[i];
            b += x[i] * d * y[i];
        }
    }
    a = wave_sum64(a);
    b = wave_sum64(b);
    if ((threadIdx.x & 63) == 0) {
        sh[0][threadIdx.x >> 6] = a;
        sh[1][threadIdx.x >> 6] = b;
    }
    __syncthreads();
    if (threadIdx.x < 2) part[2 * blockIdx.x + threadIdx.x] = (sh[threadIdx.x][0] + sh[threadIdx.x][1]) + (sh[threadIdx.x][2] + sh[threadIdx.x][3]);
}

// independent set: key = state (0 out, 1 undecided, 2 in) << 62 | hash | row
constexpr unsigned long long kOut = 0ull, kUndecided = 1ull << 62, kIn = 2ull << 62;

__global__ void k_mis_init(int64_t n, const double* __restrict__ dinv, unsigned long long* __restrict__ t) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    // zero rows (Dirichlet) take no part
    t[i] = dinv[i] > 0.0
               ? kUndecided | ((unsigned long long)(mix32((uint32_t)i + 0x9e3779b9u) >> 2) << 32) | (unsigned)i
               : kOut;
}
// the strong neighbours of each row, k_ij^2 > theta^2 k_ii k_jj: the column, or
// -1 for a weak entry
template <int G>
__global__ void __launch_bounds__(256)
k_strong(int64_t n, const int32_t* __restrict__ rp, const int32_t* __restrict__ cl, const double* __restrict__ kv,
         const double* __restrict__ dinv, double th2, int32_t* __restrict__ sc) {
    const int64_t i = (xcd_block() * 256 + threadIdx.x) / G;
    if (i >= n) return;
    const double di = dinv[i];
    for (int32_t s = rp[i] + (int32_t)(threadIdx.x % G); s < rp[i + 1]; s += G) {
        const int32_t j = cl[s];
        sc[s] = kv[s] * kv[s] * di * dinv[j] > th2 ? j : -1;
    }
}

// largest key among the row and its strong neighbours, in every lane of the row
template <int G>
__device__ __forceinline__ unsigned long long mis_max(int64_t i, const int32_t* __restrict__ rp,
                                                      const int32_t* __restrict__ sc,
                                                      const unsigned long long* __restrict__ t) {
    unsigned long long best = t[i];
    for (int32_t s = rp[i] + (int32_t)(threadIdx.x % G); s < rp[i + 1]; s += G) {
        const int32_t j = sc[s];
        const unsigned long long q = j >= 0 ? t[j] : 0ull;
        best = q > best ? q : best;
    }
#pragma unroll
    for (int o = G / 2; o > 0; o >>= 1) {
        const unsigned long long q = __shfl_xor(best, o, 64);
        best = q > best ? q : best;
    }
    return best;
}
template <int G>
__global__ void __launch_bounds__(256)
k_mis_spread(int64_t n, const int32_t* __restrict__ rp, const int32_t* __restrict__ sc,
             const unsigned long long* __restrict__ t, unsigned long long* __restrict__ a) {
    const int64_t i = (xcd_block() * 256 + threadIdx.x) / G;
    if (i >= n) return;
    const unsigned long long best = mis_max<G>(i, rp, sc, t);
    if (threadIdx.x % G == 0) a[i] = best;
}
// second spreading step and the decision: a row whose key is the largest
// within distance 2 joins, one with a member within distance 2 leaves
template <int G>
__global__ void __launch_bounds__(256)
k_mis_decide(int64_t n, const int32_t* __restrict__ rp, const int32_t* __restrict__ sc,
             const unsigned long long* __restrict__ a, unsigned long long* __restrict__ t) {
    const int64_t i = (xcd_block() * 256 + threadIdx.x) / G;
    if (i >= n) return;
    const unsigned long long own = t[i];
    if ((own >> 62) != 1) return;  // all lanes of the row
    const unsigned long long best = mis_max<G>(i, rp, sc, a);
    if (threadIdx.x % G) return;
    if (best == own) t[i] = kIn | (own & ~(3ull << 62));
    else if ((best >> 62) == 2) t[i] = kOut;
}
__global__ void k_mis_flag(int64_t n, const unsigned long long* __restrict__ t, int32_t* __restrict__ flag) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) flag[i] = (t[i] >> 62) == 2 ? 1 : 0;
}
__global__ void k_agg_roots(int64_t n, const int32_t* __restrict__ flag, const int32_t* __restrict__ id,
                            int32_t* __restrict__ agg) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) agg[i] = flag[i] ? id[i] : -1;
}
// an unassigned row joins the aggregate of its strongest assigned neighbour
// (the first of equals); in: the assignment before this pass
template <int G>
__global__ void __launch_bounds__(256)
k_agg_join(int64_t n, const int32_t* __restrict__ rp, const int32_t* __restrict__ sc, const double* __restrict__ kv,
           const int32_t* __restrict__ in, int32_t* __restrict__ out) {
    const int64_t i = (xcd_block() * 256 + threadIdx.x) / G;
    if (i >= n) return;
    int32_t g = in[i];
    if (g < 0) {  // all lanes of the row
        double best = 0.0;
        int32_t at = INT32_MAX;
        for (int32_t s = rp[i] + (int32_t)(threadIdx.x % G); s < rp[i + 1]; s += G) {
            const int32_t j = sc[s];
            const double w = fabs(kv[s]);
            if (j >= 0 && w > best && in[j] >= 0) {
                best = w;
                at = s;
            }
        }
#pragma unroll
        for (int o = G / 2; o > 0; o >>= 1) {
            const double w = __shfl_xor(best, o, 64);
            const int32_t q = __shfl_xor(at, o, 64);
            if (w > best || (w == best && q < at)) {
                best = w;
                at = q;
            }
        }
        if (at != INT32_MAX) g = in[sc[at]];
    }
    if (threadIdx.x % G == 0) out[i] = g;
}

// P = (I - w D^-1 K) P_0 row by row: first the number of distinct aggregates
// among a row's columns, then the entries in the order of first appearance.
// One thread per row for short rows; for long ones (below) the quadratic
// search is spread over a wave, also where a single row is long: the pole of a
// sphere of meridians has an entry and a third of an aggregate for each, and
// at 1,000 of them one thread's search took about 100 ms, twice.
template <bool FILL>
__global__ void k_prolongator(int64_t n, const int32_t* __restrict__ rp, const int32_t* __restrict__ cl,
                              const double* __restrict__ kv, const double* __restrict__ dinv, double w,
                              const int32_t* __restrict__ agg, const int32_t* __restrict__ pp,
                              int32_t* __restrict__ count_or_cols, double* __restrict__ pv) {
    const int64_t i = xcd_block() * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int32_t r0 = rp[i], r1 = rp[i + 1];
    const double wd = w * dinv[i];
    const int32_t own = agg[i];
    int32_t at = FILL ? pp[i] : 0;
    if (wd > 0.0) {
        for (int32_t s = r0; s < r1; ++s) {
            const int32_t g = agg[cl[s]];
            if (g < 0) continue;
            bool seen = false;
            for (int32_t q = r0; q < s && !seen; ++q) seen = agg[cl[q]] == g;
            if (seen) continue;
            if (FILL) {
                double v = 0.0;
                for (int32_t q = s; q < r1; ++q)
                    if (agg[cl[q]] == g) v += kv[q];
                count_or_cols[at] = g;
                pv[at] = (g == own ? 1.0 : 0.0) - wd * v;
            }
            ++at;
        }
    }
    if (!FILL) count_or_cols[i] = at;
}
// one wave per row: each lane holds one entry of a chunk of 64 and meets all
// entries of the row in order (lane reads), summing those of its aggregate;
// the first lane of an aggregate writes.  Sums and order as above.
template <bool FILL>
__global__ void __launch_bounds__(256)
k_prolongator_wave(int64_t n, const int32_t* __restrict__ rp, const int32_t* __restrict__ cl,
                   const double* __restrict__ kv, const double* __restrict__ dinv, double w,
                   const int32_t* __restrict__ agg, const int32_t* __restrict__ pp, int32_t* __restrict__ count_or_cols,
                   double* __restrict__ pv) {
    const int64_t i = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (i >= n) return;  // whole wave
    const int lane = threadIdx.x & 63;
    const int32_t r0 = rp[i], r1 = rp[i + 1];
    const double wd = w * dinv[i];
    const int32_t own = agg[i];
    int32_t at = FILL ? pp[i] : 0;
    if (wd > 0.0) {
        for (int32_t a = r0; a < r1; a += 64) {
            const int32_t g = (a + lane < r1) ? agg[cl[a + lane]] : -1;
            bool seen = g < 0;
            double v = 0.0;
            for (int32_t b = r0; b < r1; b += 64) {
                const bool in = b + lane < r1;
                const int32_t gq = in ? agg[cl[b + lane]] : -1;
                const double kq = in ? kv[b + lane] : 0.0;
                const int cnt = r1 - b < 64 ? r1 - b : 64;
                for (int o = 0; o < cnt; ++o) {
                    const int32_t go = __builtin_amdgcn_readlane(gq, o);
                    const double ko = __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(kq), o),
                                                       __builtin_amdgcn_readlane(__double2loint(kq), o));
                    if (go == g) {
                        v += ko;
                        seen = seen || b + o < a + lane;
                    }
                }
            }
            const unsigned long long first = __ballot(!seen);
            if (FILL && !seen) {
                const int32_t q = at + __popcll(first & ((1ull << lane) - 1));
                count_or_cols[q] = g;
                pv[q] = (g == own ? 1.0 : 0.0) - wd * v;
            }
            at += __popcll(first);
        }
    }
    if (!FILL && lane == 0) count_or_cols[i] = at;
}

// transpose of P: entries per coarse row, then each entry to a free place of
// its row (in any order), then each row sorted by the fine row
__global__ void k_count_cols(int64_t nnz, const int32_t* __restrict__ pc, int32_t* __restrict__ cnt) {
    const int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (s < nnz) atomicAdd(cnt + pc[s], 1);
}
__global__ void k_scatter_cols(int64_t n, const int32_t* __restrict__ pp, const int32_t* __restrict__ pc,
                               const double* __restrict__ pv, const int32_t* __restrict__ tp, int32_t* __restrict__ fill,
                               int32_t* __restrict__ tc, double* __restrict__ tv) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    for (int32_t s = pp[i]; s < pp[i + 1]; ++s) {
        const int32_t g = pc[s];
        const int32_t q = tp[g] + atomicAdd(fill + g, 1);
        tc[q] = (int32_t)i;
        tv[q] = pv[s];
    }
}
__device__ __forceinline__ void wave_fence() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}
// one wave per row: an entry's place is the number of smaller ones (a row's
// entries are distinct), counted over the row's keys in LDS, four a read; a
// row of more than 1,024 counts in memory.  118k
// tet vertices: 109 -> 30 us a level (one key a read from memory before).
__global__ void __launch_bounds__(256)
k_sort_rows(int64_t nc, const int32_t* __restrict__ tp, const int32_t* __restrict__ ti, const double* __restrict__ vi,
            int32_t* __restrict__ to, double* __restrict__ vo) {
    constexpr int kKeys = 1024;
    __shared__ __align__(16) int32_t s_keys[4][kKeys];
    const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int64_t r = (int64_t)blockIdx.x * 4 + wv;
    if (r >= nc) return;  // no workgroup barrier follows
    const int32_t a = tp[r], len = tp[r + 1] - a;
    const bool in_lds = len <= kKeys;
    int32_t* keys = s_keys[wv];
    if (in_lds) {
        for (int q = lane; q < (len + 3) / 4 * 4; q += 64) keys[q] = q < len ? ti[a + q] : INT32_MAX;
        wave_fence();
    }
    for (int e = lane; e < len; e += 64) {
        const int32_t key = ti[a + e];
        int32_t rank = 0;
        if (in_lds) {
            for (int q = 0; q < len; q += 4) {
                const int4 k = *reinterpret_cast<const int4*>(keys + q);
                rank += (k.x < key) + (k.y < key) + (k.z < key) + (k.w < key);
            }
        } else {
            for (int q = 0; q < len; ++q) rank += ti[a + q] < key;
        }
        to[a + rank] = key;
        vo[a + rank] = vi[a + e];
    }
}

// ---- C = X Y, one wave per row of X --------------------------------------------
// The row's distinct columns live in a hash table of HS slots in LDS (linear
// probing).  Counting: lanes insert the rows of Y in any order.  Filling:
// the rows of Y are added one after another, the lanes of a step holding
// distinct columns, so a value's terms are summed in the order of X's
// entries; an entry's place in the output row is the number of smaller
// columns.  A row with more than 3/4 HS distinct columns sets over[0].
// Bound by the latency of its dependent LDS steps (one per entry of X's row):
// the rows of Y are on their way before their turn.  118k tet vertices, all six
// products:
// 1.40 -> 0.98 ms.
template <int HS>
__device__ __forceinline__ int hash_slot(volatile int32_t* keys, int32_t key) {
    int h = (int)(mix32((uint32_t)key) & (HS - 1));
    for (int tries = 0; tries < HS; ++tries) {
        const int32_t q = keys[h];
        if (q == key) return h;
        if (q < 0) {
            const int32_t was = atomicCAS(const_cast<int32_t*>(keys) + h, -1, key);
            if (was < 0 || was == key) return h;
        }
        h = (h + 1) & (HS - 1);
    }
    return -1;
}

template <int HS, bool FILL>
__global__ void __launch_bounds__(256)
k_spgemm(int64_t n, const int32_t* __restrict__ xp, const int32_t* __restrict__ xc, const double* __restrict__ xv,
         const int32_t* __restrict__ yp, const int32_t* __restrict__ yc, const double* __restrict__ yv,
         const int32_t* __restrict__ cp, int32_t* __restrict__ count_or_cols, double* __restrict__ cv,
         int* __restrict__ over) {
    __shared__ int32_t s_keys[4][HS];
    __shared__ double s_vals[FILL ? 4 : 1][FILL ? HS : 1];
    __shared__ int32_t s_list[FILL ? 4 : 1][FILL ? HS : 1], s_slot[FILL ? 4 : 1][FILL ? HS : 1];
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int64_t row = (int64_t)blockIdx.x * 4 + wv;
    if (row >= n) return;  // no workgroup barrier follows
    volatile int32_t* keys = s_keys[wv];
    volatile double* vals = s_vals[FILL ? wv : 0];
    for (int h = lane; h < HS; h += 64) {
        keys[h] = -1;
        if (FILL) vals[h] = 0.0;
    }
    wave_fence();
    const int32_t a = xp[row], b = xp[row + 1];
    if (!FILL) {
        int mine = 0;
        // lanes over X's entries; more than HS distinct columns: hash_slot gives
        // up after a search of the whole table, and the lane with it
        for (int32_t e = a + lane; e < b && !mine; e += 64) {
            const int32_t j = xc[e];
            for (int32_t q = yp[j]; q < yp[j + 1] && !mine; ++q) mine = hash_slot<HS>(keys, yc[q]) < 0;
        }
        wave_fence();
        int cnt = 0;
        for (int h = lane; h < HS; h += 64) cnt += keys[h] >= 0;
        for (int o = 32; o > 0; o >>= 1) cnt += __shfl_xor(cnt, o, 64);
        if (__any(mine) || cnt > HS * 3 / 4) {
            if (lane == 0) over[0] = 1;
        }
        if (lane == 0) count_or_cols[row] = cnt;
        return;
    }
    // 64 entries of X's row and their rows' bounds side by side, then the rows of
    // Y four at a time: the next four are loaded while these are added
    for (int32_t e0 = a; e0 < b; e0 += 64) {
        const bool in = e0 + lane < b;
        const int32_t j = in ? xc[e0 + lane] : 0;
        const double xl = in ? xv[e0 + lane] : 0.0;
        const int32_t y0 = in ? yp[j] : 0, y1 = in ? yp[j + 1] : 0;
        const int cnt = b - e0 < 64 ? b - e0 : 64;
        int32_t c[4], cn[4];
        double v[4], vn[4];
        auto load4 = [&](int o0, int32_t (&cc)[4], double (&vv)[4]) {
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int o = o0 + u < 64 ? o0 + u : 63;
                const int32_t q = __builtin_amdgcn_readlane(y0, o) + lane;
                const bool ok = o0 + u < cnt && q < __builtin_amdgcn_readlane(y1, o);
                cc[u] = ok ? yc[q] : -1;
                vv[u] = ok ? yv[q] : 0.0;
            }
        };
        load4(0, c, v);
        for (int o0 = 0; o0 < cnt; o0 += 4) {
            load4(o0 + 4, cn, vn);
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int o = o0 + u < 64 ? o0 + u : 63;
                const double x = __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(xl), o),
                                                  __builtin_amdgcn_readlane(__double2loint(xl), o));
                if (c[u] >= 0) {
                    const int h = hash_slot<HS>(keys, c[u]);
                    if (h >= 0) vals[h] = vals[h] + x * v[u];
                }
                const int32_t r1 = o0 + u < cnt ? __builtin_amdgcn_readlane(y1, o) : 0;
                for (int32_t q = __builtin_amdgcn_readlane(y0, o) + 64 + lane; q < r1; q += 64) {
                    const int h = hash_slot<HS>(keys, yc[q]);
                    if (h >= 0) vals[h] = vals[h] + x * yv[q];
                }
                wave_fence();
            }
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                c[u] = cn[u];
                v[u] = vn[u];
            }
        }
    }
    // the table's columns packed into a list, then ranked against it
    const int32_t base = cp[row], cnt = cp[row + 1] - base;
    volatile int32_t* list = s_list[FILL ? wv : 0];
    volatile int32_t* slot = s_slot[FILL ? wv : 0];
    int c = 0;
    for (int h0 = 0; h0 < HS; h0 += 64) {
        const int32_t key = keys[h0 + lane];
        const unsigned long long bal = __ballot(key >= 0);
        const int at = c + __popcll(bal & ((1ull << lane) - 1));
        if (key >= 0) {
            list[at] = key;
            slot[at] = h0 + lane;
        }
        c += __popcll(bal);
    }
    wave_fence();
    for (int q = lane; q < c; q += 64) {
        const int32_t key = list[q];
        int32_t rank = 0;
        for (int o = 0; o < c; ++o) rank += list[o] < key;
        if (rank < cnt) {
            count_or_cols[base + rank] = key;
            cv[base + rank] = vals[slot[q]];
        }
    }
}

// dense copy of the coarsest matrix
__global__ void k_amg_dense(int n, const int32_t* __restrict__ rp, const int32_t* __restrict__ cl,
                            const double* __restrict__ kv, double* __restrict__ g) {
    const int i = blockIdx.x;
    for (int j = threadIdx.x; j < n; j += blockDim.x) g[i * n + j] = 0.0;
    __syncthreads();
    for (int32_t s = rp[i] + (int32_t)threadIdx.x; s < rp[i + 1]; s += blockDim.x) g[i * n + cl[s]] = kv[s];
}
// inverse = T T^T from the upper triangular T with T^T G T = I
__global__ void k_amg_inverse(int n, const double* __restrict__ t, double* __restrict__ g) {
    const int i = blockIdx.x;
    for (int j = threadIdx.x; j < n; j += blockDim.x) {
        double a = 0.0;
        for (int k = i > j ? i : j; k < n; ++k) a += t[i * n + k] * t[j * n + k];
        g[i * n + j] = a;
    }
}

// ---- cycle --------------------------------------------------------------------
// Every kernel works on row-major blocks of m columns, rows in XCD-contiguous
// ranges, G lanes for each row and column.  The finest level's ELL rows take
// one lane (its slots are loaded, then the gathers go out together; bound by
// HBM); CSR rows take 1 to 16 by their mean length, a lane every G-th entry
// and the sums combined in a fixed order: with one lane a row of 12 entries
// took 4.7 us a launch and one of 70 entries 35 us on levels that fill a
// fraction of the chip, all of it latency.

// this lane's share of sum over row i of K of kv * f(column); W > 0: ELL rows
// of W slots (double, G == 1)
template <int W, int G, typename T, typename F>
__device__ __forceinline__ T row_part(int64_t i, int lane, const int32_t* __restrict__ rp,
                                      const int32_t* __restrict__ cl, const T* __restrict__ kv, F&& f) {
    T a = T(0);
    if constexpr (W > 0) {
        static_assert(sizeof(T) == 8, "the block kernels have their own ELL rows");
#pragma unroll
        for (int k0 = 0; k0 < W; k0 += 8) {
            const int4 ca = *reinterpret_cast<const int4*>(cl + i * W + k0);
            const int4 cb = *reinterpret_cast<const int4*>(cl + i * W + k0 + 4);
            const double2* vp = reinterpret_cast<const double2*>(kv + i * W + k0);
            const double2 v0 = vp[0], v1 = vp[1], v2 = vp[2], v3 = vp[3];
            const double g0 = f(ca.x), g1 = f(ca.y), g2 = f(ca.z), g3 = f(ca.w);
            const double g4 = f(cb.x), g5 = f(cb.y), g6 = f(cb.z), g7 = f(cb.w);
            a += v0.x * g0;
            a += v0.y * g1;
            a += v1.x * g2;
            a += v1.y * g3;
            a += v2.x * g4;
            a += v2.y * g5;
            a += v3.x * g6;
            a += v3.y * g7;
        }
    } else {
        int32_t s = rp[i] + lane;
        const int32_t r1 = rp[i + 1];
        for (; s + 3 * G < r1; s += 4 * G) {
            const T g0 = f(cl[s]), g1 = f(cl[s + G]), g2 = f(cl[s + 2 * G]), g3 = f(cl[s + 3 * G]);
            a += kv[s] * g0;
            a += kv[s + G] * g1;
            a += kv[s + 2 * G] * g2;
            a += kv[s + 3 * G] * g3;
        }
        for (; s < r1; s += G) a += kv[s] * f(cl[s]);
    }
    return a;
}
// the row's sum, in every one of its G lanes
template <int W, int G, typename T, typename F>
__device__ __forceinline__ T row_sum(int64_t i, int lane, const int32_t* __restrict__ rp,
                                     const int32_t* __restrict__ cl, const T* __restrict__ kv, F&& f) {
    T a = row_part<W, G>(i, lane, rp, cl, kv, f);
#pragma unroll
    for (int o = G / 2; o > 0; o >>= 1) a += __shfl_xor(a, o, 64);
    return a;
}
// row, column and lane of a thread; false beyond the block's end
template <int G>
__device__ __forceinline__ bool place(int64_t n, int m, int64_t& i, int& c, int& lane) {
    const int64_t gid = xcd_block() * 256 + threadIdx.x;
    const int64_t t = gid / G;
    lane = (int)(gid % G);
    i = m == 1 ? t : t / m;
    c = m == 1 ? 0 : (int)(t - i * m);
    return i < n;
}

// the degree-2 smoother from x = 0: with x1 = s D^-1 b,
// x = (1 + c1) x1 + c2 D^-1 (b - K x1)
template <int W, int G>
__global__ void __launch_bounds__(256)
k_amg_pre(int64_t n, int m, const int32_t* __restrict__ rp, const int32_t* __restrict__ cl,
          const double* __restrict__ kv, const double* __restrict__ dinv, const double* __restrict__ b,
          double* __restrict__ x, double s, double c1, double c2, const int* __restrict__ status) {
    if (status && status[0]) return;
    int64_t i;
    int c, lane;
    if (!place<G>(n, m, i, c, lane)) return;
    const double di = dinv[i], bi = b[i * m + c];
    const double a = row_sum<W, G>(i, lane, rp, cl, kv, [&](int32_t j) { return dinv[j] * b[(int64_t)j * m + c]; });
    if (lane == 0) x[i * m + c] = (1.0 + c1) * s * di * bi + c2 * di * (bi - s * a);
}
// MODE 0: out = b - K x; 1: out = x + g D^-1 (b - K x);
// 2: out = w0 x + w1 out + g D^-1 (b - K x); 3: as 2, and the workgroup's
// partial sums of b . out per column (m <= 4) into part[block * m + column]
template <int W, int G, int MODE>
__global__ void __launch_bounds__(256)
k_amg_step(int64_t n, int m, const int32_t* __restrict__ rp, const int32_t* __restrict__ cl,
           const double* __restrict__ kv, const double* __restrict__ dinv, const double* __restrict__ b,
           const double* __restrict__ x, double* __restrict__ out, double w0, double w1, double g,
           double* __restrict__ part, const int* __restrict__ status) {
    if (status && status[0]) return;
    int64_t i;
    int c, lane;
    const bool in = place<G>(n, m, i, c, lane);
    double dot = 0.0;
    if (in) {
        const int64_t o = i * m + c;
        const double bi = b[o];
        const double r = bi - row_sum<W, G>(i, lane, rp, cl, kv, [&](int32_t j) { return x[(int64_t)j * m + c]; });
        if (lane == 0) {
            double v = r;
            if (MODE >= 1) v = (MODE == 1 ? x[o] : w0 * x[o] + w1 * out[o]) + g * dinv[i] * r;
            out[o] = v;
            dot = bi * v;
        }
    }
    if constexpr (MODE == 3) {
        __shared__ double sh[4][4];
        for (int q = 0; q < m; ++q) {
            const double t = wave_sum64(in && c == q ? dot : 0.0);
            if ((threadIdx.x & 63) == 0) sh[q][threadIdx.x >> 6] = t;
        }
        __syncthreads();
        if ((int)threadIdx.x < m)
            part[(int64_t)blockIdx.x * m + threadIdx.x] =
                (sh[threadIdx.x][0] + sh[threadIdx.x][1]) + (sh[threadIdx.x][2] + sh[threadIdx.x][3]);
    }
}
// out (+)= M in for the transfer operators
template <bool ADD, int G>
__global__ void __launch_bounds__(256)
k_amg_transfer(int64_t n, int m, const int32_t* __restrict__ mp, const int32_t* __restrict__ mc,
               const double* __restrict__ mv, const double* __restrict__ in, double* __restrict__ out,
               const int* __restrict__ status) {
    if (status && status[0]) return;
    int64_t i;
    int c, lane;
    if (!place<G>(n, m, i, c, lane)) return;
    const double a = row_sum<0, G>(i, lane, mp, mc, mv, [&](int32_t j) { return in[(int64_t)j * m + c]; });
    if (lane == 0) {
        if (ADD) out[i * m + c] += a;
        else out[i * m + c] = a;
    }
}

// the tail: every level from `first` on for one column per workgroup, the
// vectors in LDS.  A level's vectors start at `off` (rows of the tail's
// levels before it).
template <typename T>
struct TailLevel {
    int n, off;
    const int32_t *rp, *cl;
    const T *kv, *dinv;
    const int32_t *pp, *pc, *tp, *tc;
    const T *pv, *tv;
    T s, c1, c2;
};
template <typename T>
struct TailDesc {
    int count;  // levels, the last one with the inverse
    TailLevel<T> lv[kMaxLevels];
    const double* ginv;
};
constexpr int kTailThreads = 1024;

// put(i, sum over row i of kv * v) for the rows of a CSR matrix, v in LDS,
// four lanes a row
template <typename T, typename P>
__device__ __forceinline__ void tail_rows(int n, const int32_t* __restrict__ rp, const int32_t* __restrict__ cl,
                                          const T* __restrict__ kv, const T* v, P&& put) {
    constexpr int G = 4;
    for (int t = threadIdx.x; t < n * G; t += kTailThreads) {
        const int i = t / G, lane = t % G;
        const T a = row_sum<0, G>(i, lane, rp, cl, kv, [&](int32_t j) { return v[j]; });
        if (lane == 0) put(i, a);
    }
}

template <typename T>
__global__ void __launch_bounds__(kTailThreads)
k_amg_tail(int ld, const TailDesc<T>* __restrict__ desc, const T* __restrict__ b, T* __restrict__ x,
           const int* __restrict__ status) {
    if (status && status[0]) return;
    __shared__ T sb[kTailSum], sx[kTailSum], sy[kTailSum];
    __shared__ double red[kTailThreads];
    const int tid = threadIdx.x, col = blockIdx.x;
    const int count = desc->count;
    {
        const int n = desc->lv[0].n;
        for (int i = tid; i < n; i += kTailThreads) sb[i] = b[(int64_t)i * ld + col];
    }
    __syncthreads();
    // down: smooth from zero, restrict the residual
    for (int l = 0; l + 1 < count; ++l) {
        const TailLevel<T>& lv = desc->lv[l];
        const T* bl = sb + lv.off;
        T* xl = sx + lv.off;
        T* yl = sy + lv.off;
        for (int i = tid; i < lv.n; i += kTailThreads) yl[i] = lv.s * lv.dinv[i] * bl[i];
        __syncthreads();
        tail_rows<T>(lv.n, lv.rp, lv.cl, lv.kv, yl, [&](int i, T a) {
            xl[i] = (T(1) + lv.c1) * yl[i] + lv.c2 * lv.dinv[i] * (bl[i] - a);
        });
        __syncthreads();
        tail_rows<T>(lv.n, lv.rp, lv.cl, lv.kv, xl, [&](int i, T a) { yl[i] = bl[i] - a; });
        __syncthreads();
        const TailLevel<T>& nx = desc->lv[l + 1];
        tail_rows<T>(nx.n, lv.tp, lv.tc, lv.tv, yl, [&](int i, T a) { sb[nx.off + i] = a; });
        __syncthreads();
    }
    // the last level: x = K^-1 b, 8 threads a row
    {
        const TailLevel<T>& lv = desc->lv[count - 1];
        const int n = lv.n;  // <= 128
        const int i = tid & 127, part = tid >> 7;
        double a = 0.0;
        if (i < n)
            for (int k = part; k < n; k += kTailThreads / 128) a += desc->ginv[k * n + i] * (double)sb[lv.off + k];
        red[tid] = a;
        __syncthreads();
        if (tid < n) {
            double t = 0.0;
#pragma unroll
            for (int p = 0; p < kTailThreads / 128; ++p) t += red[tid + 128 * p];
            sx[lv.off + tid] = (T)t;
        }
        __syncthreads();
    }
    // up: correct, smooth
    for (int l = count - 2; l >= 0; --l) {
        const TailLevel<T>& lv = desc->lv[l];
        const T* bl = sb + lv.off;
        const T* xc = sx + desc->lv[l + 1].off;
        T* xl = sx + lv.off;
        T* yl = sy + lv.off;
        for (int i = tid; i < lv.n; i += kTailThreads)
            xl[i] += row_sum<0, 1>(i, 0, lv.pp, lv.pc, lv.pv, [&](int32_t j) { return xc[j]; });
        __syncthreads();
        tail_rows<T>(lv.n, lv.rp, lv.cl, lv.kv, xl,
                     [&](int i, T a) { yl[i] = xl[i] + lv.s * lv.dinv[i] * (bl[i] - a); });
        __syncthreads();
        tail_rows<T>(lv.n, lv.rp, lv.cl, lv.kv, yl, [&](int i, T a) {
            xl[i] = (T(1) + lv.c1) * yl[i] - lv.c1 * xl[i] + lv.c2 * lv.dinv[i] * (bl[i] - a);
        });
        __syncthreads();
    }
    const int n = desc->lv[0].n;
    for (int i = tid; i < n; i += kTailThreads) x[(int64_t)i * ld + col] = sx[i];
}

// ---- block cycle: FP32 blocks of the eigensolver ------------------------------
// Rows of ld columns (ld a multiple of 4), LPR lanes of four columns a row, the
// entries of a row taken four at a time so that four gathers are in flight;
// E8: the finest level's ELL rows of 8 slots, staged in LDS by one coalesced
// load of the workgroup.  Bound by HBM on the finest level (a block of 64
// columns of 655,362 rows is 168 MB; the gathers of the locality-ordered rows
// hit L2) and by launch latency on the others.
enum { kBlkPre = 0, kBlkRes = 1, kBlkSt1 = 2, kBlkSt2 = 3, kBlkMix = 4 };

__device__ __forceinline__ float4 f4mul(float w, const float4& a) {
    return make_float4(w * a.x, w * a.y, w * a.z, w * a.w);
}
__device__ __forceinline__ void f4add(float4& y, float w, const float4& a) {
    y.x += w * a.x;
    y.y += w * a.y;
    y.z += w * a.z;
    y.w += w * a.w;
}
// sum over `len` entries (cols, vals) of vals * v[cols, c0 .. c0 + 3], times
// dscale[col] when given; a partial last group repeats `self` with weight 0
template <bool DS>
__device__ __forceinline__ float4 blk_gather(const int32_t* cols, const float* vals, int len, int32_t self,
                                             const float* __restrict__ dscale, const float* __restrict__ v, int ld,
                                             int c0) {
    float4 a0 = make_float4(0.f, 0.f, 0.f, 0.f), a1 = a0;
    for (int s = 0; s < len; s += 4) {
        int32_t j[4];
        float w[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const bool in = s + q < len;
            j[q] = in ? cols[s + q] : self;
            w[q] = in ? vals[s + q] : 0.f;
            if (DS) w[q] *= dscale[j[q]];
        }
        float4 x[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) x[q] = *reinterpret_cast<const float4*>(v + (int64_t)j[q] * ld + c0);
        f4add(a0, w[0], x[0]);
        f4add(a1, w[1], x[1]);
        f4add(a0, w[2], x[2]);
        f4add(a1, w[3], x[3]);
    }
    f4add(a0, 1.f, a1);
    return a0;
}

// kBlkPre: out = w0 D^-1 b + g D^-1 (b - w1 K D^-1 b); kBlkRes: out = b - g K x;
// kBlkMix: out = w0 out + w1 b - g K x;
// kBlkSt1: out = x + g D^-1 (b - K x); kBlkSt2: out = w0 x + w1 out + g D^-1 (b - K x)
template <int MODE, int LPR, bool E8>
__global__ void __launch_bounds__(256)
k_blk_step(int64_t n, int ld, const int32_t* __restrict__ rp, const int32_t* __restrict__ cl,
           const float* __restrict__ kv, const float* __restrict__ dinv, const float* __restrict__ b,
           const float* __restrict__ x, float* __restrict__ out, float w0, float w1, float g) {
    constexpr int kRows = 256 / LPR;
    __shared__ __align__(16) int32_t s_cols[E8 ? kRows * 8 : 4];
    __shared__ __align__(16) float s_kv[E8 ? kRows * 8 : 4];
    const int64_t blk = xcd_block();
    const int64_t row = (blk * 256 + threadIdx.x) / LPR;
    if (E8) {
        const int64_t base = blk * kRows * 8;
        for (int t = threadIdx.x; t < kRows * 8; t += 256) {
            const bool in = base + t < n * 8;
            s_cols[t] = in ? cl[base + t] : 0;
            s_kv[t] = in ? kv[base + t] : 0.f;
        }
        __syncthreads();
    }
    if (row >= n) return;
    const int32_t r0 = E8 ? 0 : rp[row];
    const int len = E8 ? 8 : rp[row + 1] - r0;
    const int32_t* cols = E8 ? s_cols + (threadIdx.x / LPR) * 8 : cl + r0;
    const float* vals = E8 ? s_kv + (threadIdx.x / LPR) * 8 : kv + r0;
    const float di = dinv[row];
    for (int c0 = (int)(threadIdx.x % LPR) * 4; c0 < ld; c0 += LPR * 4) {
        const int64_t o = row * ld + c0;
        const float4 bi = *reinterpret_cast<const float4*>(b + o);
        float4 y;
        if (MODE == kBlkPre) {
            const float4 a = blk_gather<true>(cols, vals, len, (int32_t)row, dinv, b, ld, c0);
            y = f4mul(w0 * di + g * di, bi);
            f4add(y, -g * di * w1, a);
        } else {
            const float4 a = blk_gather<false>(cols, vals, len, (int32_t)row, nullptr, x, ld, c0);
            if (MODE == kBlkRes) {
                y = bi;
                f4add(y, -g, a);
            } else if (MODE == kBlkMix) {
                y = f4mul(w0, *reinterpret_cast<const float4*>(out + o));
                f4add(y, w1, bi);
                f4add(y, -g, a);
            } else {
                const float4 xi = *reinterpret_cast<const float4*>(x + o);
                float4 r = bi;
                f4add(r, -1.f, a);
                if (MODE == kBlkSt1) {
                    y = xi;
                } else {
                    y = f4mul(w0, xi);
                    f4add(y, w1, *reinterpret_cast<const float4*>(out + o));
                }
                f4add(y, g * di, r);
            }
        }
        *reinterpret_cast<float4*>(out + o) = y;
    }
}
// out += P in: a fine row has at most a few entries
template <int LPR>
__global__ void __launch_bounds__(256)
k_blk_prolong(int64_t n, int ld, const int32_t* __restrict__ mp, const int32_t* __restrict__ mc,
              const float* __restrict__ mv, const float* __restrict__ in, float* __restrict__ out) {
    const int64_t row = (xcd_block() * 256 + threadIdx.x) / LPR;
    if (row >= n) return;
    const int32_t r0 = mp[row];
    const int len = mp[row + 1] - r0;
    for (int c0 = (int)(threadIdx.x % LPR) * 4; c0 < ld; c0 += LPR * 4) {
        const int64_t o = row * ld + c0;
        float4 y = *reinterpret_cast<const float4*>(out + o);
        if (len > 0) f4add(y, 1.f, blk_gather<false>(mc + r0, mv + r0, len, mc[r0], nullptr, in, ld, c0));
        *reinterpret_cast<float4*>(out + o) = y;
    }
}
// out = R in: a coarse row gathers the fine rows of its whole neighbourhood
// (some 60 of a triangle mesh, 200 to 400 of a tet mesh) and there are few of
// them, so a row is one serial chain of gathers unless its entries are split:
// a wave a row, whose 64 / LPR groups of lanes take contiguous parts; their
// sums are added pairwise by shuffles (35,937 tet vertices, 30 pairs: a whole solve
// 39.6 -> 32.6 ms, of which one lane group a row spent 3.6 ms here).
template <int LPR>
__global__ void __launch_bounds__(256)
k_blk_restrict(int64_t n, int ld, const int32_t* __restrict__ mp, const int32_t* __restrict__ mc,
               const float* __restrict__ mv, const float* __restrict__ in, float* __restrict__ out) {
    constexpr int kParts = 64 / LPR;
    const int64_t row = xcd_block() * 4 + (threadIdx.x >> 6);
    if (row >= n) return;  // whole wave exits together
    const int lane = (int)(threadIdx.x & 63), part = lane / LPR;
    const int32_t r0 = mp[row];
    const int len = mp[row + 1] - r0;
    const int per = ((len + kParts - 1) / kParts + 3) / 4 * 4;
    const int s0 = min(part * per, len), cnt = min(per, len - s0);
    for (int cb = 0; cb < ld; cb += LPR * 4) {
        const int c0 = cb + (lane % LPR) * 4;
        float4 y = make_float4(0.f, 0.f, 0.f, 0.f);
        if (c0 < ld && cnt > 0) y = blk_gather<false>(mc + r0 + s0, mv + r0 + s0, cnt, mc[r0 + s0], nullptr, in, ld, c0);
#pragma unroll
        for (int d = LPR; d < 64; d *= 2) {
            y.x += __shfl_xor(y.x, d);
            y.y += __shfl_xor(y.y, d);
            y.z += __shfl_xor(y.z, d);
            y.w += __shfl_xor(y.w, d);
        }
        if (c0 < ld && part == 0) *reinterpret_cast<float4*>(out + row * ld + c0) = y;
    }
}
// b = the columns perm[0 .. m - 1] of W (all in order when perm is null) in
// FP32, columns m .. ld - 1 zero
template <typename WT>
__global__ void k_blk_in(int64_t n, int m, int ld, const WT* __restrict__ W, int ldw, const int32_t* __restrict__ perm,
                         float* __restrict__ b) {
    const int64_t gid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (gid >= n * ld) return;
    const int64_t i = gid / ld;
    const int c = (int)(gid - i * ld);
    b[gid] = c < m ? (float)W[i * ldw + (perm ? perm[c] : c)] : 0.f;
}
// the same columns of W = w1 x1 + w2 x2 (+ w3 x3); with perm, the total - m
// other columns perm[m ..] times dinv (Jacobi)
template <typename WT>
__global__ void k_blk_out(int64_t n, int m, int total, int ld, const float* __restrict__ x1,
                          const float* __restrict__ x2, const float* __restrict__ x3, double w1, double w2, double w3,
                          const double* __restrict__ dinv, const int32_t* __restrict__ perm, WT* __restrict__ W,
                          int ldw) {
    const int64_t gid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (gid >= n * total) return;
    const int64_t i = gid / total;
    const int c = (int)(gid - i * total);
    WT* w = W + i * ldw + (perm ? perm[c] : c);
    if (c >= m) {
        *w = (WT)((double)*w * dinv[i]);
        return;
    }
    const int64_t o = i * ld + c;
    double v = w1 * (double)x1[o] + w2 * (double)x2[o];
    if (x3) v += w3 * (double)x3[o];
    *w = (WT)v;
}
__global__ void k_narrow(int64_t cnt, const double* __restrict__ s, float* __restrict__ d) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < cnt) d[i] = (float)s[i];
}
// K's values in the slots of an ELL copy of its pattern (padding: 0)
__global__ void k_amg_ell(int64_t n, int W, const int32_t* __restrict__ rp, const double* __restrict__ kv,
                          float* __restrict__ ekv) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int32_t r0 = rp[i], len = rp[i + 1] - r0;
    for (int q = 0; q < W; ++q) ekv[i * W + q] = q < len ? (float)kv[r0 + q] : 0.f;
}

__global__ void k_fill_one(int64_t n, const double* __restrict__ dinv, double* __restrict__ x) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) x[i] = dinv[i] > 0.0 ? 1.0 : 0.0;
}

constexpr int kRB = 256;  // blocks of the Rayleigh quotient

}  // namespace

double amg_condition(lh_ctx* ctx, int64_t n, const int32_t* rp, const int32_t* cl, const double* kv,
                     const double* dinv) {
    DevBuf x(n * 8), y(n * 8), part(2 * kRB * 8);
    k_fill_one<<<nblocks(n, 256), 256, 0, ctx->stream>>>(n, dinv, x.as<double>());
    k_amg_power<8><<<nblocks_xcd(n * 8, 256), 256, 0, ctx->stream>>>(n, rp, cl, kv, dinv, x.as<double>(), y.as<double>());
    k_amg_rayleigh<<<kRB, 256, 0, ctx->stream>>>(n, dinv, x.as<double>(), y.as<double>(), part.as<double>());
    LH_CHECK_LAUNCH();
    double hp[2 * kRB], d = 0.0, k = 0.0;
    d2h(ctx, hp, part.p, sizeof(hp));
    for (int q = 0; q < kRB; ++q) {
        d += hp[2 * q];
        k += hp[2 * q + 1];
    }
    return k > 0.0 ? 2.0 * d / k : 1e30;
}

template <typename X>
X* Amg::own(size_t count) {
    keep.emplace_back(std::max<size_t>(count, 1) * sizeof(X));
    return keep.back().as<X>();
}

bool Amg::setup(lh_ctx* c, int64_t n0, int64_t nnz0, const int32_t* rp0, const int32_t* cl0, const double* kv0,
                int ell_w, const int32_t* ecl, const double* ekv, double coarse_shift) {
    ctx = c;
    levels.clear();
    keep.clear();
    hipStream_t st = ctx->stream;
    DevBuf flags(64);         // [0] bad diagonal, [1] hash table too small, [2 + level] longest row
    static_assert((2 + kMaxLevels) * 4 <= 64, "flags");
    memset_d(ctx, flags.p, 0, 64);
    int* bad = flags.as<int>();
    int* over = bad + 1;
    int64_t n = n0, nnz = nnz0;
    const int32_t *rp = rp0, *cl = cl0;
    const double* kv = kv0;
    DevBuf x(n0 * 8), y(n0 * 8), part(2 * kRB * 8), gersh(n0 * 8), key(n0 * 8), key2(n0 * 8), agg(n0 * 4), agg2(n0 * 4),
        cnt((n0 + 1) * 4), idx((n0 + 1) * 4), strong;
    double theta = kTheta;
    for (int l = 0; l < kMaxLevels; ++l) {
        levels.emplace_back();
        AmgLevel& lv = levels.back();
        lv.n = n;
        lv.nnz = nnz;
        lv.rp = rp;
        lv.cl = cl;
        lv.d.kv = kv;
        double* dinv = own<double>(n);
        lv.d.dinv = dinv;
        if (l == 0 && ell_w) {
            lv.W = ell_w;
            lv.ecl = ecl;
            lv.ekv = ekv;
        }
        const unsigned nb = nblocks(n, 256), nbx = nblocks_xcd(n, 256);
        const int g = lanes_for(nnz, n);
        const unsigned nbg = nblocks_xcd(n * g, 256);
        with_lanes(g, [&](auto G) { k_amg_diag<G.v><<<nbg, 256, 0, st>>>(n, rp, cl, kv, dinv, gersh.as<double>(), x.as<double>(), bad, bad + 2 + l); });
        LH_CHECK_LAUNCH();
        if (n <= kCoarsest) {
            // last level: its inverse
            DevBuf g((size_t)n * n * 8), t((size_t)n * n * 8), stt(64);
            ginv.alloc((size_t)n * n * 8);
            k_amg_dense<<<(unsigned)n, 128, 0, st>>>((int)n, rp, cl, kv, g.as<double>());
            LH_CHECK_LAUNCH();
            cholinv(ctx, (int)n, g.as<double>(), t.as<double>(), coarse_shift, stt.as<int>());
            k_amg_inverse<<<(unsigned)n, 128, 0, st>>>((int)n, t.as<double>(), ginv.as<double>());
            LH_CHECK_LAUNCH();
            int hs = 0, hb[2] = {0, 0};
            const Xfer q[2] = {{&hs, stt.p, 4}, {hb, flags.p, 8}};
            d2h_n(ctx, q, 2);
            if (hs || hb[0] || hb[1] || l == 0) return false;
            break;
        }
        double *xa = x.as<double>(), *ya = y.as<double>();
        for (int q = 0; q < kPowerSteps; ++q) {
            with_lanes(g, [&](auto G) { k_amg_power<G.v><<<nbg, 256, 0, st>>>(n, rp, cl, kv, dinv, xa, ya); });
            if (q + 1 < kPowerSteps) std::swap(xa, ya);
        }
        k_amg_rayleigh<<<kRB, 256, 0, st>>>(n, dinv, xa, ya, part.as<double>());
        LH_CHECK_LAUNCH();
        // aggregates
        strong.ensure((size_t)nnz * 4);
        const double th2 = theta * theta;
        theta *= 0.5;
        auto* ta = key.as<unsigned long long>();
        auto* tb = key2.as<unsigned long long>();
        k_mis_init<<<nb, 256, 0, st>>>(n, dinv, ta);
        int32_t* sc = strong.as<int32_t>();
        with_lanes(g, [&](auto G) {
            k_strong<G.v><<<nbg, 256, 0, st>>>(n, rp, cl, kv, dinv, th2, sc);
            for (int r = 0; r < kMisRounds; ++r) {
                k_mis_spread<G.v><<<nbg, 256, 0, st>>>(n, rp, sc, ta, tb);
                k_mis_decide<G.v><<<nbg, 256, 0, st>>>(n, rp, sc, tb, ta);
            }
        });
        k_mis_flag<<<nb, 256, 0, st>>>(n, ta, cnt.as<int32_t>());
        LH_CHECK_LAUNCH();
        exclusive_scan_i32(ctx, cnt.as<int32_t>(), idx.as<int32_t>(), n);
        k_agg_roots<<<nb, 256, 0, st>>>(n, cnt.as<int32_t>(), idx.as<int32_t>(), agg.as<int32_t>());
        int32_t *ga = agg.as<int32_t>(), *gb = agg2.as<int32_t>();
        for (int r = 0; r < 3; ++r) {
            with_lanes(g, [&](auto G) { k_agg_join<G.v><<<nbg, 256, 0, st>>>(n, rp, sc, kv, ga, gb); });
            std::swap(ga, gb);
        }
        LH_CHECK_LAUNCH();
        double hp[2 * kRB];
        int32_t nc32 = 0;
        int hb[2 + kMaxLevels] = {};
        {
            const Xfer q[3] = {{hp, part.p, sizeof(hp)}, {&nc32, idx.as<int32_t>() + n, 4}, {hb, flags.p, sizeof(hb)}};
            d2h_n(ctx, q, 3);
        }
        double xdx = 0.0, xkx = 0.0;
        for (int q = 0; q < kRB; ++q) {
            xdx += hp[2 * q];
            xkx += hp[2 * q + 1];
        }
        const double lmax = xdx > 0.0 ? xkx / xdx : 0.0;
        const int64_t nc = nc32;
        // a stalled coarsening, a bad diagonal or a meaningless estimate: no hierarchy
        if (hb[0] || hb[1] || nc < 1 || nc > n * 7 / 10 || !(lmax > 0.0) || !std::isfinite(lmax)) return false;
        if (l == 0) rough = lmax;
        lv.bmax = std::min(1.1 * lmax, kSmoothTop);
        k_amg_guard<<<nb, 256, 0, st>>>(n, gersh.as<double>(), kGuard * lv.bmax, dinv);
        LH_CHECK_LAUNCH();
        const double w = 4.0 / (3.0 * lv.bmax);
        // P
        int32_t* pp = own<int32_t>(n + 1);
        const bool long_rows = nnz > kLongRow * n || hb[2 + l] > 0;
        if (long_rows)
            k_prolongator_wave<false><<<nblocks(n, 4), 256, 0, st>>>(n, rp, cl, kv, dinv, w, ga, nullptr,
                                                                     cnt.as<int32_t>(), nullptr);
        else
            k_prolongator<false><<<nbx, 256, 0, st>>>(n, rp, cl, kv, dinv, w, ga, nullptr, cnt.as<int32_t>(), nullptr);
        LH_CHECK_LAUNCH();
        exclusive_scan_i32(ctx, cnt.as<int32_t>(), pp, n);
        // one entry per distinct aggregate of a row: at most nnz
        int32_t* pc = own<int32_t>(nnz);
        double* pv = own<double>(nnz);
        if (long_rows)
            k_prolongator_wave<true><<<nblocks(n, 4), 256, 0, st>>>(n, rp, cl, kv, dinv, w, ga, pp, pc, pv);
        else
            k_prolongator<true><<<nbx, 256, 0, st>>>(n, rp, cl, kv, dinv, w, ga, pp, pc, pv);
        LH_CHECK_LAUNCH();
        int32_t pnnz = 0;
        d2h(ctx, &pnnz, pp + n, 4);
        // P^T
        int32_t* tp = own<int32_t>(nc + 1);
        int32_t* tc = own<int32_t>(pnnz);
        double* tv = own<double>(pnnz);
        {
            DevBuf fill((nc + 1) * 4), t2((size_t)std::max(pnnz, 1) * 4), v2((size_t)std::max(pnnz, 1) * 8);
            memset_d(ctx, cnt.p, 0, nc * 4);
            memset_d(ctx, fill.p, 0, nc * 4);
            k_count_cols<<<nblocks(std::max(pnnz, 1), 256), 256, 0, st>>>(pnnz, pc, cnt.as<int32_t>());
            LH_CHECK_LAUNCH();
            exclusive_scan_i32(ctx, cnt.as<int32_t>(), tp, nc);
            k_scatter_cols<<<nb, 256, 0, st>>>(n, pp, pc, pv, tp, fill.as<int32_t>(), t2.as<int32_t>(), v2.as<double>());
            k_sort_rows<<<nblocks(nc, 4), 256, 0, st>>>(nc, tp, t2.as<int32_t>(), v2.as<double>(), tc, tv);
            LH_CHECK_LAUNCH();
            if (!fill.pooled || !t2.pooled || !v2.pooled) HIPX(hipStreamSynchronize(st));  // they go out of scope
        }
        lv.nc = nc;
        lv.pnnz = pnnz;
        lv.pp = pp;
        lv.pc = pc;
        lv.d.pv = pv;
        lv.tp = tp;
        lv.tc = tc;
        lv.d.rv = tv;
        // K P, then P^T (K P): tables of 256 columns, of 1,024 where a row
        // overflows them
        auto product = [&](int64_t rows, const int32_t* xp, const int32_t* xc, const double* xv, const int32_t* yp,
                           const int32_t* yc, const double* yv, int32_t*& op, int32_t*& oc, double*& ov,
                           std::vector<DevBuf>& into) -> int32_t {
            const unsigned g = nblocks(rows, 4);
            auto get = [&](size_t bytes) -> void* {
                into.emplace_back(bytes);
                return into.back().p;
            };
            op = static_cast<int32_t*>(get((rows + 1) * 4));
            bool wide = false;
            int32_t total = 0;
            for (;;) {
                if (wide)
                    k_spgemm<1024, false><<<g, 256, 0, st>>>(rows, xp, xc, xv, yp, yc, yv, nullptr, cnt.as<int32_t>(),
                                                             nullptr, over);
                else
                    k_spgemm<256, false><<<g, 256, 0, st>>>(rows, xp, xc, xv, yp, yc, yv, nullptr, cnt.as<int32_t>(),
                                                            nullptr, over);
                LH_CHECK_LAUNCH();
                exclusive_scan_i32(ctx, cnt.as<int32_t>(), op, rows);
                int o = 0;
                const Xfer q[2] = {{&total, op + rows, 4}, {&o, over, 4}};
                d2h_n(ctx, q, 2);
                if (!o) break;
                if (wide) return -1;
                wide = true;
                memset_d(ctx, over, 0, 4);
            }
            oc = static_cast<int32_t*>(get((size_t)std::max(total, 1) * 4));
            ov = static_cast<double*>(get((size_t)std::max(total, 1) * 8));
            if (wide)
                k_spgemm<1024, true><<<g, 256, 0, st>>>(rows, xp, xc, xv, yp, yc, yv, op, oc, ov, over);
            else
                k_spgemm<256, true><<<g, 256, 0, st>>>(rows, xp, xc, xv, yp, yc, yv, op, oc, ov, over);
            LH_CHECK_LAUNCH();
            return total;
        };
        std::vector<DevBuf> tmp;
        int32_t *ap = nullptr, *ac = nullptr, *np_ = nullptr, *nc_ = nullptr;
        double *av = nullptr, *nv_ = nullptr;
        if (product(n, rp, cl, kv, pp, pc, pv, ap, ac, av, tmp) < 0) return false;
        const int32_t cnnz = product(nc, tp, tc, tv, ap, ac, av, np_, nc_, nv_, keep);
        if (cnnz < 0) return false;
        for (const DevBuf& t : tmp)
            if (!t.pooled) {
                HIPX(hipStreamSynchronize(st));  // K P goes out of scope
                break;
            }
        n = nc;
        nnz = cnnz;
        rp = np_;
        cl = nc_;
        kv = nv_;
        if (l + 1 == kMaxLevels) return false;
    }
    // the tail: the levels of at most kTailRows rows, kTailSum together
    const int last = (int)levels.size() - 1;
    tail = last;
    int64_t sum = levels[last].n;
    while (tail > 0 && levels[tail - 1].n <= kTailRows && levels[tail - 1].nnz <= kTailNnz &&
           sum + levels[tail - 1].n <= kTailSum)
        sum += levels[--tail].n;
    return true;
}

template <typename T>
void Amg::describe_tail() {
    const int last = (int)levels.size() - 1;
    TailDesc<T> d{};
    d.count = last - tail + 1;
    d.ginv = ginv.as<double>();
    int off = 0;
    for (int l = tail; l <= last; ++l) {
        const AmgLevel& lv = levels[l];
        const AmgOps<T>& o = lv.ops(T());
        TailLevel<T>& t = d.lv[l - tail];
        t.n = (int)lv.n;
        t.off = off;
        off += (int)lv.n;
        t.rp = lv.rp;
        t.cl = lv.cl;
        t.kv = o.kv;
        t.dinv = o.dinv;
        t.pp = lv.pp;
        t.pc = lv.pc;
        t.pv = o.pv;
        t.tp = lv.tp;
        t.tc = lv.tc;
        t.tv = o.rv;
        const Cheb2 k = cheb2(lv.bmax);
        t.s = (T)k.s;
        t.c1 = (T)k.c1;
        t.c2 = (T)k.c2;
    }
    tail_desc.alloc(sizeof(TailDesc<T>));
    h2d(ctx, tail_desc.p, &d, sizeof(d));
}

void Amg::prepare(int m_) {
    m = m_;
    describe_tail<double>();
    size_t total = 0;
    for (int l = 0; l <= tail; ++l) total += 4 * (size_t)levels[l].n * m;
    work.alloc(total * 8);
    double* p = work.as<double>();
    wb.clear();
    wx.clear();
    wy.clear();
    wr.clear();
    for (int l = 0; l <= tail; ++l) {
        const size_t s = (size_t)levels[l].n * m;
        wb.push_back(p);
        wx.push_back(p + s);
        wy.push_back(p + 2 * s);
        wr.push_back(p + 3 * s);
        p += 4 * s;
    }
}

namespace {

// lanes of four columns for a block row
template <typename F>
void with_row_lanes(int lpr, F&& f) {
    switch (lpr) {
        case 1: f(IntC<1>{}); break;
        case 2: f(IntC<2>{}); break;
        case 4: f(IntC<4>{}); break;
        case 8: f(IntC<8>{}); break;
        case 16: f(IntC<16>{}); break;
        case 32: f(IntC<32>{}); break;
        default: f(IntC<64>{}); break;
    }
}

}  // namespace

void Amg::cycle(int l, const double* b, double* x, double* part, const int* status) {
    hipStream_t st = ctx->stream;
    if (l == tail) {
        k_amg_tail<double><<<(unsigned)m, kTailThreads, 0, st>>>(m, tail_desc.as<TailDesc<double>>(), b, x, status);
        LH_CHECK_LAUNCH();
        return;
    }
    const AmgLevel& lv = levels[l];
    const Cheb2 k = cheb2(lv.bmax);
    double *y = wy[l], *r = wr[l];
    const int gk = lv.W ? 1 : lanes_for(lv.nnz, lv.n);
    const unsigned nk = nblocks_xcd(lv.n * m * gk, 256);
    const int32_t* cl = lv.W ? lv.ecl : lv.cl;
    const double* kv = lv.W ? lv.ekv : lv.d.kv;
    // f(W, G) with the level's slots per row and lanes per row
    auto with_k = [&](auto&& f) {
        switch (lv.W) {
            case 8: f(IntC<8>{}, IntC<1>{}); break;
            case 16: f(IntC<16>{}, IntC<1>{}); break;
            case 24: f(IntC<24>{}, IntC<1>{}); break;
            case 32: f(IntC<32>{}, IntC<1>{}); break;
            default: with_lanes(gk, [&](auto g) { f(IntC<0>{}, g); });
        }
        LH_CHECK_LAUNCH();
    };
    with_k([&](auto w, auto g) {
        k_amg_pre<w.v, g.v><<<nk, 256, 0, st>>>(lv.n, m, lv.rp, cl, kv, lv.d.dinv, b, x, k.s, k.c1, k.c2, status);
    });
    with_k([&](auto w, auto g) {
        k_amg_step<w.v, g.v, 0><<<nk, 256, 0, st>>>(lv.n, m, lv.rp, cl, kv, lv.d.dinv, b, x, r, 0.0, 0.0, 0.0,
                                                    nullptr, status);
    });
    const int gt = lanes_for(lv.pnnz, lv.nc), gp = lanes_for(lv.pnnz, lv.n);
    with_lanes(gt, [&](auto g) {
        k_amg_transfer<false, g.v><<<nblocks_xcd(lv.nc * m * gt, 256), 256, 0, st>>>(lv.nc, m, lv.tp, lv.tc, lv.d.rv, r,
                                                                                   wb[l + 1], status);
    });
    LH_CHECK_LAUNCH();
    cycle(l + 1, wb[l + 1], wx[l + 1], nullptr, status);
    with_lanes(gp, [&](auto g) {
        k_amg_transfer<true, g.v><<<nblocks_xcd(lv.n * m * gp, 256), 256, 0, st>>>(lv.n, m, lv.pp, lv.pc, lv.d.pv,
                                                                                 wx[l + 1], x, status);
    });
    LH_CHECK_LAUNCH();
    with_k([&](auto w, auto g) {
        k_amg_step<w.v, g.v, 1><<<nk, 256, 0, st>>>(lv.n, m, lv.rp, cl, kv, lv.d.dinv, b, x, y, 0.0, 0.0, k.s,
                                                    nullptr, status);
    });
    if (part)
        with_k([&](auto w, auto g) {
            k_amg_step<w.v, g.v, 3><<<nk, 256, 0, st>>>(lv.n, m, lv.rp, cl, kv, lv.d.dinv, b, y, x, 1.0 + k.c1,
                                                        -k.c1, k.c2, part, status);
        });
    else
        with_k([&](auto w, auto g) {
            k_amg_step<w.v, g.v, 2><<<nk, 256, 0, st>>>(lv.n, m, lv.rp, cl, kv, lv.d.dinv, b, y, x, 1.0 + k.c1,
                                                        -k.c1, k.c2, nullptr, status);
        });
}

int Amg::dot_blocks() const {
    if (m > 4 || tail == 0) return 0;
    const AmgLevel& lv = levels[0];
    return (int)nblocks_xcd(lv.n * m * (lv.W ? 1 : lanes_for(lv.nnz, lv.n)), 256);
}

void Amg::apply(const double* R, double* Z, double* part, const int* status) { cycle(0, R, Z, part, status); }

// ---- blocks ---------------------------------------------------------------------
// Two or three cycles combined by the Chebyshev iteration on [lo, kBlkHi], where
// the eigenvalues of M K lie (at most 1; the smallest 0.4 to 0.6 on smooth
// surfaces, 0.1 on rough ones).  With d_1 = x_1 / theta, x_1 = M b:
//   d_k = p_k d_{k-1} + q_k x_k, z_k = z_{k-1} + d_k, x_k = M r_k, r_k = b - K z_{k-1},
// where K x_1 = theta (b - r_2) spares r_3 one product.  The eigensolver then
// needs about the iterations that the exact inverse of K would give it (50
// pairs at 10,242 vertices: 18 with two cycles or the inverse, 24 with one
// cycle, 21 with the Chebyshev-Jacobi polynomial of degree 16; 10 pairs: 14, 13, 21
// and 24; on a surface with noise of two edge lengths 15 with three cycles, 14
// with the inverse, 21 with two).  Three from kManyRows rows on, where an
// iteration's other work is ten times a cycle's; two below, where a cycle is
// launch latency and costs a seventh of an iteration.  Whole solves of caps of an
// ellipsoid with two | three cycles, ms, 10 pairs and 50: 52,418 rows 8.7 | 9.6, 31.9 | 33.5;
// 104,853 11.5 | 11.9, 50.2 | 54.0; 163,842 17.2 | 17.7, 77.5 | 75.7; 655,362,
// 50 pairs, 28 | 22 iterations.
// Three too where the estimate of lambda_max(D^-1 K) is above kRough (surfaces
// reach 2.3 with noise of two edge lengths, tets jittered by 0.18 of the spacing
// 2.1, by 0.2, which makes flat ones, 2.8 to 3.8): the cycle leaves a few of the
// flat elements' modes (eigenvalues 0.03), so 35,937 vertices jittered by 0.25 took
// 41 iterations and 24 ms (10 pairs), by 0.28 33 and 37 (30 pairs) with two, 31
// and 22, 22 and 29 with three; by 0.2, 20 and 12.5 against 18 and 13.3.
constexpr double kBlkHi = 1.02, kBlkLo2 = 0.35, kBlkLo3 = 0.2;
constexpr int64_t kManyRows = 131072;
constexpr double kRough = 2.5;

void Amg::prepare_blocks(int m_, int ell_w, const int32_t* ecl) {
    m = m_;
    ld = (m + 3) / 4 * 4;
    hipStream_t st = ctx->stream;
    auto narrow = [&](const double* s, int64_t cnt) {
        float* d = own<float>(cnt);
        k_narrow<<<nblocks(std::max<int64_t>(cnt, 1), 256), 256, 0, st>>>(cnt, s, d);
        LH_CHECK_LAUNCH();
        return d;
    };
    const int last = (int)levels.size() - 1;
    for (int l = 0; l <= last; ++l) {
        AmgLevel& lv = levels[l];
        lv.f.kv = narrow(lv.d.kv, lv.nnz);
        lv.f.dinv = narrow(lv.d.dinv, lv.n);
        if (l < last) {
            lv.f.pv = narrow(lv.d.pv, lv.pnnz);
            lv.f.rv = narrow(lv.d.rv, lv.pnnz);
        }
    }
    AmgLevel& l0 = levels[0];
    if (ell_w == 8 && tail > 0) {
        float* e = own<float>((size_t)l0.n * 8);
        k_amg_ell<<<nblocks(l0.n, 256), 256, 0, st>>>(l0.n, 8, l0.rp, l0.d.kv, e);
        LH_CHECK_LAUNCH();
        l0.W = 8;
        l0.ecl = ecl;
        l0.ekv32 = e;
    }
    describe_tail<float>();
    cycles = l0.n >= kManyRows || rough > kRough ? 3 : 2;
    size_t total = cycles * (size_t)l0.n * ld;
    for (int l = 0; l <= tail; ++l) total += (l == 0 || l < tail ? 4 : 2) * (size_t)levels[l].n * ld;
    work.alloc(total * 4);
    float* p = work.as<float>();
    auto take = [&](int64_t n) {
        float* q = p;
        p += (size_t)n * ld;
        return q;
    };
    bin = take(l0.n);
    bx1 = take(l0.n);
    if (cycles == 3) bx2 = take(l0.n);
    for (int l = 0; l <= tail; ++l) {
        fb.push_back(take(levels[l].n));
        fx.push_back(take(levels[l].n));
        if (l == 0 || l < tail) {
            fy.push_back(take(levels[l].n));
            fr.push_back(take(levels[l].n));
        }
    }
}

template <int MODE>
void Amg::blk_step(int l, int w, const float* b, const float* x, float* out, float w0, float w1, float g) {
    const AmgLevel& lv = levels[l];
    const bool e8 = lv.W == 8 && lv.ekv32;
    const int lpr = std::min(64, vec_lanes(w, 4));
    const unsigned nb = nblocks_xcd(lv.n * lpr, 256);
    const int32_t* cl = e8 ? lv.ecl : lv.cl;
    const float* kv = e8 ? lv.ekv32 : lv.f.kv;
    auto go = [&](auto L) {
        if (e8)
            k_blk_step<MODE, L.v, true><<<nb, 256, 0, ctx->stream>>>(lv.n, w, lv.rp, cl, kv, lv.f.dinv, b, x, out, w0,
                                                                     w1, g);
        else
            k_blk_step<MODE, L.v, false><<<nb, 256, 0, ctx->stream>>>(lv.n, w, lv.rp, cl, kv, lv.f.dinv, b, x, out, w0,
                                                                      w1, g);
        LH_CHECK_LAUNCH();
    };
    with_row_lanes(lpr, go);
}

void Amg::cycle_blocks(int l, int w, const float* b, float* x) {
    if (l == tail) {
        k_amg_tail<float><<<(unsigned)w, kTailThreads, 0, ctx->stream>>>(w, tail_desc.as<TailDesc<float>>(), b, x,
                                                                        nullptr);
        LH_CHECK_LAUNCH();
        return;
    }
    const AmgLevel& lv = levels[l];
    const Cheb2 k = cheb2(lv.bmax);
    const int lpr = std::min(64, vec_lanes(w, 4));
    blk_step<kBlkPre>(l, w, b, nullptr, x, (float)((1.0 + k.c1) * k.s), (float)k.s, (float)k.c2);
    blk_step<kBlkRes>(l, w, b, x, fr[l], 0.f, 0.f, 1.f);
    with_row_lanes(lpr, [&](auto L) {
        k_blk_restrict<L.v><<<nblocks_xcd(lv.nc * 64, 256), 256, 0, ctx->stream>>>(lv.nc, w, lv.tp, lv.tc, lv.f.rv, fr[l],
                                                                                 fb[l + 1]);
    });
    LH_CHECK_LAUNCH();
    cycle_blocks(l + 1, w, fb[l + 1], fx[l + 1]);
    with_row_lanes(lpr, [&](auto L) {
        k_blk_prolong<L.v><<<nblocks_xcd(lv.n * lpr, 256), 256, 0, ctx->stream>>>(lv.n, w, lv.pp, lv.pc, lv.f.pv,
                                                                                fx[l + 1], x);
    });
    LH_CHECK_LAUNCH();
    blk_step<kBlkSt1>(l, w, b, x, fy[l], 0.f, 0.f, (float)k.s);
    blk_step<kBlkSt2>(l, w, b, fy[l], x, (float)(1.0 + k.c1), (float)-k.c1, (float)k.c2);
}

template <typename WT>
void Amg::apply_blocks(WT* W, int ldw, int cols, int total, const int32_t* perm) {
    if (cols > m) LH_THROW(LH_ERR_ARG, "multigrid block width %d exceeds %d", cols, m);
    const int w = (cols + 3) / 4 * 4;
    const int64_t n = levels[0].n;
    const double lo = cycles == 3 ? kBlkLo3 : kBlkLo2;
    const double th = 0.5 * (kBlkHi + lo), de = 0.5 * (kBlkHi - lo), sig = th / de;
    const double rho1 = 1.0 / sig, rho2 = 1.0 / (2.0 * sig - rho1), rho3 = 1.0 / (2.0 * sig - rho2);
    const double p2 = rho2 * rho1, q2 = 2.0 * rho2 / de, p3 = rho3 * rho2, q3 = 2.0 * rho3 / de;
    k_blk_in<<<nblocks(n * w, 256), 256, 0, ctx->stream>>>(n, cols, w, W, ldw, perm, bin);
    LH_CHECK_LAUNCH();
    cycle_blocks(0, w, bin, bx1);
    blk_step<kBlkRes>(0, w, bin, bx1, fb[0], 0.f, 0.f, (float)(1.0 / th));
    const unsigned nb = nblocks(n * total, 256);
    const double* di = levels[0].d.dinv;
    if (cycles == 2) {
        cycle_blocks(0, w, fb[0], fx[0]);
        k_blk_out<WT><<<nb, 256, 0, ctx->stream>>>(n, cols, total, w, bx1, fx[0], nullptr, (1.0 + p2) / th, q2, 0.0, di,
                                                   perm, W, ldw);
    } else {
        cycle_blocks(0, w, fb[0], bx2);
        blk_step<kBlkMix>(0, w, fb[0], bx2, bin, (float)-p2, (float)(1.0 + p2), (float)q2);  // r_3 over b
        cycle_blocks(0, w, bin, fx[0]);
        k_blk_out<WT><<<nb, 256, 0, ctx->stream>>>(n, cols, total, w, bx1, bx2, fx[0],
                                                   (1.0 + p2 + p3 * p2) / th, (1.0 + p3) * q2, q3, di, perm, W, ldw);
    }
    LH_CHECK_LAUNCH();
}
template void Amg::apply_blocks<double>(double*, int, int, int, const int32_t*);
template void Amg::apply_blocks<float>(float*, int, int, int, const int32_t*);

}  // namespace lh

extern "C" int lh_cycle_apply(lh_ctx* ctx, lh_csr* A, const double* R, int nc, double* Z) {
    if (!ctx || !A || !R || !Z || nc < 1 || A->dtype != LH_F64) return LH_ERR_ARG;
    LH_API_BEGIN(ctx)
    HIPX(hipSetDevice(ctx->device));
    const int64_t n = A->n();
    lh::Amg amg;
    if (!amg.setup(ctx, n, A->nnz(), A->pat->rowptr.as<int32_t>(), A->pat->cols.as<int32_t>(), A->vals.as<double>(), 0,
                   nullptr, nullptr, lh::Amg::kShiftF64))
        LH_THROW(LH_ERR_NUMERIC, "lh_cycle_apply: no multigrid hierarchy for this matrix");
    amg.prepare(nc);
    const size_t bytes = (size_t)n * nc * 8;
    DevBuf r(bytes), z(bytes);
    lh::h2d(ctx, r.p, R, bytes);
    amg.apply(r.as<double>(), z.as<double>(), nullptr, nullptr);
    lh::d2h(ctx, Z, z.p, bytes);
    LH_API_END(ctx)
}
