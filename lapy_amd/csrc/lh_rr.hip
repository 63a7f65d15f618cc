// Rayleigh-Ritz eigensolver for an orthonormal trial basis: the smallest nev
// eigenpairs of a small dense symmetric H (N <= 192), FP64.
//
// Five kernels on the library stream, each bound by the latency of its
// dependent steps on one workgroup (or one wave per eigenpair):
//  1. k_rr_tri (one workgroup, 512 threads): H is held in registers, each
//     row spread over the 16 lanes of one DPP row, and reduced to
//     tridiagonal form by Householder reflections, two barriers per step.
//     The reflectors, the tridiagonal T and its Gershgorin bounds are parked
//     in global memory.
//  2. k_rr_bisect (one wave per wanted eigenvalue): multisection on T scaled
//     by a power of two to ||T|| <= 1, the 64 lanes evaluating Sturm counts
//     (sign changes of the leading minors) at 64 interior points (65-fold
//     bracket reduction per round).
//  3. k_rr_invit (one wave per eigenvalue; only the first of a group of
//     numerically equal eigenvalues works): inverse iteration with the LU
//     factors of T - lambda I (same scaling) in LDS, Gram-Schmidt inside the
//     group.
//  4. k_rr_back (one wave per eigenvector): Z := Q Y, the reflectors applied
//     in reverse order, two at a time, loaded eight pairs ahead into registers.
//  5. k_rr_polish (one workgroup): Newton-Schulz orthonormalisation of Z in
//     the small space, Z := Z (3 I - Z^T Z) / 2 (inverse iteration leaves
//     orthogonality errors ~ eps ||T|| / gap; each step squares them; up to
//     three steps, none for a basis with ||Z^T Z - I|| >= 1/2), its products
//     on the matrix cores from 32 columns up.
//
// Replaces the dense Rayleigh-Ritz step ARPACK performs inside eigsh
// (lapy/solver.py:713-715) for the block solver.
#include "lh_dense.hpp"

#include <cmath>

namespace lh {

namespace {

constexpr int NB = 1024;
constexpr int NMAX = kRRStdMaxN;
constexpr int PK = NMAX * (NMAX + 1) / 2;

__device__ __forceinline__ double wsum(double v) { return wave_sum64(v); }

__device__ __forceinline__ void stamp(unsigned long long* prof, int slot) {
    if (prof && threadIdx.x == 0 && blockIdx.x == 0) prof[slot] = wall_clock64();
}

// work layout (doubles): reflectors R[k][i] (N rows of NP = N rounded up to 32,
// entry i > k of reflector k in place), d (N), e (N), tau (N),
// bounds (4: lo, hi, ||T||, -), lam (nev), Y (nev x N, column g contiguous),
// Z (N x nev row-major)
__host__ __device__ constexpr int rr_stride(int N) { return (N + 31) / 32 * 32; }

struct RRWork {
    double *R, *d, *e, *tau, *bnd, *lam, *Y, *Z;
    __host__ __device__ RRWork(double* w, int N, int nev) {
        R = w;
        d = R + (size_t)N * rr_stride(N);
        e = d + N;
        tau = e + N;
        bnd = tau + N;
        lam = bnd + 4;
        Y = lam + nev;
        Z = Y + (size_t)N * nev;
    }
};

// number of eigenvalues of T below x: sign changes of the leading principal
// minors p_{i+1} = (d_i - x) p_i - e_{i-1}^2 p_{i-1}.  The caller scales T so
// that ||T|| <= 1 and raises e^2 to 1e-60 at least, so that a vanishing minor
// (which counts as positive) is followed by one of the sign that its
// predecessor's asks for; the pair is rescaled by a power of two every 8 steps,
// in which it changes by 1e-240 to 1e4 at most.  Three FP64 instructions and the
// sign's three a step; the quotient form q_i = (d_i - x) - e^2 / q_{i-1}, whose
// reciprocal alone is a chain of nine, took 89 us a call at N = 192 against
// 43 us.  N8: N rounded up to 8; d is padded with 2 there (no x is above 1).
__device__ int sturm(const double* d, const double* e2, int N8, double x) {
    int cnt = 0;
    double pm = 0.0, p = 1.0;
    for (int i0 = 0; i0 < N8; i0 += 8) {
        double dd[8], ee[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            dd[u] = d[i0 + u];
            ee[u] = e2[i0 + u];
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const double q = fma(dd[u] - x, p, -(ee[u] * pm));
            pm = p;
            p = q;
            cnt += (int)((unsigned)(__double2hiint(p) ^ __double2hiint(pm)) >> 31);
        }
        const int ex = ilogb(fmax(fabs(p), fabs(pm)));  // never both 0
        p = ldexp(p, -ex);
        pm = ldexp(pm, -ex);
    }
    return cnt;
}

// LU with partial pivoting of T - lam I into ws (1/u0, u1, u2, l, swapped: 5
// arrays of NMAX).  The caller scales T to ||T|| <= 1, so the pivots (a zero or
// sub-normal one replaced by tiny) have ordinary magnitudes and their
// reciprocals come from the short-latency form, stored for the solves.  Eight
// steps' entries of T are loaded ahead of their use, and branches are selects:
// a step is its reciprocal's dependent chain, without the LDS round trips that
// a load behind a store has to wait for.  d and e are readable to N + 8.
constexpr int TB = 8;
__device__ void tri_factor(const double* d, const double* e, int N, double lam, double tiny, double* ws) {
    double* iu0 = ws;
    double* u1 = ws + NMAX;
    double* u2 = ws + 2 * NMAX;
    double* lm = ws + 3 * NMAX;
    double* pv = ws + 4 * NMAX;
    double c0 = d[0] - lam, c1 = (N > 1) ? e[0] : 0.0;
    for (int i0 = 0; i0 < N - 1; i0 += TB) {
        double dn[TB], en[TB + 1];
#pragma unroll
        for (int u = 0; u < TB; ++u) dn[u] = d[i0 + u + 1] - lam;
#pragma unroll
        for (int u = 0; u <= TB; ++u) en[u] = (i0 + u < N - 1) ? e[i0 + u] : 0.0;
#pragma unroll
        for (int u = 0; u < TB; ++u) {
            const int i = i0 + u;
            if (i >= N - 1) break;
            const double sub = en[u], a1 = dn[u], b1 = en[u + 1];
            const bool sw = !(fabs(c0) >= fabs(sub) || !(fabs(sub) > 1e-300));
            const double piv = sw ? sub : (fabs(c0) > 1e-300) ? c0 : tiny;
            const double ip = rcp_nr(piv);
            const double l = (sw ? c0 : sub) * ip;
            const double x1 = sw ? a1 : c1, x2 = sw ? b1 : 0.0, y0 = sw ? c1 : a1, y1 = sw ? 0.0 : b1;
            iu0[i] = ip;
            u1[i] = x1;
            u2[i] = x2;
            lm[i] = l;
            pv[i] = sw ? 1.0 : 0.0;
            c0 = y0 - l * x1;
            c1 = y1 - l * x2;
        }
    }
    iu0[N - 1] = rcp_nr((fabs(c0) > tiny) ? c0 : tiny);
}

// solve with the factorisation; y overwritten, loads eight steps at a time as
// in the factorisation
__device__ void tri_lu_solve(const double* ws, int N, double* y) {
    const double* iu0 = ws;
    const double* u1 = ws + NMAX;
    const double* u2 = ws + 2 * NMAX;
    const double* lm = ws + 3 * NMAX;
    const double* pv = ws + 4 * NMAX;
    double a = y[0];
    for (int i0 = 0; i0 < N - 1; i0 += TB) {
        double b[TB], l[TB], s[TB];
#pragma unroll
        for (int u = 0; u < TB; ++u) {  // entries from N on are not used
            const int i = i0 + u < N - 1 ? i0 + u : N - 2;
            b[u] = y[i + 1];
            l[u] = lm[i];
            s[u] = pv[i];
        }
#pragma unroll
        for (int u = 0; u < TB; ++u) {
            const int i = i0 + u;
            if (i >= N - 1) break;
            const bool sw = s[u] != 0.0;
            const double hi = sw ? b[u] : a, lo = sw ? a : b[u];
            y[i] = hi;
            a = lo - l[u] * hi;
        }
    }
    double x1 = a * iu0[N - 1], x2 = 0.0;
    y[N - 1] = x1;
    for (int i0 = N - 2; i0 >= 0; i0 -= TB) {
        double r[TB], c1[TB], c2[TB], p[TB];
#pragma unroll
        for (int u = 0; u < TB; ++u) {
            const int i = i0 - u > 0 ? i0 - u : 0;
            r[u] = y[i];
            c1[u] = u1[i];
            c2[u] = u2[i];
            p[u] = iu0[i];
        }
#pragma unroll
        for (int u = 0; u < TB; ++u) {
            const int i = i0 - u;
            if (i < 0) break;
            const double x0 = (r[u] - c2[u] * x2 - c1[u] * x1) * p[u];
            y[i] = x0;
            x2 = x1;
            x1 = x0;
        }
    }
}

// ---- 1. tridiagonalisation ------------------------------------------------
// H lives in registers: 512 threads form 32 row groups of 16 lanes (one DPP
// row each), and the thread (group g, lane l) holds H[g + 32a][l + 16b] for
// a < CB, b < 2 CB (CB = ceil(N / 32)), a block-cyclic layout in which every
// row is spread over the 16 lanes of one group, so that row sums are DPP
// sums within a row; rows and columns from N on are zero and stay zero.  Step
// k (Householder reflector of row k = column k below the diagonal) costs two
// barriers:
//  A. the row's owner has left it in LDS (barrier 1); every group forms the
//     norm, alpha, v_0 and tau by itself, each lane keeping its columns of v;
//  B. every thread multiplies its block by v; row sums give p = tau H v for
//     the group's rows, which is published (barrier 2);
//  C. every thread forms K = tau (p . v) / 2 and w = p - K v, applies
//     H -= v w^T + w v^T to its block in registers, and the owner of row
//     k + 1 leaves it in LDS.
// The row and p are double-buffered by the parity of k, so step k + 1
// overwrites nothing that a thread still reads from step k.
// Step k belongs to phase A0 = (k + 1) / 32, in which the register rows below
// A0 and columns below 2 A0 are finished: the phases are compiled one by one,
// so that their loops run over what is left (42 % of the block on average),
// the next row is register row A0, and only the first two register columns
// and the first register row need comparisons with k.
// Bound by the dependent steps of a column (~2,000 cycles at small N, of which
// LDS and the barriers take ~500, four row sums ~430 and the reflector's scalars
// ~300) and, at N = 192, by the FP64 instructions of two waves a SIMD: 303 us a
// call at N = 192, 44 at 48.  Forming the reflector in its owner alone, with
// selects over all register rows and the store to global memory before the
// barrier, took ~4,000 cycles in which the other waves waited: 690 and 71 us.
constexpr int TRI_NT = 512;

template <int CB>
struct TriShared {
    double xbuf[2][32 * CB], pbuf[2][32 * CB];
    double sd[32 * CB], se[32 * CB], stau[32 * CB];
};

// steps k of phase A0, up to N - 3
template <int CB, int A0>
__device__ __forceinline__ void tri_phase(int N, double (&h)[CB][2 * CB], TriShared<CB>& S, double* __restrict__ R) {
    constexpr int RA = CB, CC = 2 * CB, B0 = 2 * A0, NP = 32 * CB;
    const int tid = threadIdx.x, g = tid >> 4, l = tid & 15;
    const int kend = (N - 2 < 32 * A0 + 31) ? N - 2 : 32 * A0 + 31;
    for (int k = (A0 == 0) ? 0 : 32 * A0 - 1; k < kend; ++k) {
        const int par = k & 1;
        // A. the reflector; k + 1 lies in register columns B0, B0 + 1
        double v[CC], vr[RA];
#pragma unroll
        for (int b = B0; b < CC; ++b) v[b] = S.xbuf[par][l + 16 * b];
        const double x0 = S.xbuf[par][k + 1];
#pragma unroll
        for (int a = A0; a < RA; ++a) vr[a] = S.xbuf[par][g + 32 * a];
        double s0 = 0.0, s1 = 0.0;
#pragma unroll
        for (int b = B0; b < CC; b += 2) {
            if (b == B0) {
                v[b] = (l + 16 * b <= k) ? 0.0 : v[b];
                v[b + 1] = (l + 16 * (b + 1) <= k) ? 0.0 : v[b + 1];
            }
            s0 += v[b] * v[b];
            s1 += v[b + 1] * v[b + 1];
        }
        const double xn2 = row_sum16(s0 + s1);
        double alpha = 0.0, v0 = 0.0, t = 0.0;
        if (xn2 != 0.0) {
            // the short-latency forms on the step's critical path (the
            // exact ones for extreme magnitudes; xn2 is the same in every
            // lane, so one branch runs)
            if (xn2 > 1e-280 && xn2 < 1e280) {
                const double sq = sqrt_nr(xn2);
                alpha = (x0 >= 0.0) ? -sq : sq;
                v0 = x0 - alpha;
                t = 2.0 * rcp_nr(xn2 - x0 * x0 + v0 * v0);
            } else {
                alpha = (x0 >= 0.0) ? -sqrt(xn2) : sqrt(xn2);
                v0 = x0 - alpha;
                t = 2.0 / (xn2 - x0 * x0 + v0 * v0);
            }
        }
#pragma unroll
        for (int b = B0; b < B0 + 2; ++b) v[b] = (l + 16 * b == k + 1) ? v0 : v[b];
        {
            const int i = g + 32 * A0;
            vr[A0] = (i <= k) ? 0.0 : (i == k + 1) ? v0 : vr[A0];
        }
        // B. p = tau H v for this group's rows
        double p[RA];
#pragma unroll
        for (int a = A0; a < RA; ++a) {
            double q0 = 0.0, q1 = 0.0;
#pragma unroll
            for (int b = B0; b < CC; b += 2) {
                q0 += h[a][b] * v[b];
                q1 += h[a][b + 1] * v[b + 1];
            }
            p[a] = q0 + q1;
        }
        row_sum16_each<A0>(p);
#pragma unroll
        for (int a = A0; a < RA; ++a) p[a] *= t;
        if (g + 32 * A0 <= k) p[A0] = 0.0;
        {
            double mine = p[A0];
#pragma unroll
            for (int a = A0 + 1; a < RA; ++a) mine = (l == a - A0) ? p[a] : mine;
            if (l < RA - A0) S.pbuf[par][g + 32 * (A0 + l)] = mine;
        }
        __syncthreads();
        // C. rank-2 update
        double w[CC];
        double k0 = 0.0, k1 = 0.0;
#pragma unroll
        for (int b = B0; b < CC; ++b) w[b] = S.pbuf[par][l + 16 * b];
#pragma unroll
        for (int b = B0; b < CC; b += 2) {
            k0 += w[b] * v[b];
            k1 += w[b + 1] * v[b + 1];
        }
        const double K = 0.5 * t * row_sum16(k0 + k1);
#pragma unroll
        for (int b = B0; b < CC; ++b) w[b] -= K * v[b];
#pragma unroll
        for (int a = A0; a < RA; ++a) {
            const double wr = p[a] - K * vr[a];
#pragma unroll
            for (int b = B0; b < CC; ++b) h[a][b] -= vr[a] * w[b] + wr * v[b];
        }
        if (g == ((k + 1) & 31)) {
#pragma unroll
            for (int b = B0; b < CC; ++b) S.xbuf[par ^ 1][l + 16 * b] = h[A0][b];
            if (l == ((k + 1) & 15)) S.sd[k + 1] = S.xbuf[par ^ 1][k + 1];  // this lane's own entry
        }
        if (g == ((k + 17) & 31)) {  // another wave: the reflector for the back-transformation
#pragma unroll
            for (int b = B0; b < CC; ++b) R[(int64_t)k * NP + l + 16 * b] = v[b];
            if (l == 0) {
                S.se[k] = alpha;
                S.stau[k] = t;
            }
        }
        __syncthreads();
    }
}

template <int CB>
__global__ void __launch_bounds__(TRI_NT)
k_rr_tri(int N, int nev, const double* __restrict__ G, int ldg, int sym, double* __restrict__ work,
         unsigned long long* __restrict__ prof) {
    constexpr int RA = CB, CC = 2 * CB;
    __shared__ TriShared<CB> S;
    RRWork W(work, N, nev);
    const int tid = threadIdx.x, g = tid >> 4, l = tid & 15;
    stamp(prof, 0);
    double h[RA][CC];
#pragma unroll
    for (int a = 0; a < RA; ++a) {
        const int i = g + 32 * a;
#pragma unroll
        for (int b = 0; b < CC; ++b) {
            const int j = l + 16 * b;
            const bool in = i < N && j < N;
            double x = in ? G[(int64_t)i * ldg + j] : 0.0;
            // the mirror image, read across the rows' cache lines, is the
            // same bits outside a Gram's diagonal tiles of 64
            if (in && (!sym || a / 2 == b / 4)) x = 0.5 * (x + G[(int64_t)j * ldg + i]);
            h[a][b] = x;
        }
    }
    stamp(prof, 1);
    if (g == 0) {  // row 0
#pragma unroll
        for (int b = 0; b < CC; ++b) S.xbuf[0][l + 16 * b] = h[0][b];
        if (l == 0) S.sd[0] = h[0][0];
    }
    __syncthreads();
    tri_phase<CB, 0>(N, h, S, W.R);
    if constexpr (CB > 1) tri_phase<CB, 1>(N, h, S, W.R);
    if constexpr (CB > 2) tri_phase<CB, 2>(N, h, S, W.R);
    if constexpr (CB > 3) tri_phase<CB, 3>(N, h, S, W.R);
    if constexpr (CB > 4) tri_phase<CB, 4>(N, h, S, W.R);
    if constexpr (CB > 5) tri_phase<CB, 5>(N, h, S, W.R);
    // the last 2 x 2 block (or the 1 x 1 matrix)
#pragma unroll
    for (int a = 0; a < RA; ++a) {
        const int i = g + 32 * a;
#pragma unroll
        for (int b = 0; b < CC; ++b) {
            const int j = l + 16 * b;
            if (N >= 2 && i == N - 1 && j == N - 2) S.se[N - 2] = h[a][b];
            if (i == N - 1 && j == N - 1) S.sd[N - 1] = h[a][b];
        }
    }
    if (tid == 0) {
        if (N >= 2) S.stau[N - 2] = 0.0;
        S.stau[N - 1] = 0.0;
        S.se[N - 1] = 0.0;
    }
    __syncthreads();
    for (int i = tid; i < N; i += TRI_NT) {
        W.d[i] = S.sd[i];
        W.e[i] = S.se[i];
        W.tau[i] = S.stau[i];
    }
    // Gershgorin bounds, by the first wave
    if (tid < 64) {
        double lo = S.sd[0], hi = S.sd[0], nrm = 0.0;
        for (int i = tid; i < N; i += 64) {
            const double rr = (i > 0 ? fabs(S.se[i - 1]) : 0.0) + (i < N - 1 ? fabs(S.se[i]) : 0.0);
            lo = fmin(lo, S.sd[i] - rr);
            hi = fmax(hi, S.sd[i] + rr);
            nrm = fmax(nrm, fabs(S.sd[i]) + rr);
        }
        for (int o = 32; o > 0; o >>= 1) {
            lo = fmin(lo, __shfl_xor(lo, o, 64));
            hi = fmax(hi, __shfl_xor(hi, o, 64));
            nrm = fmax(nrm, __shfl_xor(nrm, o, 64));
        }
        if (tid == 0) {
            W.bnd[0] = lo;
            W.bnd[1] = hi;
            W.bnd[2] = fmax(nrm, 1e-300);
        }
    }
    stamp(prof, 2);
}

// ---- 2. eigenvalues by multisection ----------------------------------------
__global__ void __launch_bounds__(64)
k_rr_bisect(int N, int nev, double* __restrict__ work, double* __restrict__ theta,
            unsigned long long* __restrict__ prof) {
    __shared__ double sd[NMAX], se2[NMAX];
    stamp(prof, 3);
    RRWork W(work, N, nev);
    const int j = blockIdx.x, q = threadIdx.x;
    const int N8 = (N + 7) & ~7;
    // T scaled by a power of two (exact) to ||T|| <= 1; se2[i] couples i - 1 and i
    const double sc = ldexp(1.0, -ilogb(W.bnd[2]) - 1);
    for (int i = q; i < N8; i += 64) {
        sd[i] = i < N ? W.d[i] * sc : 2.0;
        const double e = (i > 0 && i < N) ? W.e[i - 1] * sc : 0.0;
        se2[i] = fmax(e * e, 1e-60);
    }
    __syncthreads();
    const double glo = W.bnd[0] * sc, ghi = W.bnd[1] * sc, tnorm = W.bnd[2] * sc;
    double a = glo - 1e-14 * tnorm, b = ghi + 1e-14 * tnorm;
    for (int it = 0; it < 24; ++it) {
        const double h = (b - a) / 65.0;
        const double x = a + (q + 1) * h;
        const bool pred = sturm(sd, se2, N8, x) > j;
        const unsigned long long bal = __ballot(pred);
        const int first = bal ? (__ffsll((long long)bal) - 1) : 64;
        const double nb = (first < 64) ? a + (first + 1) * h : b;
        const double na = (first > 0) ? a + first * h : a;
        a = na;
        b = nb;
        if (b - a <= 2.2e-16 * (fabs(a) + fabs(b)) + 1e-17 * tnorm) break;
    }
    if (q == 0) {
        const double lam = 0.5 * (a + b) / sc;
        W.lam[j] = lam;
        theta[j] = lam;
    }
}

// ---- 3. eigenvectors of T by inverse iteration ------------------------------
// lane q owns the entries i = q, q + 64, q + 128 of every vector it touches
__device__ __forceinline__ double wave_dot3(const double* y, const double* z, int N) {
    double s = 0.0;
    for (int i = threadIdx.x; i < N; i += 64) s += y[i] * z[i];
    return wsum(s);
}

__global__ void __launch_bounds__(64)
k_rr_invit(int N, int nev, double* __restrict__ work) {
    __shared__ double sd[NMAX + TB], se[NMAX + TB], ws[5 * NMAX], y[NMAX];
    RRWork W(work, N, nev);
    const int j = blockIdx.x, q = threadIdx.x;
    const double tnorm = W.bnd[2];
    const double* lam = W.lam;
    const double scale_j = fmax(fabs(lam[j]), 1e-6 * tnorm);
    const bool leader = (j == 0) || (lam[j] - lam[j - 1] > 1e-7 * scale_j);
    if (!leader) return;  // whole wave
    int gend = j + 1;
    while (gend < nev && lam[gend] - lam[gend - 1] <= 1e-7 * fmax(fabs(lam[gend]), 1e-6 * tnorm)) ++gend;
    // T and the shifts scaled by a power of two (exact) to ||T|| <= 1: the
    // iterates grow like 1 / (eps ||T||) and their squared norms must stay
    // finite and normal whatever the magnitude of H
    const double sc = ldexp(1.0, -ilogb(tnorm) - 1);
    for (int i = q; i < N; i += 64) {
        sd[i] = W.d[i] * sc;
        se[i] = W.e[i] * sc;
    }
    const double tiny = 2.2e-16 * tnorm * sc;
    for (int g = j; g < gend; ++g) {
        for (int i = q; i < N; i += 64) y[i] = 1.0 + 0.1 * (double)((7 * i + 3 * g) % 11);
        __syncthreads();
        if (q == 0) tri_factor(sd, se, N, lam[g] * sc + (double)(g - j) * 8.0 * tiny, tiny, ws);
        for (int itr = 0; itr < 2; ++itr) {
            __syncthreads();
            if (q == 0) tri_lu_solve(ws, N, y);
            __syncthreads();
            // Gram-Schmidt against the group's earlier vectors (Y columns
            // written by this same lane mapping), then normalise
            for (int h = j; h < g; ++h) {
                const double* yh = W.Y + (int64_t)h * N;
                const double s = wave_dot3(y, yh, N);
                for (int i = q; i < N; i += 64) y[i] -= s * yh[i];
            }
            const double nn = 1.0 / sqrt(fmax(wave_dot3(y, y, N), 1e-300));
            for (int i = q; i < N; i += 64) y[i] *= nn;
        }
        for (int i = q; i < N; i += 64) W.Y[(int64_t)g * N + i] = y[i];
    }
}

// ---- 4. back-transformation Z = Q Y ----------------------------------------
// One wave per eigenvector (rows q, q + 64, q + 128 in lane q), one
// workgroup each, so the vectors spread over CUs.  The N - 2 reflectors are
// applied in dependent pairs: with s1 = t1 v1.z, the second one's s2 =
// t2 (v2.z - s1 v2.v1), and the three dot products of a pair run through the
// cross-lane stages together.  The entries are loaded BACK_PD pairs ahead into
// a register ring: they come from another XCD's L2, which takes ~1 us.  Bound by
// the dependent stages of the pairs: 39 us a call at N = 192 (76 us with one
// reflector at a time, four ahead, its loads behind branches).
constexpr int BACK_PD = 8;

__global__ void __launch_bounds__(64)
k_rr_back(int N, int nev, double* __restrict__ work, unsigned long long* __restrict__ prof) {
    __shared__ double tau[NMAX + 2];
    stamp(prof, 4);
    RRWork W(work, N, nev);
    const int g = blockIdx.x, q = threadIdx.x;
    for (int i = q; i < N; i += 64) tau[i + 1] = W.tau[i];
    if (q == 0) tau[0] = 0.0;  // "reflector -1": the partner of an odd last one
    const double* yg = W.Y + (int64_t)g * N;
    double z0 = (q < N) ? yg[q] : 0.0;
    double z1 = (q + 64 < N) ? yg[q + 64] : 0.0;
    double z2 = (q + 128 < N) ? yg[q + 128] : 0.0;
    // reflector k acts on rows k+1 .. N-1: loaded without a branch, from a
    // row and entry that exist, and masked when it is used
    const int NP = rr_stride(N);
    auto vload = [&](int k, int row) -> double {
        return W.R[(int64_t)(k > 0 ? k : 0) * NP + (row < NP ? row : NP - 1)];
    };
    auto masked = [&](double v, int k, int row) -> double { return (row > k && row < N) ? v : 0.0; };
    double ring[BACK_PD][6];
#pragma unroll
    for (int d = 0; d < BACK_PD; ++d) {
        const int k = N - 3 - 2 * d;
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            ring[d][c] = vload(k, q + 64 * c);
            ring[d][3 + c] = vload(k - 1, q + 64 * c);
        }
    }
    __syncthreads();  // tau staged
    for (int k0 = N - 3; k0 >= 0; k0 -= 2 * BACK_PD) {
#pragma unroll
        for (int d = 0; d < BACK_PD; ++d) {
            const int k = k0 - 2 * d;
            if (k < 0) break;
            double v[6];
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                v[c] = masked(ring[d][c], k, q + 64 * c);
                v[3 + c] = k > 0 ? masked(ring[d][3 + c], k - 1, q + 64 * c) : 0.0;
            }
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                ring[d][c] = vload(k - 2 * BACK_PD, q + 64 * c);
                ring[d][3 + c] = vload(k - 2 * BACK_PD - 1, q + 64 * c);
            }
            const double t1 = tau[k + 1], t2 = tau[k];
            double s[3] = {v[0] * z0 + v[1] * z1 + v[2] * z2, v[3] * z0 + v[4] * z1 + v[5] * z2,
                           v[3] * v[0] + v[4] * v[1] + v[5] * v[2]};
            wave_sum64_each(s);
            const double a1 = t1 * s[0];
            const double a2 = t2 * (s[1] - a1 * s[2]);
            z0 -= a1 * v[0] + a2 * v[3];
            z1 -= a1 * v[1] + a2 * v[4];
            z2 -= a1 * v[2] + a2 * v[5];
        }
    }
    if (q < N) W.Z[(int64_t)q * nev + g] = z0;
    if (q + 64 < N) W.Z[(int64_t)(q + 64) * nev + g] = z1;
    if (q + 128 < N) W.Z[(int64_t)(q + 128) * nev + g] = z2;
}

// ---- 5. orthonormalisation in the small space and output --------------------
typedef double d4_t __attribute__((ext_vector_type(4)));
// rows of Z and E in LDS when the products run on the matrix cores: two
// doubles longer than nev, against bank conflicts between rows, where that
// fits (N = nev = 96 does not)
__device__ __forceinline__ int pol_ld(int N, int nev) {
    return nev >= 32 && (N + nev) * (nev + 2) <= PK ? nev + 2 : nev;
}
// 16 x 16 tiles of Z a wave updates: 60 at most wherever Z and E fit into LDS
// (N = 192, nev = 65 .. 70 and N = 145 .. 147, nev = 81)
constexpr int kPolTiles = 4;
constexpr int pol_tiles_max() {
    int most = 0;
    for (int N = 1; N <= NMAX; ++N)
        for (int nev = 1; nev <= N; ++nev)
            if ((N + nev) * nev <= PK && (N + 15) / 16 * ((nev + 15) / 16) > most)
                most = (N + 15) / 16 * ((nev + 15) / 16);
    return most;
}
static_assert(pol_tiles_max() <= kPolTiles * (NB / 64), "a tile of Z without a wave");

__global__ void __launch_bounds__(NB)
k_rr_polish(int N, int nev, double* __restrict__ work, double* __restrict__ C, int* __restrict__ status,
            unsigned long long* __restrict__ prof) {
    __shared__ double Zs[PK];  // Z (N x nev), then E (nev x nev) behind it
    __shared__ double red[32];
    stamp(prof, 5);
    RRWork W(work, N, nev);
    const int tid = threadIdx.x;
    const int nz = N * nev, ld = pol_ld(N, nev);
    if ((N + nev) * ld <= PK) {
        double* E = Zs + N * ld;
        for (int idx = tid; idx < nz; idx += NB) Zs[(idx / nev) * ld + idx % nev] = W.Z[idx];
        __syncthreads();
        if (nev >= 32) {
            // both products on the matrix cores (v_mfma_f64_16x16x4f64, operands
            // from LDS): at N = 192, nev = 64 10 tiles of 48 instructions on the
            // 16 waves for E, then 48 of 16, three a wave, for the update.  In
            // 4 x 4 register tiles on the vector units the call took 53 us, now 28.
            const int lane = tid & 63, wv = tid >> 6, il = lane & 15, kg = lane >> 4;
            const int nt = (nev + 15) / 16, nr = (N + 15) / 16;
            const int ntri = nt * (nt + 1) / 2, nupd = nr * nt;
            for (int pass = 0; pass < 3; ++pass) {
                // E = Z^T Z - I: lower-triangle tiles, mirrored
                double emax = 0.0;
                for (int t = wv; t < ntri; t += NB / 64) {
                    int ta = 0, first = 0;
                    while (first + ta + 1 <= t) first += ++ta;
                    const int tb = t - first;
                    const int ca = 16 * ta + il, cb = 16 * tb + il;
                    const bool ina = ca < nev, inb = cb < nev;
                    const double* za = Zs + (ina ? ca : 0);
                    const double* zb = Zs + (inb ? cb : 0);
                    d4_t acc = {0.0, 0.0, 0.0, 0.0};
                    for (int i0 = 0; i0 < N; i0 += 4) {
                        const int i = i0 + kg;
                        const bool in = i < N;
                        const int o = (in ? i : 0) * ld;
                        const double x = za[o], y = zb[o];
                        acc = __builtin_amdgcn_mfma_f64_16x16x4f64(ina && in ? x : 0.0, inb && in ? y : 0.0, acc, 0,
                                                                   0, 0);
                    }
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const int i = 16 * ta + kg + 4 * r, j = cb;
                        if (i >= nev || j >= nev || j > i) continue;
                        const double ev = acc[r] - (i == j ? 1.0 : 0.0);
                        E[i * ld + j] = ev;
                        E[j * ld + i] = ev;
                        emax = fmax(emax, fabs(ev));
                    }
                }
                // block max of |E|
                for (int off = 32; off > 0; off >>= 1) emax = fmax(emax, __shfl_xor(emax, off, 64));
                __syncthreads();
                if ((tid & 63) == 0) red[tid >> 6] = emax;
                __syncthreads();
                double em = 0.0;
#pragma unroll
                for (int w = 0; w < NB / 64; ++w) em = fmax(em, red[w]);
                // Newton-Schulz needs ||E|| < 1; a basis that far off is left as it is
                if (em >= 0.5 || (pass > 0 && em <= 1e-8)) break;
                // Z <- Z - Z E / 2: up to kPolTiles 16 x 16 tiles a wave, written
                // after a barrier once every tile has been read
                d4_t acc[kPolTiles];
#pragma unroll
                for (int u = 0; u < kPolTiles; ++u) {
                    acc[u] = (d4_t){0.0, 0.0, 0.0, 0.0};
                    const int t = wv + (NB / 64) * u;
                    if (t >= nupd) continue;
                    const int row = 16 * (t / nt) + il, col = 16 * (t % nt) + il;
                    const bool inr = row < N, inc = col < nev;
                    const double* zr = Zs + (inr ? row : 0) * ld;
                    for (int k0 = 0; k0 < nev; k0 += 4) {
                        const int k = k0 + kg;
                        const bool in = k < nev;
                        const double x = zr[in ? k : 0], y = E[(in ? k : 0) * ld + (inc ? col : 0)];
                        acc[u] = __builtin_amdgcn_mfma_f64_16x16x4f64(inr && in ? x : 0.0, inc && in ? y : 0.0, acc[u],
                                                                      0, 0, 0);
                    }
                }
                __syncthreads();
#pragma unroll
                for (int u = 0; u < kPolTiles; ++u) {
                    const int t = wv + (NB / 64) * u;
                    if (t >= nupd) continue;
                    const int col = 16 * (t % nt) + il;
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const int row = 16 * (t / nt) + kg + 4 * r;
                        if (row < N && col < nev) Zs[row * ld + col] -= 0.5 * acc[u][r];
                    }
                }
                __syncthreads();
                if (em <= 1e-8) break;  // one step leaves ~ em^2: rounding level
            }
        } else {
            // few columns: one output per thread keeps more threads busy
            for (int pass = 0; pass < 3; ++pass) {
                // E = Z^T Z - I (symmetric: lower entries computed, mirrored)
                double emax = 0.0;
                for (int idx = tid; idx < nev * nev; idx += NB) {
                    const int a = idx / nev, b = idx - a * nev;
                    if (b > a) continue;
                    double s0 = 0.0, s1 = 0.0;
                    int i = 0;
                    for (; i + 1 < N; i += 2) {
                        s0 += Zs[i * nev + a] * Zs[i * nev + b];
                        s1 += Zs[(i + 1) * nev + a] * Zs[(i + 1) * nev + b];
                    }
                    if (i < N) s0 += Zs[i * nev + a] * Zs[i * nev + b];
                    const double ev = (s0 + s1) - (a == b ? 1.0 : 0.0);
                    E[a * nev + b] = ev;
                    E[b * nev + a] = ev;
                    emax = fmax(emax, fabs(ev));
                }
                // block max of |E|
                for (int off = 32; off > 0; off >>= 1) emax = fmax(emax, __shfl_xor(emax, off, 64));
                __syncthreads();
                if ((tid & 63) == 0) red[tid >> 6] = emax;
                __syncthreads();
                double em = 0.0;
    #pragma unroll
                for (int w = 0; w < NB / 64; ++w) em = fmax(em, red[w]);
                // Newton-Schulz needs ||E|| < 1; a basis that far off is left as it is
                if (em >= 0.5 || (pass > 0 && em <= 1e-8)) break;
                // Z <- Z - Z E / 2 ; each thread owns entries idx = tid + NB * u
                constexpr int U = (PK + NB - 1) / NB;
                double nz_[U];
    #pragma unroll
                for (int u = 0; u < U; ++u) {
                    const int idx = tid + NB * u;
                    nz_[u] = 0.0;
                    if (idx < nz) {
                        const int i = idx / nev, c = idx - i * nev;
                        double s = 0.0;
                        for (int h = 0; h < nev; ++h) s += Zs[i * nev + h] * E[h * nev + c];
                        nz_[u] = Zs[idx] - 0.5 * s;
                    }
                }
                __syncthreads();
    #pragma unroll
                for (int u = 0; u < U; ++u) {
                    const int idx = tid + NB * u;
                    if (idx < nz) Zs[idx] = nz_[u];
                }
                __syncthreads();
                if (em <= 1e-8) break;  // one step leaves ~ em^2: rounding level
            }
        }
        for (int idx = tid; idx < nz; idx += NB) C[idx] = Zs[(idx / nev) * ld + idx % nev];
    } else {
        for (int idx = tid; idx < nz; idx += NB) C[idx] = W.Z[idx];
    }
    if (tid == 0) status[0] = 0;
    stamp(prof, 6);
}

}  // namespace

size_t rr_std_work_doubles(int N, int nev) { return (size_t)N * rr_stride(N) + 3 * (size_t)N + 4 + nev + 2 * (size_t)N * nev + 64; }

void rr_std(lh_ctx* ctx, int N, int nev, const double* G, int ldg, double* C, double* theta, double* work,
            int* status, unsigned long long* prof, bool mirrored) {
    const int sym = mirrored ? 1 : 0;
    if (N > kRRStdMaxN || nev > N || N < 1 || nev < 1)
        LH_THROW(LH_ERR_ARG, "rr_std: N=%d nev=%d out of range", N, nev);
    switch ((N + 31) / 32) {
        case 1: k_rr_tri<1><<<1, TRI_NT, 0, ctx->stream>>>(N, nev, G, ldg, sym, work, prof); break;
        case 2: k_rr_tri<2><<<1, TRI_NT, 0, ctx->stream>>>(N, nev, G, ldg, sym, work, prof); break;
        case 3: k_rr_tri<3><<<1, TRI_NT, 0, ctx->stream>>>(N, nev, G, ldg, sym, work, prof); break;
        case 4: k_rr_tri<4><<<1, TRI_NT, 0, ctx->stream>>>(N, nev, G, ldg, sym, work, prof); break;
        case 5: k_rr_tri<5><<<1, TRI_NT, 0, ctx->stream>>>(N, nev, G, ldg, sym, work, prof); break;
        default: k_rr_tri<6><<<1, TRI_NT, 0, ctx->stream>>>(N, nev, G, ldg, sym, work, prof); break;
    }
    LH_CHECK_LAUNCH();
    k_rr_bisect<<<nev, 64, 0, ctx->stream>>>(N, nev, work, theta, prof);
    LH_CHECK_LAUNCH();
    k_rr_invit<<<nev, 64, 0, ctx->stream>>>(N, nev, work);
    LH_CHECK_LAUNCH();
    k_rr_back<<<nev, 64, 0, ctx->stream>>>(N, nev, work, prof);
    LH_CHECK_LAUNCH();
    k_rr_polish<<<1, NB, 0, ctx->stream>>>(N, nev, work, C, status, prof);
    LH_CHECK_LAUNCH();
}

}  // namespace lh

using namespace lh;

extern "C" int lh_small_symeig(lh_ctx* ctx, int N, int nev, const double* H, double* evals, double* Z,
                               double* phase_us) {
    if (!ctx || !H || N < 1 || nev < 1 || nev > N || N > kRRStdMaxN) return LH_ERR_ARG;
    LH_API_BEGIN(ctx)
    HIPX(hipSetDevice(ctx->device));
    DevBuf dH((size_t)N * N * 8), dC((size_t)N * nev * 8), dth((size_t)nev * 8),
        work(rr_std_work_doubles(N, nev) * 8), st(64), prof(8 * 8);
    h2d(ctx, dH.p, H, (size_t)N * N * 8);
    HIPX(hipMemsetAsync(prof.p, 0, 64, ctx->stream));
    rr_std(ctx, N, nev, dH.as<double>(), N, dC.as<double>(), dth.as<double>(), work.as<double>(), st.as<int>(),
           phase_us ? prof.as<unsigned long long>() : nullptr);
    if (evals) d2h(ctx, evals, dth.p, (size_t)nev * 8);
    if (Z) d2h(ctx, Z, dC.p, (size_t)N * nev * 8);  // row-major N x nev
    if (phase_us) {
        // stamps: tri start, after load, tri end, bisect start, back start,
        // polish start, polish end (kernel starts on the in-order stream)
        unsigned long long p[8];
        d2h(ctx, p, prof.p, sizeof(p));
        int khz = 100000;
        (void)hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, ctx->device);
        for (int i = 0; i < 6; ++i) phase_us[i] = (double)(p[i + 1] - p[i]) * 1000.0 / (double)khz;
        phase_us[6] = 0.0;
    }
    HIPX(hipStreamSynchronize(ctx->stream));
    LH_API_END(ctx)
}
