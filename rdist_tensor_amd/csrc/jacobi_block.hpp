// Cyclic Jacobi eigensolver and the Jacobi pseudo-inverse of an R x R
// symmetric matrix on one workgroup of kJacobiThreads threads, shared by the dense
// kernels and the FP64 batched sweep.
#pragma once
#include "common.hpp"

namespace exafac {
namespace {

// ---------------------------------------------------------------- Jacobi
// The round-robin ("circle method") schedule over ne = 2 npair (even) indices:
// index 0 keeps position 0, the others move one position down a round, and pair
// i is positions i and ne - 1 - i.  rr_index: the index at position pos (m = ne
// - 1), which is pos itself in round 0.  rr_next: where it is a round later.
__device__ __forceinline__ int rr_index(int m, int round, int pos) {
    const int v = pos + round;
    return pos == 0 ? 0 : (v > m ? v - m : v);
}
__device__ __forceinline__ int rr_next(int m, int pos) { return pos == 0 ? 0 : (pos == 1 ? m : pos - 1); }

// Place of the element of positions a and b in the block layout: the 2 x 2
// blocks of two pairs P < Q by side of P, side of Q and block, then the pairs'
// own elements (first, cross, second).
__device__ __forceinline__ int rr_place(int npair, int a, int b) {
    const int noff = npair * (npair - 1) / 2;
    const int sa = a >= npair ? 1 : 0, sb = b >= npair ? 1 : 0;
    const int pa = sa ? 2 * npair - 1 - a : a, pb = sb ? 2 * npair - 1 - b : b;
    if (pa == pb) return 4 * noff + (sa + sb) * npair + pa;
    const int P = pa < pb ? pa : pb, Q = pa < pb ? pb : pa, sP = pa < pb ? sa : sb, sQ = pa < pb ? sb : sa;
    return (2 * sP + sQ) * noff + P * (2 * npair - P - 1) / 2 + Q - P - 1;
}

struct JacobiShared {
    int rank[kMaxRank];
    int conv[2];   // per sweep (alternating): whether any pair rotated
};

__device__ __forceinline__ int sym_index(int R, int a, int b) {
    return a <= b ? tri_index(R, a, b) : tri_index(R, b, a);
}

// Jacobi runs on one workgroup of kJacobiThreads threads (one wavefront per
// SIMD: the solver is bound by dependent FP64 latency, not by issue).
constexpr int kJacobiThreads = 256;

// Rotation of a pair from its entries of the pre-round matrix, f and g its
// first and second position: c > 0, s = t c when it rotates; c = -1 when it does
// not (|a_fg| at most eps sqrt(|a_ff a_gg|), or one is the padding index of an
// odd order).  The oracle rotates (p, q) with p < q; `swap` says that f is q,
// where the same rotation seen from (f, g) has s and t of the other sign.
struct JacobiRot {
    double c, s, t;
};

__device__ __forceinline__ JacobiRot jacobi_rot(double aff, double agg, double afg, bool valid, bool swap) {
#pragma clang fp contract(off)
    JacobiRot r{-1.0, 0.0, 0.0};
    const double thr = 2.220446049250313e-16 * sqrt(fabs(aff) * fabs(agg));
    if (valid && afg != 0.0 && fabs(afg) > thr) {
        const double tau_fg = (agg - aff) / (2.0 * afg);
        const double tau = swap ? -tau_fg : tau_fg;
        const double rt = sqrt(1.0 + tau * tau);
        const double u = 1.0 / (fabs(tau) + rt);
        const double t = tau >= 0.0 ? u : -u;
        const double c = 1.0 / sqrt(1.0 + t * t);
        const double s = t * c;
        r.c = c;
        r.s = swap ? -s : s;
        r.t = swap ? -t : t;
    }
    return r;
}

// Row i of the 2x2 product J^T w (J the rotation c, s of a pair; w0, w1
// the pair's first and second entries), as written out: c w0 - s w1 for i = 0, s w0 +
// c w1 for i = 1, w_i unchanged without rotation.  (c w0 - s w1 = c w0 +
// (-s) w1 exactly, so both rows are one product-sum with chosen factors.)
__device__ __forceinline__ double rot_row(bool rot, double c, double s, int i, double w0, double w1) {
#pragma clang fp contract(off)
    const double m0 = i == 0 ? c : s, m1 = i == 0 ? -s : c;
    return rot ? m0 * w0 + m1 * w1 : (i == 0 ? w0 : w1);
}

// Cyclic Jacobi on the packed upper triangle A (LDS) with eigenvectors V
// (LDS, R x R row-major, room for R x (R rounded up to even)); A2 (LDS) is the
// second buffer of the matrix; both have room for the triangle of the even
// order.  The same arithmetic as the oracle's orc_eigh, bit for bit: rotation
// parameters from the pre-round matrix, each upper element rotated
// rows-then-columns, the exact 2x2 diagonal, upper triangle authoritative.
//
// One barrier per round, and a round is one chain of dependent FP64 and LDS
// operations on each wavefront, so its time is the instructions of one
// wavefront.  The matrix and V are therefore held by schedule position and not
// by index: a thread owns fixed 2 x 2 blocks of two pairs (or whole pairs, or rows
// of V), reads them from fixed places and writes the result to the places of the
// next round, and no index arithmetic is left in a round but the order of the
// indices, which the element's order of rotations depends on.  Lane l of each
// wavefront computes the rotation of pair l % npair itself; a block takes its
// two by shuffles.  Both rotation orders of an element are formed and its own
// one chosen, so that the wavefront does not diverge.  Up to order 32 the
// wavefronts that have no blocks rotate V, the last one also the pairs' own
// elements; above, every wavefront does both.  The convergence flag of each
// sweep is published by thread 0 in LDS.  Afterwards A holds the result and
// sh.rank[v] is the ascending position of A[v][v] (ties by index).
// By index, with packed-triangle indices computed in each round and every
// wavefront doing blocks and rows: 146 / 344 / 2358 us for an eigendecomposition
// of order 16 / 32 / 64 (a random Gram with a repeated column); so: 102 / 234 / 971.
template <int RM>
__device__ __forceinline__ void jacobi_block(double* A, double* A2, double* V, int R, JacobiShared& sh) {
#pragma clang fp contract(off)
    static_assert(RM % 2 == 0 && RM <= 64, "the buffers hold the even order; the pairs fit half a wavefront");
    constexpr int kWaves = kJacobiThreads / 64;
    constexpr bool kSplit = RM <= 32;            // at most 120 blocks: two wavefronts
    constexpr int NBL = kSplit ? 1 : 2;          // 496 blocks at most
    constexpr int NV = kSplit ? 4 : 8;           // rows of V a lane slot rotates
    const int tid = threadIdx.x, lane = tid % 64, wave = tid / 64;
    const int n = R, ne = n + (n & 1), npair = ne / 2, m = ne - 1;
    const int noff = npair * (npair - 1) / 2, diag = 4 * noff;
    const int bwaves = kSplit ? (noff + 63) / 64 : kWaves;
    const bool has_blocks = wave < bwaves;
    const bool has_diag = wave == kWaves - 1 && lane < npair;
    // blocks: positions (P, ne-1-P) x (Q, ne-1-Q), and where each element goes
    int bP[NBL], bQ[NBL], bi[NBL], to[NBL][4];
#pragma unroll
    for (int b = 0; b < NBL; b++) {
        const int id = tid + b * kJacobiThreads;
        bi[b] = has_blocks && id < noff ? id : -1;
        int P = 0, rest = bi[b] < 0 ? 0 : id;
        while (P + 1 < npair && rest >= npair - 1 - P) { rest -= npair - 1 - P; P++; }
        bP[b] = P;
        bQ[b] = P + 1 + rest < npair ? P + 1 + rest : P;   // npair == 1 has no block
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const int ra = (u >> 1) ? m - bP[b] : bP[b], cb = (u & 1) ? m - bQ[b] : bQ[b];
            to[b][u] = rr_place(npair, rr_next(m, ra), rr_next(m, cb));
        }
    }
    const int pair = lane % npair, fpos = pair, gpos = m - pair;
    const int fnext = rr_next(m, fpos), gnext = rr_next(m, gpos);
    const int toff = rr_place(npair, fnext, fnext), tofg = rr_place(npair, fnext, gnext),
              togg = rr_place(npair, gnext, gnext);
    // rows of V: lane slots of npair lanes on the wavefronts that rotate V
    const int vslots = 64 / npair, vwaves = kSplit ? kWaves - bwaves : kWaves, vwave = kSplit ? wave - bwaves : wave;
    const int vstride = vwaves * vslots;
    const bool has_v = vwave >= 0;
    const int vrow = has_v && lane < vslots * npair ? vwave * vslots + lane / npair : n;
    // into the layout of round 0, where the index at a position is the position
    for (int e = tid; e < ne * ne; e += kJacobiThreads) {
        const int a = e / ne, b = e - a * ne;
        if (a <= b) A2[rr_place(npair, a, b)] = b < n ? A[tri_index(R, a, b)] : 0.0;
        if (a < n) V[e] = a == b ? 1.0 : 0.0;
    }
    __syncthreads();
    double* cur = A2;
    double* nxt = A;
    bool any = false;
    int sweep = 0, round = 0;
    for (;;) {
        // every read of the round first
        const double aff = cur[diag + pair], afg = cur[diag + npair + pair], agg = cur[diag + 2 * npair + pair];
        double x[NBL][2][2];
#pragma unroll
        for (int b = 0; b < NBL; b++)
#pragma unroll
            for (int u = 0; u < 4; u++) x[b][u >> 1][u & 1] = has_blocks ? cur[u * noff + (bi[b] < 0 ? 0 : bi[b])] : 0.0;
        double vf[NV], vg[NV];
#pragma unroll
        for (int u = 0; u < NV; u++) {
            const int kk = vrow + vstride * u < n ? vrow + vstride * u : 0;   // (row 0: not used)
            vf[u] = has_v ? V[kk * ne + fpos] : 0.0;
            vg[u] = has_v ? V[kk * ne + gpos] : 0.0;
        }
        const int fi = rr_index(m, round, fpos), gi = rr_index(m, round, gpos);
        const JacobiRot mine = jacobi_rot(aff, agg, afg, fi < n && gi < n, fi > gi);
        const bool rot = mine.c > 0.0;
        const bool rotates = __ballot(rot) != 0;   // the same on every wavefront
        any |= rotates;
        if (has_blocks) {
#pragma unroll
            for (int b = 0; b < NBL; b++) {
                double off[2][2];
#pragma unroll
                for (int u = 0; u < 4; u++) off[u >> 1][u & 1] = x[b][u >> 1][u & 1];
                if (rotates) {
                    const int P = bP[b], Q = bQ[b];
                    const double cP = __shfl(mine.c, P, 64), sP = __shfl(mine.s, P, 64);
                    const double cQ = __shfl(mine.c, Q, 64), sQ = __shfl(mine.s, Q, 64);
                    const bool rP = cP > 0.0, rQ = cQ > 0.0;
                    // fa: rows by P's rotation, then columns by Q's (P's index
                    // the smaller); fb: rows by Q's, then columns by P's
                    double ra_[2][2], fa[2][2], rb_[2][2], fb[2][2];
#pragma unroll
                    for (int k = 0; k < 2; k++) {
                        ra_[0][k] = rot_row(rP, cP, sP, 0, x[b][0][k], x[b][1][k]);
                        ra_[1][k] = rot_row(rP, cP, sP, 1, x[b][0][k], x[b][1][k]);
                        rb_[0][k] = rot_row(rQ, cQ, sQ, 0, x[b][k][0], x[b][k][1]);
                        rb_[1][k] = rot_row(rQ, cQ, sQ, 1, x[b][k][0], x[b][k][1]);
                    }
#pragma unroll
                    for (int i = 0; i < 2; i++) {
                        fa[i][0] = rot_row(rQ, cQ, sQ, 0, ra_[i][0], ra_[i][1]);
                        fa[i][1] = rot_row(rQ, cQ, sQ, 1, ra_[i][0], ra_[i][1]);
                        fb[i][0] = rot_row(rP, cP, sP, 0, rb_[i][0], rb_[i][1]);
                        fb[i][1] = rot_row(rP, cP, sP, 1, rb_[i][0], rb_[i][1]);
                    }
                    const int ri[2] = {rr_index(m, round, P), rr_index(m, round, m - P)};
                    const int ci[2] = {rr_index(m, round, Q), rr_index(m, round, m - Q)};
#pragma unroll
                    for (int u = 0; u < 4; u++) {
                        const int i = u >> 1, k = u & 1;
                        off[i][k] = ri[i] < ci[k] ? fa[i][k] : fb[k][i];
                    }
                }
                if (bi[b] >= 0)
#pragma unroll
                    for (int u = 0; u < 4; u++) nxt[to[b][u]] = off[u >> 1][u & 1];
            }
        }
        if (has_diag) {   // the exact 2x2 result
            nxt[toff] = rot ? aff - mine.t * afg : aff;
            nxt[togg] = rot ? agg + mine.t * afg : agg;
            nxt[tofg] = rot ? 0.0 : afg;
        }
        if (has_v) {
            // a row's lanes are in one wavefront: every read of it is above
#pragma unroll
            for (int u = 0; u < NV; u++) {
                const int kk = vrow + vstride * u;
                if (kk < n) {
                    V[kk * ne + fnext] = rot ? mine.c * vf[u] - mine.s * vg[u] : vf[u];
                    V[kk * ne + gnext] = rot ? mine.s * vf[u] + mine.c * vg[u] : vg[u];
                }
            }
        }
        const bool last = round + 1 == m;
        if (last && tid == 0) sh.conv[sweep & 1] = any ? 1 : 0;
        __syncthreads();
        double* tmp = cur;
        cur = nxt;
        nxt = tmp;
        round = last ? 0 : round + 1;
        if (last) {
            // every thread reads the same flag: the exit is uniform
            const int rotated = sh.conv[sweep & 1];
            any = false;
            if (!rotated || ++sweep == 40) break;
        }
    }
    // back to packed A and row stride R (a whole number of rounds: by index again)
    constexpr int kHold = RM * RM / kJacobiThreads;
    double ha[kHold], hv[kHold];
#pragma unroll
    for (int q = 0; q < kHold; q++) {
        const int e = tid + q * kJacobiThreads;
        if (e >= n * n) continue;
        const int a = e / n, b = e - a * n;
        ha[q] = cur[rr_place(npair, a, b)];
        hv[q] = V[a * ne + b];
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < kHold; q++) {
        const int e = tid + q * kJacobiThreads;
        if (e >= n * n) continue;
        const int a = e / n, b = e - a * n;
        if (a <= b) A[tri_index(R, a, b)] = ha[q];
        V[e] = hv[q];
    }
    __syncthreads();
    if (tid < n) {
        const double lv = A[tri_index(R, tid, tid)];
        int rk = 0;
        for (int u = 0; u < n; u++) {
            const double lu = A[tri_index(R, u, u)];
            if (lu < lv || (lu == lv && u < tid)) rk++;
        }
        sh.rank[tid] = rk;
    }
    __syncthreads();
}

// Load an R x R matrix's upper triangle (row-major source) into packed LDS.
__device__ __forceinline__ void load_upper(const double* M, int R, double* A) {
    for (int o = threadIdx.x; o < R * R; o += blockDim.x) {
        const int a = o / R, b = o - a * R;
        if (a <= b) A[tri_index(R, a, b)] = M[o];
    }
    __syncthreads();
}

template <int RM>
struct EighSharedT {
    double A[RM * (RM + 1) / 2];
    double A2[RM * (RM + 1) / 2];
    double V[RM * RM];
    JacobiShared j;
};

// compute_pinv_square: W = V diag(1/sqrt(lam)) for lam > tol else 0, in place of
// V; out = W W^T summed over ascending eigenvalues.
template <class SH>
__device__ __forceinline__ void pinv_from_jacobi(SH& sh, int R, double tol, double* __restrict__ out) {
#pragma clang fp contract(off)
    __shared__ int ord[kMaxRank];
    if (threadIdx.x < R) ord[sh.j.rank[threadIdx.x]] = threadIdx.x;
    for (int o = threadIdx.x; o < R * R; o += blockDim.x) {
        const int v = o % R;
        const double lv = sh.A[tri_index(R, v, v)];
        const double sq = lv > tol ? sqrt(lv) : 0.0;
        sh.V[o] = sq > 0.0 ? sh.V[o] / sq : 0.0;
    }
    __syncthreads();
    for (int o = threadIdx.x; o < R * R; o += blockDim.x) {
        int a = o / R, b = o % R;
        if (a > b) continue;
        double acc = 0.0;
        for (int cc = 0; cc < R; cc++) {
            const int v = ord[cc];
            acc += sh.V[a * R + v] * sh.V[b * R + v];
        }
        out[a * R + b] = acc;
        out[b * R + a] = acc;
    }
}

}  // namespace
}  // namespace exafac
