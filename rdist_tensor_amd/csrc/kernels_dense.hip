// Dense R x R and tall-skinny kernels (FP64): Gram, Jacobi eigensolver,
// pseudo-inverse, DAGAT, dsymm, column renormalisation.
//
// Reference semantics: common.h:363-443 (compute_gram, compute_pinv_square),
// common.h:696-746 (parallel_dsymm, compute_DAGAT), distmat.hpp:85-151.
#include "common.hpp"
#include "jacobi_block.hpp"
#include "wave_psd.hpp"
#include "device.hpp"
#include "dsymm.hpp"

namespace exafac {
namespace {

constexpr int kThreads = 256;

// ---------------------------------------------------------------- Gram
// Stage 2: G[a][b] = sum over the partials (upper triangle), one wavefront per
// output entry: lane l sums partials l, l+64, ... in order, then a fixed
// butterfly combines the lanes.  Lower triangle mirrored.
__global__ __launch_bounds__(kThreads) void gram_final(const double* __restrict__ part, int nparts, int R,
                                                       double* __restrict__ G) {
    const int lane = threadIdx.x % 64;
    const int R2 = R * R;
    const int o = blockIdx.x * (kThreads / 64) + threadIdx.x / 64;
    if (o >= R2) return;
    const int a = o / R, b = o % R;
    const int src = (a < b ? a : b) * R + (a < b ? b : a);
    double s = 0.0;
    for (int p = lane; p < nparts; p += 64) s += part[(int64_t)p * R2 + src];
    s = wave_sum(s);
    if (lane == 0) G[o] = s;
}

// ---------------------------------------------------------------- Gram (FP64 MFMA)
// Block partials of A^T A on v_mfma_f64_16x16x4f64 (FP64 products and sums;
// TA = double, or float converted exactly).  Operand layout: lane l holds
// X[r0 + l/16][16 t + l%16] for column tile t, which is both the A operand of
// tile (t, .) and the B operand of tile (., t); the accumulator holds
// C[4 i + l/16][l%16], i < 4.  Each wavefront takes 16-row chunks w, w+4, ...
// of the block's rows (four k-steps of 4 rows); the four wavefronts' tiles
// are added in wave order in LDS and the block writes its upper triangle.
typedef double f64x4 __attribute__((ext_vector_type(4)));

template <typename TA, int NT>
__global__ __launch_bounds__(kThreads) void gram_mfma64_partial(const TA* __restrict__ A, int64_t mb,
                                                                const uint64_t* __restrict__ m_dev, int R,
                                                                double* __restrict__ part) {
    const int64_t m = m_dev ? ((int64_t)*m_dev < mb ? (int64_t)*m_dev : mb) : mb;
    __shared__ double red[kMaxRank * kMaxRank];
    const int lane = threadIdx.x % 64, wave = threadIdx.x / 64;
    const int kr = lane / 16, kc = lane % 16;
    f64x4 acc[NT][NT];
#pragma unroll
    for (int ta = 0; ta < NT; ta++)
#pragma unroll
        for (int tb = 0; tb < NT; tb++) acc[ta][tb] = f64x4{0.0, 0.0, 0.0, 0.0};
    const int64_t nchunks = (m + 15) / 16;
    for (int64_t ch = (int64_t)blockIdx.x * 4 + wave; ch < nchunks; ch += (int64_t)gridDim.x * 4) {
        // unconditional loads (element 0 in place of a missing one, then
        // zeroed), all in flight together
        TA y[4][NT];
#pragma unroll
        for (int st = 0; st < 4; st++) {
            const int64_t r = ch * 16 + 4 * st + kr;
#pragma unroll
            for (int t = 0; t < NT; t++) {
                const int c = 16 * t + kc;
                y[st][t] = A[(r < m && c < R) ? r * R + c : 0];
            }
        }
        double x[4][NT];
#pragma unroll
        for (int st = 0; st < 4; st++) {
            const int64_t r = ch * 16 + 4 * st + kr;
#pragma unroll
            for (int t = 0; t < NT; t++) x[st][t] = (r < m && 16 * t + kc < R) ? (double)y[st][t] : 0.0;
        }
#pragma unroll
        for (int st = 0; st < 4; st++)
#pragma unroll
            for (int ta = 0; ta < NT; ta++)
#pragma unroll
                for (int tb = ta; tb < NT; tb++)
                    acc[ta][tb] = __builtin_amdgcn_mfma_f64_16x16x4f64(x[st][ta], x[st][tb], acc[ta][tb], 0, 0, 0);
    }
    for (int w = 0; w < 4; w++) {
        if (wave == w) {
#pragma unroll
            for (int ta = 0; ta < NT; ta++)
#pragma unroll
                for (int tb = ta; tb < NT; tb++)
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        const int a = 16 * ta + 4 * i + kr, b = 16 * tb + kc;
                        if (a < R && b < R) red[a * R + b] = w == 0 ? acc[ta][tb][i] : red[a * R + b] + acc[ta][tb][i];
                    }
        }
        __syncthreads();
    }
    for (int o = threadIdx.x; o < R * R; o += kThreads) {
        const int a = o / R, b = o % R;
        if (a <= b) part[(int64_t)blockIdx.x * R * R + o] = red[o];
    }
}

// Eigendecomposition of blockIdx.x-th matrix: lam ascending, V columns.
template <int NMAX>
__global__ __launch_bounds__(kJacobiThreads) void eigh_kernel(const double* __restrict__ Min, int R,
                                                        double* __restrict__ lam, double* __restrict__ Vout) {
    __shared__ EighSharedT<NMAX> sh;
    const int64_t R2 = (int64_t)R * R;
    load_upper(Min + blockIdx.x * R2, R, sh.A);
    jacobi_block<NMAX>(sh.A, sh.A2, sh.V, R, sh.j);
    for (int o = threadIdx.x; o < R * R; o += blockDim.x) {
        int u = o / R, v = o % R;
        Vout[blockIdx.x * R2 + u * R + sh.j.rank[v]] = sh.V[u * R + v];
    }
    if (threadIdx.x < R) lam[blockIdx.x * R + sh.j.rank[threadIdx.x]] = sh.A[tri_index(R, threadIdx.x, threadIdx.x)];
}

// compute_pinv_square: eigenvalues at or below tol (relative: tol x the largest
// diagonal entry) dropped.  Where the first wavefront's Gauss-Jordan inverse
// shows that none is and that the matrix is well conditioned
// (WavePsd::well_posed) it is the result: n pivots instead of the
// eigendecomposition's eight sweeps of n - 1 rounds, and nearer the 64-bit value
// (R = 32 Grams: 7e-16 against 8e-15 relative).  Otherwise the two-sided Jacobi.
template <int NMAX>
__global__ __launch_bounds__(kJacobiThreads) void pinv_kernel(const double* __restrict__ Min, int R, double tol,
                                                        double* __restrict__ out, const int* __restrict__ only_if,
                                                        int relative, int two_sided) {
    if (only_if && *only_if == 0) return;   // the same for the whole block
    typedef WavePsd<NMAX> W;
    __shared__ EighSharedT<NMAX> sh;
    __shared__ double col[NMAX], tol_sh;
    __shared__ int done;
    const int64_t R2 = (int64_t)R * R;
    const double* M = Min + blockIdx.x * R2;
    if (threadIdx.x < 64) {
        double x[W::RPL], dmax, kappa;
        W::load(M, R, x);
        const double tr = W::trace(M, R, dmax);
        if (relative) tol *= dmax;
        bool ok = false;
        if (!two_sided) {
            ok = W::inverse(col, x, R);
            ok = W::well_posed(x, tr, tol, kappa) && ok;
        }
        if (ok) W::store(out + blockIdx.x * R2, R, x);
        if (threadIdx.x == 0) {
            done = ok ? 1 : 0;
            tol_sh = tol;
        }
    }
    __syncthreads();
    if (done) return;
    load_upper(M, R, sh.A);
    jacobi_block<NMAX>(sh.A, sh.A2, sh.V, R, sh.j);
    pinv_from_jacobi(sh, R, tol_sh, out + blockIdx.x * R2);
}

// ---------------------------------------------------------------- STS computeM
// sts_cp.hpp:80-188 for target mode j.  grams: N x R x R (full symmetric), M:
// (N+2) x R x R, lam: (N+1) x R.  Slot 0 is the pseudo-inverse of the Hadamard
// product H of the other modes' Grams (eigenvalues at or below 1e-8 dropped),
// slot N the rows u / sqrt(lam) of H's eigenvectors, slot k the rows
// sqrt(lam) u of those of A_k = (later Grams) (.) slot 0.  The reference solves
// slot N, then slot 0, then each k in turn; here every slot has a workgroup of
// its own.
//
// The draws pick an eigenvector by its mass, so they depend on the vectors and
// not only on the matrix.  Where H's (or A_k's) eigenvalues are apart, the
// vectors are determined to rounding and the one-sided Jacobi's serve as well;
// slot 0 is then the Gauss-Jordan inverse, where that shows that no eigenvalue is
// dropped, so that one eigendecomposition is the longest chain.  Where two are
// closer than kGap of the largest (kappa: slot 0 carries H's condition number
// into A_k), the vectors of two solvers differ by more than about 5 eps / kGap =
// 1e-9 (a draw in 1e4 calls of J = 65536 would move), and the oracle's two-sided
// Jacobi runs, operation for operation: mostly before the first updates, when
// every Gram is near the identity.
constexpr double kGap = 1e-6;

__device__ __forceinline__ int compute_m_slot(int N, int j, int block) {
    // workgroup 0: slot N; workgroup q: the q-th k of N-1 .. 1 (k != j)
    for (int k = N - 1, q = 0; k > 0 && block > 0; k--) {
        if (k == j) continue;
        if (++q == block) return k;
    }
    return N;
}

// One wavefront per slot; status[workgroup] = 1 where it wrote its slot.
template <int NMAX>
__global__ __launch_bounds__(64) void sts_compute_m_kernel(int N, int j, int R, const double* __restrict__ grams,
                                                           double* __restrict__ M, double* __restrict__ lam,
                                                           int* __restrict__ status) {
    typedef WavePsd<NMAX> W;
    __shared__ WavePsdShared<NMAX> sh;
    const int R2 = R * R, tid = threadIdx.x;
    const int slot = compute_m_slot(N, j, blockIdx.x);
    const int lj = tid % NMAX, g = tid / NMAX;
    double a[W::RPL], x[W::RPL], later[W::RPL];
    double tr = 0.0, lo = 1e300, hi = 0.0, off2 = 0.0;
#pragma unroll
    for (int r = 0; r < W::RPL; r++) {
        const int i = g * W::RPL + r;
        const bool in = i < R && lj < R;
        const int o = in ? (i <= lj ? i * R + lj : lj * R + i) : 0;
        double h = 1.0, lt = 0.0;
        for (int k = N - 1; k >= 0; k--) {
            if (k == j) continue;
            h *= grams[k * R2 + o];
            if (k == slot) lt = h;
        }
        a[r] = in ? h : 0.0;
        later[r] = in ? lt : 0.0;
        x[r] = a[r];
        if (in && i == lj) {
            tr += h;
            lo = fmin(lo, h);
            hi = fmax(hi, h);
        } else if (in) {
            off2 = fma(h, h, off2);
        }
    }
    if (blockIdx.x == 0) W::store(M + (N + 1) * R2, R, a);
    for (int off = 32; off >= 1; off >>= 1) {
        tr += __shfl_xor(tr, off, 64);
        off2 += __shfl_xor(off2, off, 64);
        lo = fmin(lo, __shfl_xor(lo, off, 64));
        hi = fmax(hi, __shfl_xor(hi, off, 64));
    }
    // R eigenvalues in an interval of this width, about R^2 / 4 to a close
    // pair: near the identity nothing is tried
    auto spread = [&](double l, double h, double o2, double gap) {
        return R < 2 || 4.0 * (h - l + 2.0 * sqrt(o2)) > gap * R * R * h;
    };
    bool fast = spread(lo, hi, off2, kGap);
    double kappa, gap = kGap;
    if (fast) {
        fast = W::inverse(sh.col, x, R);
        fast = W::well_posed(x, tr, 1e-8, kappa) && fast;
    }
    if (fast && slot != N) {
        gap *= fmax(1.0, 1e-2 * kappa);
        lo = 1e300;
        hi = off2 = 0.0;
#pragma unroll
        for (int r = 0; r < W::RPL; r++) {
            a[r] = later[r] * x[r];
            const int i = g * W::RPL + r;
            if (i < R && lj < R && i == lj) {
                lo = fmin(lo, a[r]);
                hi = fmax(hi, a[r]);
            } else {
                off2 = fma(a[r], a[r], off2);
            }
        }
        for (int off = 32; off >= 1; off >>= 1) {
            off2 += __shfl_xor(off2, off, 64);
            lo = fmin(lo, __shfl_xor(lo, off, 64));
            hi = fmax(hi, __shfl_xor(hi, off, 64));
        }
        fast = spread(lo, hi, off2, gap);
    }
    if (fast) {
        if (slot == N) W::store(M, R, x);
        fast = W::cholesky(sh, a, R);
        if (fast) {
            W::onesided(sh, R);
            fast = !W::close_pair(sh, R, gap);
        }
    }
    if (tid == 0) status[blockIdx.x] = fast ? 1 : 0;
    if (!fast) return;
    // rows ascending by eigenvalue (slot N: descending, scaled by 1 / sqrt(lam))
    const int ne = R + (R & 1);
    for (int o = tid; o < ne * R; o += 64) {
        const int c = o / R, u = o % R, at = sh.pos[c];
        if (at < 0) continue;
        const double lv = sh.lam[c], v = sh.L[c * NMAX + u];
        if (slot == N) M[(int64_t)N * R2 + (R - 1 - at) * R + u] = lv > 1e-8 ? v / lv : 0.0;
        else M[(int64_t)slot * R2 + at * R + u] = v;
        if (u == 0) lam[(slot == N ? 0 : slot) * R + at] = lv;
    }
}

// The slots that the kernel above left: the two-sided chain in the oracle's
// order.  H's eigenvectors, W = V diag(lam^-1/2) with columns reversed, slot 0 =
// W W^T, and for slot k the eigenvectors of A_k.
template <int NMAX>
__global__ __launch_bounds__(kJacobiThreads) void sts_compute_m_exact(int N, int j, int R, const double* __restrict__ grams,
                                                                      double* __restrict__ M, double* __restrict__ lam,
                                                                      const int* __restrict__ status) {
#pragma clang fp contract(off)
    if (status[blockIdx.x] != 0) return;   // the same for the whole workgroup
    __shared__ EighSharedT<NMAX> sh;
    __shared__ double Wm[NMAX * NMAX], later[NMAX * (NMAX + 1) / 2], s0[NMAX * (NMAX + 1) / 2];
    __shared__ int ord[NMAX];
    const int R2 = R * R, tid = threadIdx.x, nt = blockDim.x;
    const int slot = compute_m_slot(N, j, blockIdx.x);
    for (int o = tid; o < R2; o += nt) {
        const int p = o / R, q = o % R;
        if (p > q) continue;
        double h = 1.0, lt = 0.0;
        for (int k = N - 1; k >= 0; k--) {
            if (k == j) continue;
            h *= grams[k * R2 + o];
            if (k == slot) lt = h;
        }
        sh.A[tri_index(R, p, q)] = h;
        later[tri_index(R, p, q)] = lt;
    }
    __syncthreads();
    jacobi_block<NMAX>(sh.A, sh.A2, sh.V, R, sh.j);
    if (tid < R) ord[sh.j.rank[tid]] = tid;
    __syncthreads();
    for (int o = tid; o < R2; o += nt) {
        const int u = o / R, vs = o % R;          // vs = sorted column
        const int v = ord[vs];
        const double lv = sh.A[tri_index(R, v, v)];
        Wm[u * R + R - 1 - vs] = lv > 1e-8 ? sh.V[u * R + v] / sqrt(lv) : 0.0;
    }
    if (slot == N && tid < R) lam[sh.j.rank[tid]] = sh.A[tri_index(R, tid, tid)];
    __syncthreads();
    for (int o = tid; o < R2; o += nt) {
        const int p = o / R, q = o % R;
        if (p > q) continue;
        double acc = 0.0;
        for (int c = 0; c < R; c++) acc += Wm[p * R + c] * Wm[q * R + c];
        s0[tri_index(R, p, q)] = acc;
    }
    __syncthreads();
    if (slot == N) {
        for (int o = tid; o < R2; o += nt) {
            const int p = o / R, q = o % R;
            M[(int64_t)N * R2 + o] = Wm[q * R + p];
            M[o] = s0[sym_index(R, p, q)];
        }
        return;
    }
    for (int e = tid; e < tri_size(R); e += nt) sh.A[e] = later[e] * s0[e];
    __syncthreads();
    jacobi_block<NMAX>(sh.A, sh.A2, sh.V, R, sh.j);
    if (tid < R) {
        ord[sh.j.rank[tid]] = tid;
        lam[slot * R + sh.j.rank[tid]] = sh.A[tri_index(R, tid, tid)];
    }
    __syncthreads();
    for (int o = tid; o < R2; o += nt) {
        const int vs = o / R, u = o % R;
        const int v = ord[vs];
        const double lv = sh.A[tri_index(R, v, v)];
        M[(int64_t)slot * R2 + vs * R + u] = sh.V[u * R + v] * sqrt(lv > 0.0 ? lv : 0.0);
    }
}

// Eigen trees (PartitionTree(R, 1, R) per non-target mode k): leaves are the
// outer products of the rows of M[offset(k)], internal nodes sum their
// children; every node is then multiplied elementwise by G_k
// (sts_cp.hpp:179-187, partition_tree.hpp:117-187).
//
// Block (x, k) builds packed elements [64 x, 64 x + 64) of every node of mode
// k's tree in LDS (node-major), level by level in the heap order the row trees
// use, and writes them in the output precision TO with the node stride's
// padding zeroed.
// kEigCols columns per block keep the LDS tile under 64 KB: 64 for R <= 45,
// 32 above.
inline int eig_cols(int R) { return R <= 45 ? 64 : 32; }
template <typename TO>
__global__ __launch_bounds__(kThreads) void eig_tree_kernel(int N, int j, int R, const double* __restrict__ M,
                                                            const double* __restrict__ grams, TreeGeom ge,
                                                            TO* __restrict__ eig_nodes, int S, int kEigCols) {
    extern __shared__ double T[];   // node_count x kEigCols
    const int k = blockIdx.y;
    if (k == j || k >= N) return;
    const int P = tri_size(R), R2 = R * R;
    const int col = threadIdx.x % kEigCols, grp = threadIdx.x / kEigCols, ngrp = blockDim.x / kEigCols;
    const int e = blockIdx.x * kEigCols + col;
    int a = 0, b = 0;
    if (e < P) {
        while (a + 1 < R && tri_index(R, a + 1, a + 1) <= e) a++;
        b = a + (e - tri_index(R, a, a));
    }
    const int off = (k + 1 == j) ? k + 2 : k + 1;
    const double* W = M + (int64_t)off * R2;
    const int nodes = (int)ge.node_count;
    const int first_leaf = nodes - (int)ge.leaf_count;
    for (int i = grp; i < (int)ge.leaf_count; i += ngrp) {
        const int c = first_leaf + i;
        const int v = (int)ge.leaf_idx(c);
        T[c * kEigCols + col] = e < P ? W[v * R + a] * W[v * R + b] : 0.0;
    }
    __syncthreads();
    int start = (int)ge.nodes_before_lfill, end = first_leaf;
    for (int lvl = (int)ge.lfill_level; lvl >= 0; lvl--) {
        for (int c = start + grp; c < end; c += ngrp)
            T[c * kEigCols + col] = 0.0 + (T[(2 * c + 1) * kEigCols + col] + T[(2 * c + 2) * kEigCols + col]);
        __syncthreads();
        end = start;
        start = ((start + 1) / 2) - 1;
    }
    if (e >= S) return;
    const double g = e < P ? grams[(int64_t)k * R2 + a * R + b] : 0.0;
    TO* out = eig_nodes + (int64_t)k * nodes * S;
    for (int c = grp; c < nodes; c += ngrp) out[(int64_t)c * S + e] = (TO)(T[c * kEigCols + col] * g);
}

// res_i = u_i^T G u_i: sum_c u_c (sum_b u_b G[b][c]), each sum in order, in FP64
// (TA = float: rows of the mixed path, converted exactly).  One thread per row,
// which holds it in registers and takes four columns of G at a time (LDS, every
// lane the same address): four independent chains, and no load in the inner
// loop but G's.  RMAX is R rounded up to 8, the columns past R are zero; rows of
// short modes are spread over 64-thread workgroups.  2000 rows, R = 16: 36 ->
// 5.7 us (one column at a time, the row read again for each).
template <typename TA, int RMAX>
__global__ __launch_bounds__(kThreads) void dagat_kernel(const TA* __restrict__ A, int64_t m, int R,
                                                         const double* __restrict__ G, double* __restrict__ res) {
    typedef double d2 __attribute__((ext_vector_type(2)));
    __shared__ __align__(16) double g[RMAX * RMAX];
    for (int e = threadIdx.x; e < RMAX * RMAX; e += blockDim.x) {
        const int b = e / RMAX, c = e % RMAX;
        g[e] = b < R && c < R ? G[b * R + c] : 0.0;
    }
    __syncthreads();
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < m; i += (int64_t)gridDim.x * blockDim.x) {
        const TA* a = A + i * R;
        double u[RMAX];
#pragma unroll
        for (int b = 0; b < RMAX; b++) u[b] = (double)a[b < R ? b : 0];
#pragma unroll
        for (int b = 0; b < RMAX; b++) u[b] = b < R ? u[b] : 0.0;
        double r = 0.0;
        for (int c = 0; c < R; c += 4) {
            double uc[4], t[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
            for (int q = 0; q < 4; q++) uc[q] = (double)a[c + q < R ? c + q : 0];
#pragma unroll
            for (int b = 0; b < RMAX; b++) {
                const d2 x = *reinterpret_cast<const d2*>(g + b * RMAX + c);
                const d2 y = *reinterpret_cast<const d2*>(g + b * RMAX + c + 2);
                t[0] += u[b] * x[0];
                t[1] += u[b] * x[1];
                t[2] += u[b] * y[0];
                t[3] += u[b] * y[1];
            }
#pragma unroll
            for (int q = 0; q < 4; q++)
                if (c + q < R) r += uc[q] * t[q];
        }
        res[i] = r;
    }
}

// Column sums of squares, stage 1: part[block][c].
__global__ __launch_bounds__(kThreads) void col_sumsq_partial(const double* __restrict__ U, int64_t m, int R,
                                                              double* __restrict__ part) {
    __shared__ double red[kThreads];
    const int lanes = kThreads / R;           // rows processed in parallel
    const int c = threadIdx.x % R, rl = threadIdx.x / R;
    double acc = 0.0;
    if (rl < lanes) {
        const int64_t rows_per_block = (m + gridDim.x - 1) / gridDim.x;
        const int64_t r0 = blockIdx.x * rows_per_block;
        const int64_t r1 = r0 + rows_per_block < m ? r0 + rows_per_block : m;
        // eight rows in flight, added in order (2000 rows, R = 16: 17 -> 6.5 us)
        int64_t i = r0 + rl;
        for (; i + 7 * lanes < r1; i += 8 * lanes) {
            double v[8];
#pragma unroll
            for (int q = 0; q < 8; q++) v[q] = U[(i + q * lanes) * R + c];
#pragma unroll
            for (int q = 0; q < 8; q++) acc += v[q] * v[q];
        }
        for (; i < r1; i += lanes) {
            const double v = U[i * R + c];
            acc += v * v;
        }
    }
    red[threadIdx.x] = acc;
    __syncthreads();
    if (threadIdx.x < R) {
        double s = 0.0;
        for (int l = 0; l < lanes; l++) s += red[l * R + threadIdx.x];
        part[(int64_t)blockIdx.x * R + threadIdx.x] = s;
    }
}

// One wavefront per column: lane l sums partials l, l+64, ... in order, then
// a fixed butterfly; sigma = sqrt of the total.
__global__ __launch_bounds__(kThreads) void col_sumsq_final(const double* __restrict__ part, int nparts, int R,
                                                            double* __restrict__ sigma) {
    const int lane = threadIdx.x % 64;
    const int c = blockIdx.x * (kThreads / 64) + threadIdx.x / 64;
    if (c >= R) return;
    double s = 0.0;
    for (int p = lane; p < nparts; p += 64) s += part[(int64_t)p * R + c];
    s = wave_sum(s);
    if (lane == 0) sigma[c] = sqrt(s);
}

// U /= sigma by columns.  With few partials (part, at most kScaleParts of them)
// every workgroup adds them up itself, as col_sumsq_final does, and the first one
// writes sigma: a launch less, which is most of the time for short modes.
constexpr int kScaleParts = 16;
__global__ __launch_bounds__(kThreads) void scale_cols_kernel(double* __restrict__ U, int64_t m, int R,
                                                              double* __restrict__ sigma,
                                                              const double* __restrict__ part, int nparts) {
    __shared__ double sg[kMaxRank];
    if (threadIdx.x < R) {
        double s;
        if (part) {
            double v[kScaleParts];   // the lanes of that kernel's butterfly; the others hold zero
#pragma unroll
            for (int p = 0; p < kScaleParts; p++) v[p] = p < nparts ? part[(int64_t)p * R + threadIdx.x] : 0.0;
#pragma unroll
            for (int off = kScaleParts / 2; off >= 1; off >>= 1)
#pragma unroll
                for (int p = 0; p < off; p++) v[p] += v[p + off];
            s = sqrt(v[0]);
            if (blockIdx.x == 0) sigma[threadIdx.x] = s;
        } else {
            s = sigma[threadIdx.x];
        }
        sg[threadIdx.x] = s;
    }
    __syncthreads();
    const RowMap rm(R);
    if (!rm.on()) return;
    const double sc = sg[rm.c];
    for (int64_t i = rm.first(); i < m; i += rm.step()) U[i * R + rm.c] = U[i * R + rm.c] / sc;
}

__global__ __launch_bounds__(kThreads) void cos_init_kernel(double* __restrict__ U, int64_t m, int R) {
    const int64_t total = m * R;
    for (int64_t o = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; o < total; o += (int64_t)gridDim.x * blockDim.x)
        U[o] = cos((double)(uint64_t)o);
}

// sum_ab (prod_k G_k)[a][b] sigma_a sigma_b  (chain_had_prod over all modes).
__global__ __launch_bounds__(kThreads) void chain_had_norm_kernel(const double* __restrict__ grams, int N, int R,
                                                                  const double* __restrict__ sigma,
                                                                  double* __restrict__ out,
                                                                  double* __restrict__ size) {
    __shared__ double red[kThreads];
    const int R2 = R * R;
    double acc = 0.0;
    for (int o = threadIdx.x; o < R2; o += blockDim.x) {
        double p = 1.0;
        for (int k = 0; k < N; k++) p *= grams[(int64_t)k * R2 + o];
        acc += p * sigma[o / R] * sigma[o % R];
    }
    red[threadIdx.x] = acc;
    __syncthreads();
    if (threadIdx.x == 0) {
        double s = 0.0;
        for (int t = 0; t < kThreads; t++) s += red[t];
        *out = s;
    }
    if (threadIdx.x >= 64 && threadIdx.x < 64 + R) {   // (beside the sum, on another wavefront)
        const int r = threadIdx.x - 64;
        double p = fabs(sigma[r]);
        for (int k = 0; k < N; k++) p *= sqrt(grams[(int64_t)k * R2 + r * (R + 1)]);
        size[r] = p;
    }
}

// chain_had_prod (common.h:521-545): out = elementwise product of the Grams
// of every mode but `exclude`, multiplied in mode order.
__global__ __launch_bounds__(kThreads) void chain_had_kernel(const double* __restrict__ grams, int N, int exclude,
                                                             int R, double* __restrict__ out) {
    const int R2 = R * R;
    for (int o = threadIdx.x; o < R2; o += blockDim.x) {
        double p = 1.0;
        for (int k = 0; k < N; k++)
            if (k != exclude) p *= grams[(int64_t)k * R2 + o];
        out[o] = p;
    }
}

__global__ __launch_bounds__(kThreads) void preprocess_kernel(double* __restrict__ v, int64_t n, int kind) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        if (kind == 1) v[i] = log(v[i] + 1.0);
        else if (kind == 2) v[i] = 1.0;
    }
}

__global__ __launch_bounds__(kThreads) void sumsq_partial(const double* __restrict__ v, int64_t n,
                                                          double* __restrict__ part) {
    __shared__ double red[kThreads];
    double acc = 0.0;
    const int64_t per = (n + gridDim.x - 1) / gridDim.x;
    const int64_t lo = blockIdx.x * per, hi = lo + per < n ? lo + per : n;
    for (int64_t i = lo + threadIdx.x; i < hi; i += kThreads) acc += v[i] * v[i];
    red[threadIdx.x] = acc;
    __syncthreads();
    for (int w = kThreads / 2; w > 0; w >>= 1) {
        if (threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}

__global__ __launch_bounds__(kThreads) void plainsum_partial(const double* __restrict__ v, int64_t n,
                                                             double* __restrict__ part) {
    __shared__ double red[kThreads];
    double acc = 0.0;
    const int64_t per = (n + gridDim.x - 1) / gridDim.x;
    const int64_t lo = blockIdx.x * per, hi = lo + per < n ? lo + per : n;
    for (int64_t i = lo + threadIdx.x; i < hi; i += kThreads) acc += v[i];
    red[threadIdx.x] = acc;
    __syncthreads();
    for (int w = kThreads / 2; w > 0; w >>= 1) {
        if (threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}

__global__ void sum_final(const double* __restrict__ part, int nparts, double* __restrict__ out) {
    if (threadIdx.x != 0) return;
    double s = 0.0;
    for (int p = 0; p < nparts; p++) s += part[p];
    *out = s;
}

// packed[e] = M[a][b] for the packed upper element e = (a, b), zero for e in
// [tri_size(R), tri_pad256(R)).
__global__ void pack_upper_kernel(const double* __restrict__ M, int R, double* __restrict__ packed) {
    const int P = tri_size(R);
    for (int e = threadIdx.x; e < tri_pad256(R); e += blockDim.x) {
        if (e >= P) {
            packed[e] = 0.0;
            continue;
        }
        int a = 0;
        while (a + 1 < R && tri_index(R, a + 1, a + 1) <= e) a++;
        int b = a + (e - tri_index(R, a, a));
        packed[e] = M[a * R + b];
    }
}

}  // namespace

namespace k {

template <typename TA>
static void gram_mfma64(hipStream_t s, const TA* A, int64_t m, int R, double* G, DevBuf& part,
                        const uint64_t* m_dev = nullptr) {
    const int nb = (int)grid_for((m + 15) / 16, 4, 1024);
    part.ensure((size_t)nb * R * R * sizeof(double));
    const dim3 grid(nb), block(kThreads);
    switch ((R + 15) / 16) {
        case 1: hipLaunchKernelGGL((gram_mfma64_partial<TA, 1>), grid, block, 0, s, A, m, m_dev, R, part.as<double>()); break;
        case 2: hipLaunchKernelGGL((gram_mfma64_partial<TA, 2>), grid, block, 0, s, A, m, m_dev, R, part.as<double>()); break;
        case 3: hipLaunchKernelGGL((gram_mfma64_partial<TA, 3>), grid, block, 0, s, A, m, m_dev, R, part.as<double>()); break;
        default: hipLaunchKernelGGL((gram_mfma64_partial<TA, 4>), grid, block, 0, s, A, m, m_dev, R, part.as<double>()); break;
    }
    EX_HIP(hipGetLastError());
    gram_final_launch(s, part.as<double>(), nb, R, G);
}

// G = A^T A with the block partials in a caller-owned buffer of part_bytes:
// the block count is capped so that the partials fit (fewer, longer blocks;
// the sum is the same up to its grouping).  Allocates nothing.
void gram_into(hipStream_t s, const double* A, int64_t m, int R, double* G, double* part, size_t part_bytes) {
    const int64_t fit = (int64_t)(part_bytes / ((size_t)R * R * sizeof(double)));
    EX_CHECK(fit >= 1, 4, "Gram partials do not fit the scratch buffer");
    int nb = (int)grid_for((m + 15) / 16, 4, 1024);
    if (nb > fit) nb = (int)fit;
    const dim3 grid(nb), block(kThreads);
    switch ((R + 15) / 16) {
        case 1: hipLaunchKernelGGL((gram_mfma64_partial<double, 1>), grid, block, 0, s, A, m, nullptr, R, part); break;
        case 2: hipLaunchKernelGGL((gram_mfma64_partial<double, 2>), grid, block, 0, s, A, m, nullptr, R, part); break;
        case 3: hipLaunchKernelGGL((gram_mfma64_partial<double, 3>), grid, block, 0, s, A, m, nullptr, R, part); break;
        default: hipLaunchKernelGGL((gram_mfma64_partial<double, 4>), grid, block, 0, s, A, m, nullptr, R, part); break;
    }
    EX_HIP(hipGetLastError());
    gram_final_launch(s, part, nb, R, G);
}

void gram(hipStream_t s, const double* A, int64_t m, int R, double* G, DevBuf& part, const uint64_t* m_dev) {
    gram_mfma64<double>(s, A, m, R, G, part, m_dev);
}

void gram_f32in(hipStream_t s, const float* A, int64_t m, int R, double* G, DevBuf& part, const uint64_t* m_dev) {
    gram_mfma64<float>(s, A, m, R, G, part, m_dev);
}

void gram_final_launch(hipStream_t s, const double* part, int nb, int R, double* G) {
    hipLaunchKernelGGL(gram_final, dim3((R * R + 3) / 4), dim3(kThreads), 0, s, part, nb, R, G);
    EX_HIP(hipGetLastError());
}

void col_sumsq_final_launch(hipStream_t s, const double* part, int nb, int R, double* sigma) {
    hipLaunchKernelGGL(col_sumsq_final, dim3((R + 3) / 4), dim3(kThreads), 0, s, part, nb, R, sigma);
    EX_HIP(hipGetLastError());
}

// The R x R solves, sized to the rank: 16, 32 or 64.
#define PSD_DISPATCH(R, KERNEL, GRID, STREAM, ...)                                                                     \
    do {                                                                                                              \
        if ((R) <= 16) hipLaunchKernelGGL((KERNEL<16>), GRID, dim3(kJacobiThreads), 0, STREAM, __VA_ARGS__);     \
        else if ((R) <= 32) hipLaunchKernelGGL((KERNEL<32>), GRID, dim3(kJacobiThreads), 0, STREAM, __VA_ARGS__); \
        else hipLaunchKernelGGL((KERNEL<64>), GRID, dim3(kJacobiThreads), 0, STREAM, __VA_ARGS__);               \
    } while (0)

void eigh(hipStream_t s, const double* A, int R, double* lam, double* V, int ncopies) {
    PSD_DISPATCH(R, eigh_kernel, dim3(ncopies), s, A, R, lam, V);
    EX_HIP(hipGetLastError());
}

void pinv(hipStream_t s, const double* M, int R, double tol, double* out, int ncopies, const int* only_if,
          bool relative, bool two_sided) {
    PSD_DISPATCH(R, pinv_kernel, dim3(ncopies), s, M, R, tol, out, only_if, relative ? 1 : 0, two_sided ? 1 : 0);
    EX_HIP(hipGetLastError());
}

template <typename TA>
void dagat_rows(hipStream_t s, const TA* A, int64_t m, int R, const double* G, double* res) {
    const int threads = m < 65536 ? 64 : kThreads;
    const dim3 grid(grid_for(m, threads, 4096));
#define DAGAT(K) \
    case K: hipLaunchKernelGGL((dagat_kernel<TA, 8 * K>), grid, dim3(threads), 0, s, A, m, R, G, res); break
    switch ((R + 7) / 8) {
        DAGAT(1);
        DAGAT(2);
        DAGAT(3);
        DAGAT(4);
        DAGAT(5);
        DAGAT(6);
        DAGAT(7);
        DAGAT(8);
        default: EX_CHECK(false, 1, "rank out of range");
    }
#undef DAGAT
    EX_HIP(hipGetLastError());
}

void dagat(hipStream_t s, const double* A, int64_t m, int R, const double* G, double* res) {
    dagat_rows<double>(s, A, m, R, G, res);
}

void dagat32(hipStream_t s, const float* A, int64_t m, int R, const double* G, double* res) {
    dagat_rows<float>(s, A, m, R, G, res);
}

void dsymm(hipStream_t s, const double* G, const double* Y, int64_t m, int R, double* out) {
    dsymm_tile<double>(s, G, Y, m, R, out);
}

void normalize_cols(hipStream_t s, double* U, int64_t m, int R, double* sigma, DevBuf& part) {
    const int nb = (int)grid_for(m, 1024, 1024);
    part.ensure((size_t)nb * R * sizeof(double));
    hipLaunchKernelGGL(col_sumsq_partial, dim3(nb), dim3(kThreads), 0, s, U, m, R, part.as<double>());
    if (nb > kScaleParts) col_sumsq_final_launch(s, part.as<double>(), nb, R, sigma);
    hipLaunchKernelGGL(scale_cols_kernel, dim3(grid_for(m, kThreads / R, 8192)), dim3(kThreads), 0, s, U, m, R, sigma,
                       nb > kScaleParts ? nullptr : part.as<double>(), nb);
    EX_HIP(hipGetLastError());
}

void cos_init(hipStream_t s, double* U, int64_t m, int R) {
    hipLaunchKernelGGL(cos_init_kernel, dim3(grid_for(m * R, kThreads, 8192)), dim3(kThreads), 0, s, U, m, R);
    EX_HIP(hipGetLastError());
}

void chain_had_norm(hipStream_t s, const double* grams, int N, int R, const double* sigma, double* out, double* size) {
    hipLaunchKernelGGL(chain_had_norm_kernel, dim3(1), dim3(kThreads), 0, s, grams, N, R, sigma, out, size);
    EX_HIP(hipGetLastError());
}

void chain_had(hipStream_t s, const double* grams, int N, int exclude, int R, double* out) {
    hipLaunchKernelGGL(chain_had_kernel, dim3(1), dim3(kThreads), 0, s, grams, N, exclude, R, out);
    EX_HIP(hipGetLastError());
}

void preprocess(hipStream_t s, double* vals, int64_t nnz, int kind) {
    if (kind == 0 || nnz == 0) return;
    hipLaunchKernelGGL(preprocess_kernel, dim3(grid_for(nnz, kThreads, 8192)), dim3(kThreads), 0, s, vals, nnz, kind);
    EX_HIP(hipGetLastError());
}

void sumsq(hipStream_t s, const double* v, int64_t n, double* out, DevBuf& part) {
    int nb = (int)grid_for(n, 4096, 1024);
    part.ensure((size_t)nb * sizeof(double));
    hipLaunchKernelGGL(sumsq_partial, dim3(nb), dim3(kThreads), 0, s, v, n, part.as<double>());
    hipLaunchKernelGGL(sum_final, dim3(1), dim3(64), 0, s, part.as<double>(), nb, out);
    EX_HIP(hipGetLastError());
}

int plain_sum_blocks(int64_t n) { return (int)grid_for(n, 4096, 1024); }

void plain_sum(hipStream_t s, const double* v, int64_t n, double* out, DevBuf& part) {
    const int nb = plain_sum_blocks(n);
    part.ensure((size_t)nb * sizeof(double));
    hipLaunchKernelGGL(plainsum_partial, dim3(nb), dim3(kThreads), 0, s, v, n, part.as<double>());
    hipLaunchKernelGGL(sum_final, dim3(1), dim3(64), 0, s, part.as<double>(), nb, out);
    EX_HIP(hipGetLastError());
}

void sts_compute_m(hipStream_t s, int N, int j, int R, const double* grams, double* M, double* lam) {
    // one workgroup per slot: N and every k in 1 .. N-1, k != j
    int jobs = 1;
    for (int k = 1; k < N; k++) jobs += k != j ? 1 : 0;
    int* status = reinterpret_cast<int*>(lam + (int64_t)(N + 1) * R);
    if (R <= 16) hipLaunchKernelGGL(sts_compute_m_kernel<16>, dim3(jobs), dim3(64), 0, s, N, j, R, grams, M, lam, status);
    else if (R <= 32) hipLaunchKernelGGL(sts_compute_m_kernel<32>, dim3(jobs), dim3(64), 0, s, N, j, R, grams, M, lam, status);
    else hipLaunchKernelGGL(sts_compute_m_kernel<64>, dim3(jobs), dim3(64), 0, s, N, j, R, grams, M, lam, status);
    PSD_DISPATCH(R, sts_compute_m_exact, dim3(jobs), s, N, j, R, grams, M, lam, status);
    EX_HIP(hipGetLastError());
}

void eig_tree_build(hipStream_t s, int N, int j, int R, const double* M, const double* grams, double* eig_nodes) {
    TreeGeom ge;
    ge.init(R, 1);
    const int S = tri_stride(R), cols = eig_cols(R);
    const size_t lds = (size_t)ge.node_count * cols * sizeof(double);
    hipLaunchKernelGGL(eig_tree_kernel<double>, dim3((S + cols - 1) / cols, N), dim3(kThreads), lds, s, N, j, R, M,
                       grams, ge, eig_nodes, S, cols);
    EX_HIP(hipGetLastError());
}

void eig_tree_build32(hipStream_t s, int N, int j, int R, const double* M, const double* grams, float* eig_nodes) {
    TreeGeom ge;
    ge.init(R, 1);
    const int S = tri_stride32(R), cols = eig_cols(R);
    const size_t lds = (size_t)ge.node_count * cols * sizeof(double);
    hipLaunchKernelGGL(eig_tree_kernel<float>, dim3((S + cols - 1) / cols, N), dim3(kThreads), lds, s, N, j, R, M,
                       grams, ge, eig_nodes, S, cols);
    EX_HIP(hipGetLastError());
}

void pack_upper(hipStream_t s, const double* M, int R, double* packed) {
    hipLaunchKernelGGL(pack_upper_kernel, dim3(1), dim3(kThreads), 0, s, M, R, packed);
    EX_HIP(hipGetLastError());
}

}  // namespace k
}  // namespace exafac
