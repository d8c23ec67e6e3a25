// FP64 solves of a symmetric positive definite n x n matrix (n <= NMAX) on ONE
// wavefront: Gauss-Jordan inverse, pivoted Cholesky factor, and the
// eigendecomposition by one-sided Jacobi on that factor.  They serve matrices
// whose solution rounding determines well; the callers keep the two-sided
// Jacobi (jacobi_block.hpp) for singular, ill-conditioned and indefinite ones.
//
// What bounds them is the latency of a serial chain (n pivots; about eight
// sweeps of n - 1 rounds), so a step is kept inside one wavefront: operands in
// registers, exchanges by DPP or a few LDS words, and no workgroup barrier.
// On an MI355X, against the two-sided Jacobi on four wavefronts (one barrier
// and a divide and square-root chain a round), per launch:
//   pseudo-inverse         R = 8 70 -> 4 us, 16 147 -> 5, 25 295 -> 15,
//                          32 416 -> 18, 64 2818 -> 85
//   computeM, three modes  R = 16 429 -> 43 us, 32 1039 -> 156, 64 7141 -> 820
#pragma once
#include "common.hpp"

namespace exafac {
namespace {

__device__ __forceinline__ void wave_psd_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// 1 / x and 1 / sqrt(x) from the hardware estimate and Newton steps
// (x_{k+1} = x_k + x_k (1 - a x_k); y_{k+1} = y_k + y_k (1 - a y_k^2) / 2), two
// for a result within an ulp or so, one where an angle only has to be near.
template <int STEPS>
__device__ __forceinline__ double newton_rcp(double a) {
    double x = __builtin_amdgcn_rcp(a);
#pragma unroll
    for (int q = 0; q < STEPS; q++) x = fma(x, fma(-a, x, 1.0), x);
    return x;
}
template <int STEPS>
__device__ __forceinline__ double newton_rsqrt(double a) {
    double y = __builtin_amdgcn_rsq(a);
#pragma unroll
    for (int q = 0; q < STEPS; q++) y = fma(0.5 * y, fma(-a * y, y, 1.0), y);
    return y;
}

// The value of the lane below (UP) or above: inside rows of 16 lanes, or
// across the wavefront.  Lanes without a source get 0.
template <int CTRL>
__device__ __forceinline__ double dpp_move(double v) {
    const uint64_t u = (uint64_t)__double_as_longlong(v);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)u, CTRL, 0xF, 0xF, true);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(u >> 32), CTRL, 0xF, 0xF, true);
    return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}
template <bool ROW16, bool UP>
__device__ __forceinline__ double lane_next(double v) {
    // row_shr:1 / row_shl:1, wave_shr:1 / wave_shl:1
    return dpp_move<ROW16 ? (UP ? 0x111 : 0x101) : (UP ? 0x138 : 0x130)>(v);
}

// v + the value of lane ^ 32 (or ^ 16): the two halves are swapped between two
// copies of v, whose sum is then the same in both partners.
__device__ __forceinline__ double add_xor32(double v) {
    const uint64_t u = (uint64_t)__double_as_longlong(v);
    const auto l = __builtin_amdgcn_permlane32_swap((uint32_t)u, (uint32_t)u, false, false);
    const auto h = __builtin_amdgcn_permlane32_swap((uint32_t)(u >> 32), (uint32_t)(u >> 32), false, false);
    return __longlong_as_double((long long)(((uint64_t)h[0] << 32) | l[0])) +
           __longlong_as_double((long long)(((uint64_t)h[1] << 32) | l[1]));
}
__device__ __forceinline__ double add_xor16(double v) {
    const uint64_t u = (uint64_t)__double_as_longlong(v);
    const auto l = __builtin_amdgcn_permlane16_swap((uint32_t)u, (uint32_t)u, false, false);
    const auto h = __builtin_amdgcn_permlane16_swap((uint32_t)(u >> 32), (uint32_t)(u >> 32), false, false);
    return __longlong_as_double((long long)(((uint64_t)h[0] << 32) | l[0])) +
           __longlong_as_double((long long)(((uint64_t)h[1] << 32) | l[1]));
}

template <int NMAX>
struct WavePsdShared {
    double col[NMAX];           // the column being eliminated
    double L[NMAX * NMAX];      // column c at L[c * NMAX + i]
    double lam[NMAX];           // eigenvalue of column c
    int pos[NMAX];              // its ascending position (ties by c), -1: the padding column of an odd order
};

// Lane layouts: a matrix column per lane j = lane % NMAX, its rows g RPL + r
// (g = lane / NMAX) in registers; a pair of columns per lane p = lane % PL, its
// rows g PR + r (g = lane / PL).
template <int NMAX>
struct WavePsd {
    static constexpr int RPL = NMAX * NMAX / 64;
    static constexpr int PL = NMAX / 2;
    static constexpr int PR = NMAX * PL / 64;
    typedef WavePsdShared<NMAX> Shared;

    static __device__ __forceinline__ int lane() { return (int)(threadIdx.x % 64); }

    // The symmetric matrix whose upper triangle is M's (row-major n x n); zero past n.
    static __device__ __forceinline__ void load(const double* __restrict__ M, int n, double (&a)[RPL]) {
        const int j = lane() % NMAX, g = lane() / NMAX;
#pragma unroll
        for (int r = 0; r < RPL; r++) {
            const int i = g * RPL + r;
            const bool in = i < n && j < n;
            const double v = M[in ? (i <= j ? i * n + j : j * n + i) : 0];
            a[r] = in ? v : 0.0;
        }
    }
    // out = the symmetric matrix with a's upper triangle.
    static __device__ __forceinline__ void store(double* __restrict__ out, int n, const double (&a)[RPL]) {
        const int j = lane() % NMAX, g = lane() / NMAX;
#pragma unroll
        for (int r = 0; r < RPL; r++) {
            const int i = g * RPL + r;
            if (i <= j && j < n) {
                out[i * n + j] = a[r];
                out[j * n + i] = a[r];
            }
        }
    }

    // In-place Gauss-Jordan inverse, pivots in order.  The row of pivot k is
    // its column with the sign turned where k' < k has been eliminated.
    // Returns whether every pivot was positive.
    static __device__ __forceinline__ bool inverse(double (&col)[NMAX], double (&a)[RPL], int n) {
        const int j = lane() % NMAX, g = lane() / NMAX;
        bool ok = true;
        auto step = [&](int k, auto row) {
            if (j == k)
#pragma unroll
                for (int r = 0; r < RPL; r++) col[g * RPL + r] = a[r];
            wave_psd_sync();
            const double piv = col[k], cj = col[j];
            double c[RPL];
#pragma unroll
            for (int r = 0; r < RPL; r++) c[r] = col[g * RPL + r];
            wave_psd_sync();
            ok = ok && piv > 0.0;
            const double inv = 1.0 / piv;
            const double w = j == k ? inv : (j < k ? -cj : cj) * inv;
            const double z = j == k ? 0.0 : 1.0;
#pragma unroll
            for (int r = 0; r < RPL; r++) {
                const double v = fma(-c[r], w, a[r] * z);
                a[r] = row(r) ? w : v;
            }
        };
        if constexpr (RPL <= 16) {
            // the pivot's register is known at compile time: one select per step
            for (int kb = 0, gk = 0; kb < n; kb += RPL, gk++) {
#pragma unroll
                for (int kr = 0; kr < RPL; kr++)
                    if (kb + kr < n) step(kb + kr, [&](int r) { return r == kr && g == gk; });
            }
        } else {
            for (int k = 0; k < n; k++) step(k, [&](int r) { return g * RPL + r == k; });
        }
        return ok;
    }

    // Whether the inverse x of a matrix of trace tr shows that every eigenvalue
    // of the matrix is above tol (the smallest one is at least 1 / |x|_F; the
    // margin of 4 covers x's rounding) and that its condition number is below
    // 1e6, where x is within 1e-10 of any other solver's result.  kappa = |x|_F
    // tr, a bound on the condition number.
    static __device__ __forceinline__ bool well_posed(const double (&x)[RPL], double tr, double tol, double& kappa) {
        double s = 0.0;
#pragma unroll
        for (int r = 0; r < RPL; r++) s = fma(x[r], x[r], s);
        for (int off = 32; off >= 1; off >>= 1) s += __shfl_xor(s, off, 64);
        const double nrm = sqrt(s);
        kappa = nrm * tr;
        return nrm * tol * 4.0 < 1.0 && kappa < 1e6;   // false for NaN
    }

    // Whether two of sh.lam's eigenvalues are closer than rel times the largest.
    static __device__ __forceinline__ bool close_pair(const Shared& sh, int n, double rel) {
        const int ne = n + (n & 1), c = lane();
        double lv = c < ne ? sh.lam[c] : 0.0, top = lv;
        for (int off = 32; off >= 1; off >>= 1) top = fmax(top, __shfl_xor(top, off, 64));
        bool near = false;
        if (c < ne)
            for (int u = 0; u < ne; u++) near = near || (u != c && !(fabs(sh.lam[u] - lv) >= rel * top));
        return __ballot(near) != 0;
    }

    static __device__ __forceinline__ double trace(const double* __restrict__ M, int n, double& dmax) {
        const int j = lane();
        const double d = j < n ? M[j * n + j] : 0.0;
        double t = d, m = d;
        for (int off = 32; off >= 1; off >>= 1) {
            t += __shfl_xor(t, off, 64);
            m = fmax(m, __shfl_xor(m, off, 64));
        }
        dmax = m;
        return t;
    }

    // Pivoted Cholesky A = sum_k l_k l_k^T with the rows left in place (column
    // l_k at sh.L[k NMAX], zero at the rows eliminated before it): no swaps.
    // false: a pivot was not above n eps times the largest diagonal entry, or
    // that entry is outside [1e-100, 1e100].
    static __device__ __forceinline__ bool cholesky(Shared& sh, double (&a)[RPL], int n) {
        const int j = lane() % NMAX, g = lane() / NMAX;
#pragma unroll
        for (int r = 0; r < RPL; r++)
            if (g * RPL + r == j) sh.col[j] = a[r];
        wave_psd_sync();
        double d = sh.col[j], dmax = d;   // own diagonal entry
        wave_psd_sync();
        for (int off = 32; off >= 1; off >>= 1) dmax = fmax(dmax, __shfl_xor(dmax, off, 64));
        if (!(dmax >= 1e-100 && dmax <= 1e100)) return false;
        const double thr = (double)n * 2.220446049250313e-16 * dmax, inv = 1.0 / dmax;
        uint64_t done = 0;
        for (int k = 0; k < n; k++) {
            // the pivot: the largest remaining diagonal entry, to FP32 with the
            // column number in the low bits
            uint32_t key = 0;
            if (j < n && !((done >> j) & 1) && d > thr)
                key = (__float_as_uint((float)(d * inv)) & ~63u) | (uint32_t)(63 - j);
            for (int off = 32; off >= 1; off >>= 1) {
                const uint32_t o = __shfl_xor(key, off, 64);
                key = o > key ? o : key;
            }
            key = (uint32_t)__builtin_amdgcn_readfirstlane((int)key);
            if (key == 0) return false;
            const int p = 63 - (int)(key & 63u);
            if (j == p)
#pragma unroll
                for (int r = 0; r < RPL; r++) sh.col[g * RPL + r] = a[r];
            wave_psd_sync();
            const double rs = newton_rsqrt<2>(sh.col[p]);
            const double lj = ((done >> j) & 1) ? 0.0 : sh.col[j] * rs;
            if (g == 0) sh.L[k * NMAX + j] = lj;
            wave_psd_sync();
#pragma unroll
            for (int r = 0; r < RPL; r++) a[r] = fma(-sh.L[k * NMAX + g * RPL + r], lj, a[r]);
            d = fma(-lj, lj, d);
            done |= (uint64_t)1 << p;
        }
        return true;
    }

    // One-sided Jacobi on the n columns at sh.L: rotations from the
    // right make the columns orthogonal, L V = U diag(sqrt(lam)), so A = L L^T =
    // U diag(lam) U^T.  Afterwards column c (c < ne, n rounded up to even) at
    // sh.L[c NMAX] is sqrt(lam_c) u_c, with sh.lam and sh.pos.  A pair of
    // columns per lane; between rounds the columns move one lane along the
    // round-robin circle.  The rotation's tangent is only near its exact value
    // (one Newton step): what it leaves off the diagonal the next sweep takes.
    // c is exact to an ulp, so the columns' products sum to A throughout.
    static __device__ __forceinline__ void onesided(Shared& sh, int n) {
        constexpr bool kRow16 = PL <= 16;
        const int p = lane() % PL, g = lane() / PL;
        const int m = (n + 1) / 2;
        constexpr double tol2 = 16.0 * 2.220446049250313e-16 * 2.220446049250313e-16;
        auto across = [](double v) {
            // sum over the lanes of one pair
            if constexpr (PL <= 8) v += dpp_move<0x128>(v);   // row_ror:8
            if constexpr (PL <= 16) v = add_xor16(v);
            return add_xor32(v);
        };
        double x[PR], y[PR];
#pragma unroll
        for (int r = 0; r < PR; r++) {
            const int i = g * PR + r;
            x[r] = (p < m && i < n) ? sh.L[p * NMAX + i] : 0.0;
            y[r] = (p < m && p + m < n && i < n) ? sh.L[(p + m) * NMAX + i] : 0.0;
        }
        const bool first = p == 0, last = p == m - 1;
        double app, aqq;
        auto norms = [&]() {
            double s = 0.0, t = 0.0;
#pragma unroll
            for (int r = 0; r < PR; r++) {
                s = fma(x[r], x[r], s);
                t = fma(y[r], y[r], t);
            }
            app = across(s);
            aqq = across(t);
        };
        auto move = [&](double& top, double& bot) {
            const double t = lane_next<kRow16, true>(first ? bot : top);
            const double b = lane_next<kRow16, false>(bot);
            bot = last ? top : b;
            top = first ? top : t;
        };
        for (int sweep = 0; sweep < 40; sweep++) {
            norms();
            bool any = false;
            for (int round = 0; round < 2 * m - 1; round++) {
                double s0 = 0.0, s1 = 0.0;
#pragma unroll
                for (int r = 0; r < PR; r += 2) {
                    s0 = fma(x[r], y[r], s0);
                    s1 = fma(x[r + 1], y[r + 1], s1);
                }
                const double apq = across(s0 + s1);
                const bool rot = p < m && apq * apq > tol2 * (app * aqq);
                if (__ballot(rot) != 0) {
                    any = true;
                    const double d = aqq - app, b = 2.0 * apq;
                    const double h2 = fma(d, d, b * b);
                    const double h = h2 * newton_rsqrt<1>(h2);
                    double t = (d >= 0.0 ? b : -b) * newton_rcp<1>(fabs(d) + h);
                    t = rot ? t : 0.0;
                    const double c = newton_rsqrt<2>(fma(t, t, 1.0)), s = t * c;
#pragma unroll
                    for (int r = 0; r < PR; r++) {
                        const double u = x[r], v = y[r];
                        x[r] = fma(c, u, -(s * v));
                        y[r] = fma(s, u, c * v);
                    }
                    app = fma(-t, apq, app);
                    aqq = fma(t, apq, aqq);
                }
                if (m > 1) {
#pragma unroll
                    for (int r = 0; r < PR; r++) move(x[r], y[r]);
                    move(app, aqq);
                }
            }
            if (!any) break;
        }
        norms();
        wave_psd_sync();
        if (p < m) {
#pragma unroll
            for (int r = 0; r < PR; r++) {
                sh.L[p * NMAX + g * PR + r] = x[r];
                sh.L[(p + m) * NMAX + g * PR + r] = y[r];
            }
            if (g == 0) {
                sh.lam[p] = app;
                sh.lam[p + m] = aqq;
            }
        }
        wave_psd_sync();
        order(sh, n);
    }

    static __device__ __forceinline__ void order(Shared& sh, int n) {
        const int ne = n + (n & 1), c = lane();
        if (c < ne) {
            const double lv = sh.lam[c];
            int k = 0;
            for (int u = 0; u < ne; u++) {
                const double lu = sh.lam[u];
                k += (lu < lv || (lu == lv && u < c)) ? 1 : 0;
            }
            sh.pos[c] = k - (ne - n);
        }
        wave_psd_sync();
    }
};

}  // namespace
}  // namespace exafac
