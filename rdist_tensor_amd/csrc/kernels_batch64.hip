// Batched CP-ARLS-LEV, FP64: one sweep of every tensor of a batch as a chain of
// launches, each a phase of one mode step (accumulator_stationary.hpp:139-295
// with cp_arls_lev.hpp:25-163) for all tensors: blockIdx.y (or x) is the tensor.
//
// A mode step of one tensor is two R x R eigendecompositions, each a serial
// chain on one workgroup, and phases over its samples and rows.  One workgroup
// per tensor for all of it (as the mixed sweep runs, kernels_batch.hip) left all
// but 32 of the 256 CUs idle for 32 tensors, and its 1024 threads' registers
// spilled: 1.65 ms a mode step at R = 32, J = 8192, of which 0.8 ms outside the
// solves.  Here the phases spread over the chip, the solver has a workgroup of
// its own size, and the sampled MTTKRP runs beside the first solve.  Five sweeps
// of 32 tensors (R 8-32, 60-600 rows a mode, J = 8192): 26.4 -> 13.5 ms; a mode
// step at R = 32 takes 0.84 ms, of which the two solves 0.65.
//
// The leverage state over the nonzero rows only is that of kernels_batch.hip.
// Every sum keeps the order it has there: sweeps of a factor with few
// nonzero rows magnify a last-bit difference without bound.
#include "batch_block.hpp"
#include "jacobi_block.hpp"

namespace exafac {
namespace {

constexpr int kT = 256;
constexpr int kChunkRows = 256;                  // rows after which a Gram's groups start over
static_assert(kT == kJacobiThreads, "a solve takes one workgroup");

// A Gram is summed by 1024 / ceil(R/2)^2 groups: row r belongs to group (r % 256)
// % groups, a group adds its rows in order, and the groups are added in order.
// (At most 256 groups have rows.)
__host__ __device__ inline int gram_groups(int R) {
    const int H = (R + 1) / 2;
    return kBT / (H * H);
}
__host__ __device__ inline int gram_live_groups(int R) {
    const int g = gram_groups(R);
    return g < kChunkRows ? g : kChunkRows;
}
__host__ __device__ inline int gram_items(int R) { return gram_live_groups(R) * (R > 16 ? 3 : 1); }
// Low ranks have up to 256 groups, each of few rows and few sums: up to 32 rows a
// group, a Gram is summed by one thread per group and entry, else by one
// wavefront per group and 16 x 16 tile, which loads 16 steps of four rows at least.
// 256 tensors, J = 500, the design's and the factor's Gram: R = 1 191 + 532 -> 5 +
// 39 us by threads, R = 4 134 + 225 -> 15 + 35, R = 8 40 + 85 -> 13 + 31.  (At 128
// rows a group a thread's chain would be eight rounds of loads; the wavefronts take
// two: R = 8, J = 8192 17 us.)
__host__ __device__ inline bool gram_by_threads(int R, int64_t rows) {
    return R <= 16 && rows <= 32 * (int64_t)gram_live_groups(R);
}
__host__ __device__ inline int gram_thread_blocks(int R) { return (gram_live_groups(R) * tri_size(R) + kT - 1) / kT; }
__host__ __device__ inline int gram_wave_blocks(int R) { return (gram_items(R) + kT / 64 - 1) / (kT / 64); }
// Workgroups for a Gram of exactly `rows` rows, and of at most that many.
__host__ __device__ inline int gram_blocks(int R, int64_t rows) {
    return gram_by_threads(R, rows) ? gram_thread_blocks(R) : gram_wave_blocks(R);
}
inline int gram_blocks_bound(int R, int64_t rows) {
    const int t = gram_by_threads(R, 0) ? gram_thread_blocks(R) : 0;
    return gram_by_threads(R, rows) ? t : std::max(t, gram_wave_blocks(R));
}
// Rows of the factor update whose squares one thread of a column adds up, in
// order: q, q + norm_classes, ...
__host__ __device__ inline int norm_classes(int R) { return kBT / R; }

// ---------------------------------------------------------------- draws
// cp_arls_lev.hpp:36-163 with the row CDFs of the other modes: sample s takes row
// lower_bound(cdf_k, u) of every mode k != j, u from the generator at (sweep, j,
// k); weight = prod_k (sum_k / score_k) / J.
__global__ __launch_bounds__(kT) void b64_draw(const BatchTensor* __restrict__ ts, int j, int64_t J,
                                               const BatchCtl* __restrict__ ctl) {
    const BatchTensor& T = ts[blockIdx.y];
    const int N = T.N;
    if (j >= N) return;
    // the logarithms that every sample shares: a lane each
    __shared__ double logs[kMaxModes + 1];
    if (threadIdx.x <= (unsigned)N) {
        const int k = (int)threadIdx.x;
        logs[k] = log(k < N ? (k != j ? 0.0 + gl(T.ssum)[k] : 1.0) : (double)J);
    }
    __syncthreads();
    const int64_t s = blockIdx.x * (int64_t)kT + threadIdx.x;
    if (s >= J) return;
    double w = 0.0 - logs[N];
    uint64_t key = 0;
    for (int k = 0; k < N; k++) {
        uint32_t row = 0;
        if (k != j) {
            const BatchMode& M = T.m[k];
            const uint32_t L = gl(T.cnt)[k];
            const double ls = logs[k];
            const double u = uniform01(T.seed, stream_id(ctl->sweep, (uint32_t)j, (uint32_t)k, 0), (uint64_t)s);
            double sc = 0.0;
            if (L > 0) {
                const Gp<const double> cdf = gl((const double*)M.ccdf);
                uint32_t b = 0;
                for (uint32_t len = L; len > 1;) {
                    const uint32_t half = len >> 1;
                    b += cdf[b + half - 1] < u ? half : 0u;
                    len -= half;
                }
                b += cdf[b] < u ? 1u : 0u;
                const uint32_t idx = b < L ? b : L - 1;
                row = gl(M.list)[idx];
                sc = gl(M.csc)[idx];
            }
            w += ls - log(sc);
            if (T.m[j].shift[k] >= 0) key |= (uint64_t)row << T.m[j].shift[k];
        }
        gl(T.samples)[s * N + k] = row;
    }
    gl(T.weights)[s] = exp(w);
    gl(T.skey)[s] = key;
}

// deduplicate_design_matrix (als_optimizer.hpp:130-206) in first-occurrence
// order: a table of 2^14 LDS slots holds the first sample (index + 1) of each
// fiber key (open addressing), then the unique rank of the key in its low 16 bits
// and its multiplicity in the high 16 bits.  Writes sd, kd, wd (the square root
// of weight x multiplicity) and J_u.  Thread t takes samples t, t + 1024, ...: every access
// is coalesced (a thread's own consecutive samples cost a cache line each).
__global__ __launch_bounds__(kBT) void b64_dedup(const BatchTensor* __restrict__ ts, int j, int64_t J) {
    const BatchTensor& T = ts[blockIdx.x];
    if (j >= T.N) return;
    __shared__ uint32_t tab[1 << kTableBits];
    __shared__ uint32_t cnt[kMaxQ * kWaves];   // first occurrences per (pass, wavefront)
    constexpr uint32_t mask = (1u << kTableBits) - 1u;
    const int N = T.N, t = threadIdx.x, lane = t & 63, wave = t >> 6;
    for (int i = t; i < (1 << kTableBits); i += kBT) tab[i] = 0u;
    __syncthreads();
    uint64_t key[kMaxQ];
    uint32_t slot[kMaxQ];
#pragma unroll
    for (int q = 0; q < kMaxQ; q++) {
        const int64_t i = t + (int64_t)q * kBT;
        key[q] = i < J ? gl(T.skey)[i] : 0;
    }
#pragma unroll
    for (int q = 0; q < kMaxQ; q++) {
        const int64_t i = t + (int64_t)q * kBT;
        slot[q] = 0;
        if (i >= J) continue;
        const uint32_t me = (uint32_t)i + 1u;
        uint32_t h = table_slot(key[q]);
        while (true) {
            uint32_t cur = tab[h];
            if (cur == 0u) {
                cur = atomicCAS(&tab[h], 0u, me);
                if (cur == 0u) break;
            }
            if (gl(T.skey)[cur - 1u] == key[q]) {
                atomicMin(&tab[h], me);
                break;
            }
            h = (h + 1u) & mask;
        }
        slot[q] = h;
    }
    __syncthreads();
    uint32_t rank[kMaxQ];
    uint32_t first = 0;   // bit q: the sample is its key's first occurrence
#pragma unroll
    for (int q = 0; q < kMaxQ; q++) {
        const int64_t i = t + (int64_t)q * kBT;
        const bool f = i < J && tab[slot[q]] == (uint32_t)i + 1u;
        const uint64_t m = __ballot(f);
        rank[q] = (uint32_t)__popcll(m & ((1ull << lane) - 1ull));
        if (f) first |= 1u << q;
        if (lane == 0) cnt[q * kWaves + wave] = (uint32_t)__popcll(m);
    }
    __syncthreads();
    if (wave == 0) {   // exclusive prefix over the kMaxQ x kWaves counts, two a lane
        static_assert(kMaxQ * kWaves == 128, "two counts a lane");
        const uint32_t a = cnt[2 * lane], b = cnt[2 * lane + 1];
        uint32_t inc = a + b;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const uint32_t y = __shfl_up(inc, d, 64);
            if (lane >= d) inc += y;
        }
        cnt[2 * lane] = inc - a - b;
        cnt[2 * lane + 1] = inc - b;
        if (lane == 63) *T.ju = inc;
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < kMaxQ; q++) {
        rank[q] += cnt[q * kWaves + wave];
        if ((first >> q) & 1u) tab[slot[q]] = rank[q];
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < kMaxQ; q++)
        if (t + (int64_t)q * kBT < J) atomicAdd(&tab[slot[q]], 1u << 16);
    __syncthreads();
#pragma unroll
    for (int q = 0; q < kMaxQ; q++) {
        if (!((first >> q) & 1u)) continue;
        const int64_t i = t + (int64_t)q * kBT;
        const uint32_t u = rank[q];
        for (int k = 0; k < N; k++) gl(T.sd)[(int64_t)u * N + k] = gl(T.samples)[i * N + k];
        gl(T.kd)[u] = key[q];
        gl(T.wd)[u] = sqrt(gl(T.weights)[i] * (double)(tab[slot[q]] >> 16));
    }
}

// ---------------------------------------------------------------- design, hits
// KRP gather (accumulator_stationary.hpp:210-249): dg = prod_{k != j} U_k[s_k]
// sqrt(w) (the MTTKRP multiplies the few rows that it takes by sqrt(w) again: a
// second J x R array was a third of this kernel's bytes); and each unique sample's fiber, whose nonzeros are
// stamped (row-order positions: design row, step stamp) with their rows.  A
// workgroup takes kDesignRows design rows; the previously listed rows of factor j
// are cleared on the way.
constexpr int kDesignRows = 64;
__global__ __launch_bounds__(kT) void b64_design(const BatchTensor* __restrict__ ts, int j,
                                                 const BatchCtl* __restrict__ ctl) {
    const BatchTensor& T = ts[blockIdx.y];
    const int N = T.N, R = T.R;
    if (j >= N) return;
    const BatchMode& M = T.m[j];
    const uint32_t Ju = *gl(T.ju), c0 = blockIdx.x * kDesignRows, L = gl(T.cnt)[j];
    const int rows = kT / R, rl = threadIdx.x / R, r = threadIdx.x - rl * R;
    const Gp<double> Uj = gl(static_cast<double*>(M.U));
    if (rl < rows)
        for (uint32_t q = blockIdx.x * rows + rl; q < L; q += gridDim.x * rows) Uj[(int64_t)gl(M.list)[q] * R + r] = 0.0;
    if (c0 >= Ju) return;
    const uint32_t c1 = c0 + kDesignRows < Ju ? c0 + kDesignRows : Ju;
    if (rl < rows) {
        const Gp<double> dg = gl(static_cast<double*>(T.dg));
        for (uint32_t c = c0 + rl; c < c1; c += rows) {
            // every index, then every row entry, then the products in mode order
            uint32_t at[kMaxModes];
            double u[kMaxModes];
#pragma unroll
            for (int k = 0; k < kMaxModes; k++)
                if (k < N && k != j) at[k] = gl(T.sd)[(int64_t)c * N + k];
            const double wd = gl(T.wd)[c];
#pragma unroll
            for (int k = 0; k < kMaxModes; k++)
                if (k < N && k != j) u[k] = gl(static_cast<const double*>(T.m[k].U))[(int64_t)at[k] * R + r];
            double d = 1.0;
#pragma unroll
            for (int k = 0; k < kMaxModes; k++)
                if (k < N && k != j) d *= u[k];
            dg[(int64_t)c * R + r] = d * wd;
        }
    }
    if (threadIdx.x >= kDesignRows) return;       // one wavefront
    const uint32_t c = c0 + threadIdx.x, nf = (uint32_t)M.nfib;
    const uint32_t stamp = ctl->epoch * (uint32_t)N + (uint32_t)j + 1u;
    uint32_t hits = 0;
    if (c < c1 && nf > 0) {
        const uint64_t key = gl(T.kd)[c];
        const Gp<const uint64_t> fkey = gl(M.fkey);
        uint32_t b = 0;
        for (uint32_t len = nf; len > 1;) {
            const uint32_t half = len >> 1;
            b += fkey[b + half - 1] < key ? half : 0u;
            len -= half;
        }
        b += fkey[b] < key ? 1u : 0u;
        if (b < nf && fkey[b] == key) {
            const uint32_t e0 = gl(M.fptr)[b], e1 = gl(M.fptr)[b + 1];
            for (uint32_t e = e0; e < e1; e++) {
                const uint32_t p = gl(M.kpos)[e];
                gl(T.hu)[p] = c;
                gl(T.hstamp)[p] = stamp;
                gl(T.rstamp)[gl(M.rrow)[p]] = stamp;
            }
            hits = e1 - e0;
        }
    }
    const double h = wave_sum((double)hits);
    if (threadIdx.x == 0 && h > 0.0) atomicAdd(&T.stats[0], (unsigned long long)h);
}

// ---------------------------------------------------------------- Gram
typedef double f64x4 __attribute__((ext_vector_type(4)));

// x where the mask is all ones, 0 where it is zero.  (A select would let the
// compiler move the load under a branch and wait for each one.)
__device__ __forceinline__ double masked(double x, uint64_t mask) {
    return __longlong_as_double((long long)((uint64_t)__double_as_longlong(x) & mask));
}

// One (group, tile) of the Gram of A's rows (A, or A diag(1 / sig)) on one
// wavefront: v_mfma_f64_16x16x4 adds its four products one after the other with
// one rounding each, so a group's chain of instructions is the sum over its rows
// in order, as a chain of FMAs on one thread makes it.  Lane l holds column 16 t
// + l % 16 of the step's row l / 16; the loads of the next 16 steps (from memory that
// other XCDs wrote, about 2000 cycles) are in flight beside the products of these.
template <bool kScaled>
__device__ __forceinline__ void gram_item(Gp<const double> A, const double* sig, uint32_t rows, int R, int item,
                                          Gp<double> part) {
    constexpr int kU = 16;
    const int groups = gram_groups(R), tiles = R > 16 ? 3 : 1;
    const int g = item / tiles, tt = item - g * tiles;
    const int ta = tt == 2 ? 1 : 0, tb = tt == 0 ? 0 : 1;
    const int lane = threadIdx.x & 63, kr = lane >> 4, kc = lane & 15;
    const int ca = 16 * ta + kc, cb = 16 * tb + kc;
    const bool oka = ca < R, okb = cb < R;
    const double sa = kScaled && oka ? sig[ca] : 1.0, sb = kScaled && okb ? sig[cb] : 1.0;
    const uint32_t per = (uint32_t)(kChunkRows - g + groups - 1) / (uint32_t)groups;   // rows of a whole chunk
    const uint32_t full = rows / kChunkRows, tail = rows - full * kChunkRows;
    const uint32_t total = full * per + (tail > (uint32_t)g ? (tail - g + groups - 1) / groups : 0u);
    // The lane's next row is the at-th of the group's rows in its chunk; where the
    // groups divide a chunk, the group's rows are evenly apart and at is not needed.
    const bool even = kChunkRows % groups == 0;
    const Gp<const double> A0 = A + (oka ? ca : 0);
    const int to_b = (okb ? cb : 0) - (oka ? ca : 0);
    const int64_t step = (int64_t)4 * groups * R, skip = (int64_t)(kChunkRows - (int)per * groups) * R;
    uint32_t at = (uint32_t)kr;
    Gp<const double> p = A0 + ((int64_t)g + (int64_t)kr * groups) * R;
    auto settle = [&] {
        while (at >= per) {
            at -= per;
            p += skip;
        }
    };
    if (!even) settle();
    double xa[2][kU], xb[2][kU];
    // columns past R are any column: their sums are not stored
    auto load = [&](double (&ya)[kU], double (&yb)[kU], uint32_t st) {
        const bool whole = 4 * (st + kU) <= total;
#pragma unroll
        for (int u = 0; u < kU; u++) {
            const Gp<const double> q = whole || 4 * (st + u) + kr < total ? p : A0;
            ya[u] = q[0];
            yb[u] = q[to_b];
            p += step;
            if (!even) {
                at += 4;
                settle();
            }
        }
    };
    f64x4 acc = f64x4{0.0, 0.0, 0.0, 0.0};
    auto add = [&](const double (&ya)[kU], const double (&yb)[kU], uint32_t st) {
        if (4 * (st + kU) <= total) {
#pragma unroll
            for (int u = 0; u < kU; u++)
                acc = __builtin_amdgcn_mfma_f64_16x16x4f64(kScaled ? ya[u] / sa : ya[u], kScaled ? yb[u] / sb : yb[u],
                                                           acc, 0, 0, 0);
            return;
        }
#pragma unroll
        for (int u = 0; u < kU; u++) {
            const uint64_t in = 4 * (st + u) + kr < total ? ~0ull : 0ull;
            const double va = masked(kScaled ? ya[u] / sa : ya[u], in);
            const double vb = masked(kScaled ? yb[u] / sb : yb[u], in);
            acc = __builtin_amdgcn_mfma_f64_16x16x4f64(va, vb, acc, 0, 0, 0);
        }
    };
    const uint32_t steps = (total + 3) / 4;
    if (steps > 0) {
        load(xa[0], xb[0], 0);
        for (uint32_t st = 0; st < steps; st += 2 * kU) {
            load(xa[1], xb[1], st + kU);
            add(xa[0], xb[0], st);
            if (st + kU >= steps) break;
            load(xa[0], xb[0], st + 2 * kU);
            add(xa[1], xb[1], st + kU);
        }
    }
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int a = 16 * ta + 4 * i + kr, b = cb;
        if (a <= b && b < R) part[(int64_t)g * R * R + a * R + b] = acc[i];
    }
}

// The same sum for one group and entry (a, b) on one thread, item = group x
// tri_size(R) + entry: sixteen rows in flight, added in order.
template <bool kScaled>
__device__ __forceinline__ void gram_entry(Gp<const double> A, const double* sig, uint32_t rows, int R, int item,
                                           Gp<double> part) {
    constexpr int kU = 16;
    const int P = tri_size(R), groups = gram_groups(R), g = item / P;
    int b = item - g * P, a = 0;
    while (b >= R - a) {
        b -= R - a;
        a++;
    }
    b += a;
    const double sa = kScaled ? sig[a] : 1.0, sb = kScaled ? sig[b] : 1.0;
    uint32_t chunk = 0, at = (uint32_t)g;   // the group's next row is chunk + at
    double acc = 0.0;
    for (bool more = (uint32_t)g < rows; more;) {
        double x[kU], y[kU];
        bool in[kU];
#pragma unroll
        for (int u = 0; u < kU; u++) {
            const uint32_t r = chunk + at;
            in[u] = r < rows;
            const Gp<const double> q = A + (int64_t)(in[u] ? r : (uint32_t)g) * R;
            x[u] = q[a];
            y[u] = q[b];
            at += (uint32_t)groups;
            if (at >= (uint32_t)kChunkRows) {
                at = (uint32_t)g;
                chunk += kChunkRows;
            }
        }
#pragma unroll
        for (int u = 0; u < kU; u++) {
            const double s = fma(kScaled ? x[u] / sa : x[u], kScaled ? y[u] / sb : y[u], acc);
            acc = in[u] ? s : acc;
        }
        more = chunk + at < rows;
    }
    part[(int64_t)g * R * R + a * R + b] = acc;
}

// The workgroup's share (block of gram_blocks) of the group sums of a Gram.
// kLow: every Gram of the launch is summed by threads, so that the kernel does
// without the registers of gram_item (two workgroups a CU).
template <bool kScaled, bool kLow>
__device__ __forceinline__ void gram_share(Gp<const double> A, const double* sig, uint32_t rows, int R, int block,
                                           Gp<double> part) {
    if (kLow || gram_by_threads(R, rows)) {
        const int item = block * kT + (int)threadIdx.x;
        if (item < gram_live_groups(R) * tri_size(R)) gram_entry<kScaled>(A, sig, rows, R, item, part);
        return;
    }
    if constexpr (!kLow) {
        const int item = block * (kT / 64) + (int)(threadIdx.x >> 6);
        if (item < gram_items(R)) gram_item<kScaled>(A, sig, rows, R, item, part);
    }
}

// x[0] + x[stride] + ... (n terms, in order), sixteen loads ahead of the adds.
template <typename P>
__device__ __forceinline__ double sum_in_order(P x, int n, int stride) {
    constexpr int kU = 16;
    double t = 0.0;
    for (int q = 0; q < n; q += kU) {
        double v[kU];
#pragma unroll
        for (int u = 0; u < kU; u++) v[u] = x[(int64_t)(q + u < n ? q + u : n - 1) * stride];
#pragma unroll
        for (int u = 0; u < kU; u++) {
            const double s = t + v[u];
            t = q + u < n ? s : t;
        }
    }
    return t;
}

// Workgroup x: a share of the design Gram; the last one lists the rows that
// were stamped this step, ascending.
template <bool kLow>
__global__ __launch_bounds__(kT) void b64_gram_list(const BatchTensor* __restrict__ ts, int j,
                                                    const BatchCtl* __restrict__ ctl) {
    const BatchTensor& T = ts[blockIdx.y];
    if (j >= T.N) return;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    if (blockIdx.x + 1 < gridDim.x) {
        gram_share<false, kLow>(gl(static_cast<const double*>(T.dg)), nullptr, *gl(T.ju), T.R, (int)blockIdx.x, gl(T.gpart));
        return;
    }
    __shared__ uint32_t ws[2][kT / 64];
    const BatchMode& M = T.m[j];
    const uint32_t stamp = ctl->epoch * (uint32_t)T.N + (uint32_t)j + 1u;
    uint32_t run = 0;
    int buf = 0;
    for (int64_t c0 = 0; c0 < M.I; c0 += (int64_t)kT * kChunk, buf ^= 1) {
        const int64_t r0 = c0 + (int64_t)threadIdx.x * kChunk;
        uint32_t flags = 0;
#pragma unroll
        for (int q = 0; q < kChunk; q++)
            if (r0 + q < M.I && gl(T.rstamp)[r0 + q] == stamp) flags |= 1u << q;
        const uint32_t n = (uint32_t)__popc(flags);
        uint32_t inc = n;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const uint32_t y = __shfl_up(inc, d, 64);
            if (lane >= d) inc += y;
        }
        if (lane == 63) ws[buf][wave] = inc;
        __syncthreads();
        uint32_t off = run + inc - n, tot = 0;
#pragma unroll
        for (int q = 0; q < kT / 64; q++) {
            off += q < wave ? ws[buf][q] : 0u;
            tot += ws[buf][q];
        }
#pragma unroll
        for (int q = 0; q < kChunk; q++)
            if ((flags >> q) & 1u) gl(M.list)[off++] = (uint32_t)(r0 + q);
        run += tot;
    }
    if (threadIdx.x == 0) T.cnt[j] = run;
}

// ---------------------------------------------------------------- solves, MTTKRP
// Lanes per row of the row-wise phases: a power of two >= R, so that a row's lanes
// sit inside one wavefront.
__device__ __forceinline__ int row_lanes(int R) {
    int G = 1;
    while (G < R) G <<= 1;
    return G;
}

// Sampled MTTKRP (sort_lookup.hpp:238-375): Y row of each listed row = sum over
// its stamped positions, in row order, of x * (design row sqrt(w)).  The row's lanes
// test G positions at a time (one coalesced load of stamps); four of the hits
// among them are gathered at a time and added in ascending position.
__device__ __forceinline__ void mttkrp_rows(const BatchTensor& T, int j, uint32_t stamp, int block, int nblocks) {
    constexpr int kH = 4;
    const int R = T.R, G = row_lanes(R);
    const int rows = kT / G, rl = threadIdx.x / G, r = threadIdx.x - rl * G;
    const int gbase = (threadIdx.x & 63) - r;
    const uint64_t gmask = (1ull << G) - 1ull;
    const BatchMode& M = T.m[j];
    const Gp<const double> val = gl(static_cast<const double*>(M.rval)), dg = gl(static_cast<const double*>(T.dg));
    const Gp<double> Y = gl(static_cast<double*>(T.Yc));
    const uint32_t L = gl(T.cnt)[j];
    const int rc = r < R ? r : 0;
    for (uint32_t q0 = (uint32_t)block * rows; q0 < L; q0 += (uint32_t)nblocks * rows) {
        const uint32_t q = q0 + rl;
        uint32_t p0 = 0, p1 = 0;
        if (q < L) {
            const uint32_t row = gl(M.list)[q];
            p0 = gl(M.rowptr)[row];
            p1 = gl(M.rowptr)[row + 1];
        }
        double acc = 0.0;
        for (uint32_t p = p0; p < p1; p += G) {
            const uint32_t pp = p + r;
            const bool hit = pp < p1 && gl(T.hstamp)[pp] == stamp;
            const uint32_t hu = hit ? gl(T.hu)[pp] : 0u;
            const double hv = hit ? val[pp] : 0.0;
            uint64_t m = (__ballot(hit) >> gbase) & gmask;
            while (m) {
                bool on[kH];
                double x[kH], d[kH];
#pragma unroll
                for (int h = 0; h < kH; h++) {
                    on[h] = m != 0;
                    const int b = on[h] ? __ffsll((unsigned long long)m) - 1 : 0;
                    m &= m - 1;
                    const uint32_t u = (uint32_t)__shfl((int)hu, gbase + b, 64);
                    x[h] = __shfl(hv, gbase + b, 64);
                    d[h] = dg[(int64_t)u * R + rc] * gl(T.wd)[u];   // (row 0 where there is no hit: not used)
                }
#pragma unroll
                for (int h = 0; h < kH; h++) {
                    const double s = acc + x[h] * d[h];
                    acc = on[h] ? s : acc;
                }
            }
        }
        if (q < L && r < R) Y[(int64_t)q * R + r] = acc;
    }
}

// Workgroup 0: compute_pinv_square (common.h:405-443) of the Gram whose group sums
// are in gpart, eigenvalues <= 1e-11 dropped.  The others (with_y): the sampled
// MTTKRP, which the solve does not wait for.
__global__ __launch_bounds__(kT) void b64_solve(const BatchTensor* __restrict__ ts, int j,
                                                const BatchCtl* __restrict__ ctl) {
    const BatchTensor& T = ts[blockIdx.y];
    if (j >= T.N) return;
    if (blockIdx.x > 0) {
        mttkrp_rows(T, j, ctl->epoch * (uint32_t)T.N + (uint32_t)j + 1u, (int)blockIdx.x - 1, (int)gridDim.x - 1);
        return;
    }
    __shared__ EighSharedT<kBatchMaxRank> sh;
    const int R = T.R, groups = gram_live_groups(R);
    for (int o = threadIdx.x; o < R * R; o += kT) {
        const int a = o / R, b = o - a * R;
        if (a > b) continue;
        sh.A[tri_index(R, a, b)] = sum_in_order(gl((const double*)T.gpart) + o, groups, R * R);
    }
    __syncthreads();
    jacobi_block<kBatchMaxRank>(sh.A, sh.A2, sh.V, R, sh.j);
    pinv_from_jacobi(sh, R, 1e-11, T.gi);
}

// ---------------------------------------------------------------- factor update
// accumulator_stationary.hpp:280-289.  The rows Y Gi of the listed rows into Uc,
// and the squares of each column's classes of rows (norm_classes) into npart: a
// workgroup takes 256 / R classes.
__global__ __launch_bounds__(kT) void b64_update(const BatchTensor* __restrict__ ts, int j) {
    const BatchTensor& T = ts[blockIdx.y];
    if (j >= T.N) return;
    __shared__ double gi[kRR];
    const int R = T.R, classes = norm_classes(R), per = kT / R;
    if ((int)blockIdx.x * per >= classes) return;
    for (int o = threadIdx.x; o < R * R; o += kT) gi[o] = gl(T.gi)[o];
    __syncthreads();
    const int rl = threadIdx.x / R, r = threadIdx.x - rl * R, cl = (int)blockIdx.x * per + rl;
    if (rl >= per || cl >= classes) return;
    const uint32_t L = gl(T.cnt)[j];
    const Gp<const double> Y = gl(static_cast<const double*>(T.Yc));
    double ss = 0.0;
    for (uint32_t q = cl; q < L; q += classes) {
        double acc = 0.0;
#pragma unroll 8
        for (int b = 0; b < R; b++) acc += Y[(int64_t)q * R + b] * gi[b * R + r];
        gl(T.Uc)[(int64_t)q * R + r] = acc;
        ss += acc * acc;
    }
    T.npart[cl * R + r] = ss;
}

// sigma_c = the column norms; Gram of U_j = Uc diag(1 / sigma) over the listed
// rows (the others are zero) by the first gblocks workgroups, a share each; the
// workgroups past them write the rows of U_j.
template <bool kLow>
__global__ __launch_bounds__(kT) void b64_scale_gram(const BatchTensor* __restrict__ ts, int j, int gblocks) {
    const BatchTensor& T = ts[blockIdx.y];
    if (j >= T.N) return;
    __shared__ double sig[kBatchMaxRank], sums[kBatchNormPart];
    const int R = T.R;
    const uint32_t L = gl(T.cnt)[j];
    const int rows = kT / R, rl = threadIdx.x / R, r = threadIdx.x - rl * R;
    const int block = (int)blockIdx.x - gblocks, nblocks = (int)gridDim.x - gblocks;
    if (block < 0 && (int)blockIdx.x >= gram_blocks(R, L)) return;
    if (block > 0 && (uint32_t)block * rows >= L) return;
    for (int o = threadIdx.x; o < norm_classes(R) * R; o += kT) sums[o] = gl(T.npart)[o];
    __syncthreads();
    if (threadIdx.x < R) {
        const double sg = sqrt(sum_in_order((const double*)sums + threadIdx.x, norm_classes(R), R));
        if (block == 0) T.sigma[threadIdx.x] = sg;
        sig[threadIdx.x] = sg;
    }
    __syncthreads();
    if (block < 0) {
        gram_share<true, kLow>(gl((const double*)T.Uc), sig, L, R, (int)blockIdx.x, gl(T.gpart));
        return;
    }
    const Gp<double> U = gl(static_cast<double*>(T.m[j].U));
    if (rl < rows)
        for (uint32_t q = (uint32_t)block * rows + rl; q < L; q += (uint32_t)nblocks * rows)
            U[(int64_t)gl(T.m[j].list)[q] * R + r] = gl(T.Uc)[(int64_t)q * R + r] / sig[r];
}

// ---------------------------------------------------------------- sampler update
// cp_arls_lev.hpp:25-34: score of each listed row u^T Gp u, Gp = pinv(U_j^T U_j)
// (the row's lanes hold one entry each, t_c = sum_b u_b Gp[b][c] over broadcasts,
// then a butterfly sum of u_c t_c).
__global__ __launch_bounds__(kT) void b64_scores(const BatchTensor* __restrict__ ts, int j) {
    const BatchTensor& T = ts[blockIdx.y];
    if (j >= T.N) return;
    __shared__ double g[kRR];
    const int R = T.R, G = row_lanes(R);
    const int rows = kT / G, rl = threadIdx.x / G, r = threadIdx.x - rl * G;
    const uint32_t L = gl(T.cnt)[j];
    if (blockIdx.x * (uint32_t)rows >= L) return;
    for (int o = threadIdx.x; o < R * R; o += kT) g[o] = gl(T.gi)[o];
    __syncthreads();
    const int gbase = (threadIdx.x & 63) - r;
    const BatchMode& M = T.m[j];
    const Gp<const double> U = gl(static_cast<const double*>(M.U));
    const int rc = r < R ? r : 0;
    for (uint32_t q0 = blockIdx.x * (uint32_t)rows; q0 < L; q0 += gridDim.x * (uint32_t)rows) {
        const uint32_t q = q0 + rl;
        const double ac = (q < L && r < R) ? U[(int64_t)gl(M.list)[q] * R + r] : 0.0;
        double tc = 0.0;
        for (int b = 0; b < R; b++) tc += __shfl(ac, gbase + b, 64) * g[b * R + rc];
        double v = r < R ? ac * tc : 0.0;
        for (int off = G >> 1; off >= 1; off >>= 1) v += __shfl_xor(v, off, 64);
        if (q < L && r == 0) gl(M.csc)[q] = v;
    }
}

// Sum of the scores and the CDF of score / sum over the listed rows in ascending
// order (last entry 1): one workgroup per tensor.
__global__ __launch_bounds__(kBT) void b64_cdf(const BatchTensor* __restrict__ ts, int j) {
    const BatchTensor& T = ts[blockIdx.x];
    if (j >= T.N) return;
    __shared__ double wsd[kWaves];
    const BatchMode& M = T.m[j];
    const uint32_t L = gl(T.cnt)[j];
    // thread t sums the scores [t P, t P + P) in order, then the workgroup
    const uint32_t P = (L + kBT - 1) / kBT;
    double part = 0.0;
    for (uint32_t q = threadIdx.x * P, q1 = q + P < L ? q + P : L; q < q1; q++) part += M.csc[q];
    const double S = block_sum_f64(part, wsd);
    double carry = 0.0;
    for (uint32_t c0 = 0; c0 < L; c0 += kBT * kChunk) {
        const uint32_t q0 = c0 + threadIdx.x * kChunk;
        double loc[kChunk];
        double acc = 0.0;
#pragma unroll
        for (int q = 0; q < kChunk; q++) {
            acc += q0 + q < L ? M.csc[q0 + q] / S : 0.0;
            loc[q] = acc;
        }
        double tot = 0.0;
        const double off = carry + block_exscan_f64(acc, wsd, tot);
#pragma unroll
        for (int q = 0; q < kChunk; q++)
            if (q0 + q < L) M.ccdf[q0 + q] = q0 + q == L - 1 ? 1.0 : off + loc[q];
        carry += tot;
    }
    if (threadIdx.x == 0) {
        T.ssum[j] = S;
        atomicAdd(&T.stats[1], (unsigned long long)*T.ju);
        atomicAdd(&T.stats[2], (unsigned long long)L);
    }
}

__global__ void b64_advance(BatchCtl* ctl) {
    if (threadIdx.x != 0) return;
    ctl->sweep += 1;
    ctl->epoch += 1u;
}

}  // namespace

namespace k {

void batch_sweep64(hipStream_t s, const BatchTensor* ts, int n, int64_t J, BatchCtl* ctl, const BatchShape& shape) {
    EX_CHECK(J >= 1 && J <= kBatchMaxJ, 1, "batched sweep: J out of range");
    EX_CHECK(shape.R_max >= 1 && shape.R_max <= kBatchMaxRank && shape.R_min >= 1, 1, "batched sweep: rank out of range");
    int design_blocks = 1, factor_blocks = 1, norms = 1;   // (a Gram of the design's J rows, of a factor's)
    bool design_low = true, factor_low = true;
    for (int R = shape.R_min; R <= shape.R_max; R++) {
        design_blocks = std::max(design_blocks, gram_blocks_bound(R, J));
        factor_blocks = std::max(factor_blocks, gram_blocks_bound(R, shape.I_max));
        design_low = design_low && gram_by_threads(R, J);
        factor_low = factor_low && gram_by_threads(R, shape.I_max);
        norms = std::max(norms, (norm_classes(R) + kT / R - 1) / (kT / R));
    }
    // Workgroups of the row-wise phases: two rows a thread group for the longest
    // mode, up to 64 a tensor (a grid-stride loop takes the rest), and about 2048
    // in all: most tensors list few rows, and a workgroup that finds none still
    // takes its place (256 tensors: normalisation and Gram 108 -> 60 us).
    const unsigned rb = std::min(grid_for(shape.I_max, 16, 64), (unsigned)std::max(4, 2048 / std::max(n, 1)));
    const unsigned db = (unsigned)((J + kDesignRows - 1) / kDesignRows);
    for (int n0 = 0; n0 < n; n0 += 65535) {   // tensors are the grid's y
        const BatchTensor* t = ts + n0;
        const unsigned ny = (unsigned)std::min(n - n0, 65535);
        for (int j = 0; j < shape.N_max; j++) {
            hipLaunchKernelGGL(b64_draw, dim3(grid_for(J, kT), ny), dim3(kT), 0, s, t, j, J, ctl);
            hipLaunchKernelGGL(b64_dedup, dim3(ny), dim3(kBT), 0, s, t, j, J);
            hipLaunchKernelGGL(b64_design, dim3(db, ny), dim3(kT), 0, s, t, j, ctl);
            hipLaunchKernelGGL(design_low ? b64_gram_list<true> : b64_gram_list<false>,
                               dim3((unsigned)design_blocks + 1, ny), dim3(kT), 0, s, t, j, ctl);
            hipLaunchKernelGGL(b64_solve, dim3(1 + rb, ny), dim3(kT), 0, s, t, j, ctl);
            hipLaunchKernelGGL(b64_update, dim3((unsigned)norms, ny), dim3(kT), 0, s, t, j);
            hipLaunchKernelGGL(factor_low ? b64_scale_gram<true> : b64_scale_gram<false>,
                               dim3((unsigned)factor_blocks + rb, ny), dim3(kT), 0, s, t, j, factor_blocks);
            hipLaunchKernelGGL(b64_solve, dim3(1, ny), dim3(kT), 0, s, t, j, ctl);
            hipLaunchKernelGGL(b64_scores, dim3(rb, ny), dim3(kT), 0, s, t, j);
            hipLaunchKernelGGL(b64_cdf, dim3(ny), dim3(kBT), 0, s, t, j);
        }
    }
    hipLaunchKernelGGL(b64_advance, dim3(1), dim3(64), 0, s, ctl);
    EX_HIP(hipGetLastError());
}

}  // namespace k
}  // namespace exafac
