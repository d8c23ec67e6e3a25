// Workgroup helpers of the batched sweeps: fiber keys, searches, scans and sums.
#pragma once
#include "common.hpp"
#include "device.hpp"

namespace exafac {
namespace {

constexpr int kBT = 1024;                        // threads per workgroup
constexpr int kWaves = kBT / 64;
constexpr int kTableBits = 14;                   // deduplication slots: 2^14 >= 2 kBatchMaxJ
constexpr int kMaxQ = kBatchMaxJ / kBT;          // samples per thread at the largest J
constexpr int kLane = 8;                         // binary searches in flight per thread
constexpr int kChunk = 8;                        // entries per thread of a scan pass
constexpr int kRR = kBatchMaxRank * kBatchMaxRank;
static_assert(kBatchMaxJ * 2 <= (1 << kTableBits), "deduplication table load above 1/2");
static_assert(kBatchMaxJ < (1 << 16), "table entries pack a 16-bit index and a 16-bit count");

// A pointer out of a descriptor, known to be global memory (a generic one costs
// flat accesses, which wait for LDS as well).
template <typename T>
using Gp = __attribute__((address_space(1))) T*;
template <typename T>
__device__ __forceinline__ Gp<T> gl(T* p) {
    return (Gp<T>)p;
}

__device__ __forceinline__ uint64_t pack_key(const uint32_t* c, int N, const int* shift) {
    uint64_t key = 0;
    for (int k = 0; k < N; k++)
        if (shift[k] >= 0) key |= (uint64_t)c[k] << shift[k];
    return key;
}

__device__ __forceinline__ uint32_t table_slot(uint64_t key) {
    return (uint32_t)((key * 0x9E3779B97F4A7C15ull) >> (64 - kTableBits));
}

// Exclusive prefix over the workgroup (thread order) of one value per
// thread; *total receives the sum.  Two barriers.
__device__ uint32_t block_exscan_u32(uint32_t x, uint32_t* ws, uint32_t& total) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    uint32_t inc = x;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const uint32_t y = __shfl_up(inc, d, 64);
        if (lane >= d) inc += y;
    }
    if (lane == 63) ws[w] = inc;
    __syncthreads();
    uint32_t off = 0, tot = 0;
#pragma unroll
    for (int q = 0; q < kWaves; q++) {
        const uint32_t v = ws[q];
        off += q < w ? v : 0u;
        tot += v;
    }
    __syncthreads();
    total = tot;
    return off + inc - x;
}

__device__ double block_exscan_f64(double x, double* ws, double& total) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const double inc = wave_inclusive_scan(x, lane);
    if (lane == 63) ws[w] = inc;
    __syncthreads();
    double off = 0.0, tot = 0.0;
#pragma unroll
    for (int q = 0; q < kWaves; q++) {
        const double v = ws[q];
        if (q < w) off += v;
        tot += v;
    }
    __syncthreads();
    total = tot;
    return off + (inc - x);
}

// Sum over the workgroup, waves added in order (every thread gets it).
__device__ double block_sum_f64(double x, double* ws) {
    const double s = wave_sum(x);
    if ((threadIdx.x & 63) == 0) ws[threadIdx.x >> 6] = s;
    __syncthreads();
    double tot = 0.0;
#pragma unroll
    for (int q = 0; q < kWaves; q++) tot += ws[q];
    __syncthreads();
    return tot;
}

// lower_bound of u in the ascending array a[0, n) for kLane searches at
// once (every search takes ceil(log2 n) steps, their loads in flight
// together).  Result n when every entry is below u.
template <typename K>
__device__ __forceinline__ void lower_bounds(const K* __restrict__ a, uint32_t n, const K (&u)[kLane],
                                             uint32_t (&b)[kLane]) {
#pragma unroll
    for (int q = 0; q < kLane; q++) b[q] = 0;
    if (n == 0) return;
    for (uint32_t len = n; len > 1;) {
        const uint32_t half = len >> 1;
#pragma unroll
        for (int q = 0; q < kLane; q++) b[q] += a[b[q] + half - 1] < u[q] ? half : 0u;
        len -= half;
    }
#pragma unroll
    for (int q = 0; q < kLane; q++) b[q] += a[b[q]] < u[q] ? 1u : 0u;
}

}  // namespace
}  // namespace exafac
