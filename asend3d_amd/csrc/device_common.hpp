// Device-side helpers shared by the solve-path kernels: wavefront/block
// reductions, the deterministic last-block grid reduction and the XCD-aware
// block remap for gfx950 (256 CUs in 8 XCDs, 64-lane wavefronts).
#pragma once
#include <hip/hip_runtime.h>
#include <cstdint>

namespace asend {

constexpr int kWave = 64;
constexpr int kBlock = 256;  // threads per block for streaming kernels
constexpr int kNumXcd = 8;
constexpr int kMaxBlockWaves = 16;  // block reductions accept up to 1024 threads

// Element blocks of brick8 meshes by rows: record (e, a) holds the eight 3x3
// blocks K_ab (b = 0..7) of element e's row a, row-major, at 9 b of its
// kRecStride doubles (576 bytes, a multiple of 16); element e's records are
// contiguous, record (e, a) at kRecStride (8 e + a).  Record (e, a) is
// consumed by exactly one operator row (node conn[e][a]).
constexpr int kRecStride = 72;

// Logical block index such that each XCD (blocks are dispatched round-robin
// over the 8 XCDs) processes one contiguous range of logical blocks, so rows
// that share x-vector entries share an L2.
__device__ __forceinline__ int xcd_block(int b, int nb) {
    int per = (nb + kNumXcd - 1) / kNumXcd;
    int xcd = b % kNumXcd, idx = b / kNumXcd;
    int full = nb % kNumXcd == 0 ? kNumXcd : nb % kNumXcd;  // XCDs owning 'per' blocks
    // XCD x owns blocks x, x+8, ...; count of blocks owned by XCDs < xcd:
    int before = (xcd < full) ? xcd * per : full * per + (xcd - full) * (per - 1);
    return before + idx;
}

template <typename T>
__device__ __forceinline__ T wave_sum(T v) {
#pragma unroll
    for (int o = kWave / 2; o > 0; o >>= 1) v += __shfl_xor(v, o, kWave);
    return v;
}

template <typename T>
__device__ __forceinline__ T wave_max(T v) {
#pragma unroll
    for (int o = kWave / 2; o > 0; o >>= 1) {
        T w = __shfl_xor(v, o, kWave);
        v = v > w ? v : w;
    }
    return v;
}

// Sum of NV values over the whole block; result valid in thread 0.
template <int NV>
__device__ __forceinline__ void block_sum(double (&v)[NV]) {
    __shared__ double sh[NV][kMaxBlockWaves];
    int lane = threadIdx.x % kWave, w = threadIdx.x / kWave;
#pragma unroll
    for (int i = 0; i < NV; ++i) v[i] = wave_sum(v[i]);
    if (lane == 0)
#pragma unroll
        for (int i = 0; i < NV; ++i) sh[i][w] = v[i];
    __syncthreads();
    if (threadIdx.x == 0) {
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            double s = 0.0;
            for (int k = 0; k < (int)(blockDim.x / kWave); ++k) s += sh[i][k];
            v[i] = s;
        }
    }
    __syncthreads();
}

// A thread's share of n >= 1 partial sums of NV values, every blockDim.x-th (kBlock),
// K of them at a time in flight; added in order.
template <int NV, int K>
__device__ __forceinline__ void thread_sums_by(const double* __restrict__ partials, int n, double (&v)[NV]) {
    for (int b0 = 0; b0 < n; b0 += K * kBlock) {
        double t[K][NV];
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const int b = b0 + (int)threadIdx.x + k * kBlock;
#pragma unroll
            for (int i = 0; i < NV; ++i) t[k][i] = partials[(size_t)NV * min(b, n - 1) + i];
        }
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const bool in = b0 + (int)threadIdx.x + k * kBlock < n;
#pragma unroll
            for (int i = 0; i < NV; ++i) v[i] += in ? t[k][i] : 0.0;
        }
    }
}

// By the count, as reads past the end would be as many as those within it.  (A loop
// unrolled by the compiler takes what is left over its factor one by one: 2,048 sums
// and an update of 337,881 nodes 13.7 us, 12.1 us now; 516 and 132,098 rows 8.3 / 7.7 us.)
template <int NV>
__device__ __forceinline__ void thread_sums(const double* __restrict__ partials, int n, double (&v)[NV]) {
    if (n <= kBlock) thread_sums_by<NV, 1>(partials, n, v);
    else if (n <= 4 * kBlock) thread_sums_by<NV, 4>(partials, n, v);
    else thread_sums_by<NV, 8>(partials, n, v);
}

// Block-level partial sums for a two-kernel grid reduction: thread 0 of every
// block stores its NV sums at partials[NV*blockIdx.x + i]; a single-block
// finalize kernel launched next on the same stream combines them.
template <int NV>
__device__ __forceinline__ void block_partials(double (&v)[NV], double* partials) {
    block_sum<NV>(v);
    if (threadIdx.x == 0)
#pragma unroll
        for (int i = 0; i < NV; ++i) partials[(size_t)NV * blockIdx.x + i] = v[i];
}

// Block-level maximum of a non-negative value, same scheme.
__device__ __forceinline__ void block_partial_max(double v, double* partials) {
    __shared__ double sh[kMaxBlockWaves];
    v = wave_max(v);
    if (threadIdx.x % kWave == 0) sh[threadIdx.x / kWave] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        double m = 0.0;
        for (int k = 0; k < (int)(blockDim.x / kWave); ++k) m = m > sh[k] ? m : sh[k];
        partials[blockIdx.x] = m;
    }
}

}  // namespace asend
