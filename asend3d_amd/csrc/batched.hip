// Batched multi-right-hand-side PCG over many design variants.
//
// The operators of all variants (each assembled by its own context) are laid
// side by side as one block-diagonal sliced-ELL operator; every variant owns a
// 64-row-aligned range of block rows.  Up to kNrhs right-hand sides per variant
// advance together: one SpMM launch reads each 3x3 block once and applies it
// to all of them, and every reduction, coefficient and update is per
// (variant, rhs) system, so the whole batch costs the same number of launches
// per iteration as a single solve.  Inner solves are Jacobi PCG in FP32 inside
// FP64 iterative refinement (FP64 residual and update).
//
// Rows stand in an order of the batch's own (batch_row_order): 4 x 4 x 4 bricks of
// neighbouring nodes, one brick to a 64-row slice, whose 27 x 64 reads of X fall
// on about 216 rows.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <string>
#include <vector>

#include "asend_gpu.h"
#include "batched.hpp"
#include "device_common.hpp"
#include "kernels.hpp"

namespace asend {

namespace {

// An iteration is three launches that pass the vectors ten times: the product (P, Q)
// with p.q, the residual's update (Q, R twice) with z.q and r.r, and the
// direction (R, X and P twice), which also makes the solution's update, whose P
// it reads anyway, and p.r.  Their workgroups add up their variant's partial
// sums of the launch before themselves, so a variant has at most kVarParts workgroups
// in the product (of one slice or more) and kVarChunks row chunks (of 128 rows
// or more): 64 kB of partials per workgroup at the most.
constexpr int kVarParts = 512;
constexpr int kVarChunks = 256;
constexpr int kChunkRows = 128;

// What a workgroup of the product works on, and one of the vector kernels: in one
// load, since its fields name everything else.  Within a variant the workgroups of
// an XCD own one contiguous piece (over all variants at once, the XCDs of those
// that have converged would stand idle: 40.0 against 33.0 us for the product).
struct alignas(16) BlkInfo {
    int32_t slice0, slice1;  // slices [slice0, slice1)
    int32_t seg;             // variant
    int32_t out;             // index of the partials
};
struct alignas(16) ChunkInfo {
    int32_t row0, row1;      // rows [row0, row1)
    int32_t seg, out;
    int32_t chunk0, chunk1;  // the variant's chunks
    int32_t blk0, blk1;      // and its workgroups of the product
};

// FP64 residual R = F - K U of 8 right-hand sides; vectors are [row][3][kNrhs]; a
// wavefront takes a slice, a lane a row.
__global__ __launch_bounds__(kBlock) void k_mrhs_residual(int n_slices, const int32_t* __restrict__ sptr,
                                                          const int32_t* __restrict__ scol,
                                                          const double* __restrict__ val, const double* __restrict__ U,
                                                          double* __restrict__ R, const double* __restrict__ F,
                                                          int j0) {
    const int slice = blockIdx.x * (kBlock / kWave) + threadIdx.x / kWave;
    const int rl = threadIdx.x % kWave;
    if (slice >= n_slices) return;
    double acc[3][8];
#pragma unroll
    for (int d = 0; d < 3; ++d)
#pragma unroll
        for (int j = 0; j < 8; ++j) acc[d][j] = 0.0;
    const int k0 = sptr[slice], k1 = sptr[slice + 1];
    const int32_t* cp = scol + (int64_t)k0 * kWave + rl;
    const double* vp = val + (int64_t)k0 * 9 * kWave + rl;
    for (int k = k0; k < k1; ++k) {
        // values and columns streamed once: non-temporal, keeping U in L2
        const int64_t c = __builtin_nontemporal_load(cp);
        double a[9];
#pragma unroll
        for (int q = 0; q < 9; ++q) a[q] = __builtin_nontemporal_load(vp + q * kWave);
        const double* xc = U + c * 3 * kNrhs + j0;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const double x0 = xc[j], x1 = xc[kNrhs + j], x2 = xc[2 * kNrhs + j];
            acc[0][j] += a[0] * x0 + a[1] * x1 + a[2] * x2;
            acc[1][j] += a[3] * x0 + a[4] * x1 + a[5] * x2;
            acc[2][j] += a[6] * x0 + a[7] * x1 + a[8] * x2;
        }
        cp += kWave;
        vp += 9 * kWave;
    }
    const int64_t o = ((int64_t)slice * kWave + rl) * 3 * kNrhs + j0;
#pragma unroll
    for (int d = 0; d < 3; ++d)
#pragma unroll
        for (int j = 0; j < 8; ++j) R[o + d * kNrhs + j] = F[o + d * kNrhs + j] - acc[d][j];
}

// v of lane I of the own group of four lanes
template <int I>
__device__ __forceinline__ float quad_lane(float v) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), I * 0x55, 0xf, 0xf, true));
}

// Q = K P of all right-hand sides with the partials of P.Q per system: a workgroup
// takes slices of one variant, its four wavefronts 16 rows of each, four lanes a
// row, each with four right-hand sides.  Variants whose systems have all
// converged are skipped.
// Bound by the L1 accesses.  With a row's values component by component (9 loads
// of which the four lanes of a row read the same word) a slot cost about 240 of
// them per wavefront, 33.0 us for 56,512 rows (4 variants, brick order); values
// of a block together, one row of it in each of three lanes and passed
// between the four, 21.4 us (61 MB of values: 12.6 us at the rate of a copy).  Two groups of kSlotsAtOnce slots are in
// flight, the columns of a third.
constexpr int kLanesPerRow = 4;
constexpr int kSlotsAtOnce = 3;
__global__ __launch_bounds__(kBlock) void k_mrhs_dir_product(
    const BlkInfo* __restrict__ info, const int32_t* __restrict__ sptr, const int32_t* __restrict__ scol,
    const float* __restrict__ val, const float* __restrict__ P, float* __restrict__ Q,
    const uint8_t* __restrict__ active, double* __restrict__ partials) {
    constexpr int RPW = kWave / kLanesPerRow, NRL = kNrhs / kLanesPerRow, U = kSlotsAtOnce;
    constexpr int kWaves = kBlock / kWave;
    static_assert(kWaves * RPW == kWave && NRL == 4, "a workgroup is a slice, a lane's values one load");
    __shared__ double sh[kWaves][kNrhs];
    const BlkInfo I = info[blockIdx.x];
    if (!active[I.seg]) return;
    const int lane = threadIdx.x % kWave, w = threadIdx.x / kWave;
    const int rl = w * RPW + lane / kLanesPerRow, q = lane % kLanesPerRow, jq = q * NRL;
    const int kq = 9 * rl + 3 * (q < 3 ? q : 2);
    double t[NRL];
#pragma unroll
    for (int j = 0; j < NRL; ++j) t[j] = 0.0;
    for (int slice = I.slice0; slice < I.slice1; ++slice) {
        float acc[3][NRL];
#pragma unroll
        for (int d = 0; d < 3; ++d)
#pragma unroll
            for (int j = 0; j < NRL; ++j) acc[d][j] = 0.f;
        const int k0 = sptr[slice], n = sptr[slice + 1] - k0, groups = n / U;
        const int32_t* cp = scol + (int64_t)k0 * kWave + rl;
        const float* vp = val + (int64_t)k0 * 9 * kWave + kq;
        // group g's columns, values and X (slots past the end: the last one's)
        auto columns = [&](int g, int32_t (&c)[U]) {
#pragma unroll
            for (int u = 0; u < U; ++u) c[u] = cp[min(g * U + u, n - 1) * kWave];
        };
        auto values = [&](int g, float (&a)[U][3]) {
#pragma unroll
            for (int u = 0; u < U; ++u)
#pragma unroll
                for (int i = 0; i < 3; ++i) a[u][i] = vp[min(g * U + u, n - 1) * 9 * kWave + i];
        };
        auto fetch = [&](const int32_t (&c)[U], float (&x)[U][3][NRL]) {
#pragma unroll
            for (int u = 0; u < U; ++u)
#pragma unroll
                for (int d = 0; d < 3; ++d) {
                    const float4 f = *reinterpret_cast<const float4*>(P + ((int64_t)c[u] * 3 + d) * kNrhs + jq);
                    x[u][d][0] = f.x, x[u][d][1] = f.y, x[u][d][2] = f.z, x[u][d][3] = f.w;
                }
        };
        auto add = [&](const float (&a)[3], const float (&x)[3][NRL]) {
#pragma unroll
            for (int j = 0; j < 3; ++j) {
                const float m0 = quad_lane<0>(a[j]), m1 = quad_lane<1>(a[j]), m2 = quad_lane<2>(a[j]);
#pragma unroll
                for (int r = 0; r < NRL; ++r) {
                    acc[0][r] += m0 * x[j][r];
                    acc[1][r] += m1 * x[j][r];
                    acc[2][r] += m2 * x[j][r];
                }
            }
        };
        if (n > 0) {
            int32_t c[U];
            float a[U][3], x[U][3][NRL];
            columns(0, c);
            values(0, a);
            fetch(c, x);
            columns(1, c);
#pragma unroll 2
            for (int g = 0; g < groups; ++g) {
                float an[U][3], xn[U][3][NRL];
                values(g + 1, an);
                fetch(c, xn);
                columns(g + 2, c);
#pragma unroll
                for (int u = 0; u < U; ++u) add(a[u], x[u]);
#pragma unroll
                for (int u = 0; u < U; ++u)
#pragma unroll
                    for (int d = 0; d < 3; ++d) {
                        a[u][d] = an[u][d];
#pragma unroll
                        for (int r = 0; r < NRL; ++r) x[u][d][r] = xn[u][d][r];
                    }
            }
            // the slots of the last, partial group
#pragma unroll
            for (int u = 0; u < U - 1; ++u)
                if (groups * U + u < n) add(a[u], x[u]);
        }
        const int64_t o = ((int64_t)slice * kWave + rl) * 3 * kNrhs + jq;
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            const float4 p = *reinterpret_cast<const float4*>(P + o + d * kNrhs);
            *reinterpret_cast<float4*>(Q + o + d * kNrhs) = make_float4(acc[d][0], acc[d][1], acc[d][2], acc[d][3]);
            t[0] += (double)p.x * acc[d][0];
            t[1] += (double)p.y * acc[d][1];
            t[2] += (double)p.z * acc[d][2];
            t[3] += (double)p.w * acc[d][3];
        }
    }
#pragma unroll
    for (int m = kLanesPerRow; m < kWave; m <<= 1)
#pragma unroll
        for (int j = 0; j < NRL; ++j) t[j] += __shfl_xor(t[j], m, kWave);
    if (lane < kLanesPerRow)
#pragma unroll
        for (int j = 0; j < NRL; ++j) sh[w][jq + j] = t[j];
    __syncthreads();
    if (threadIdx.x < kNrhs) {
        double sum = 0.0;
#pragma unroll
        for (int k = 0; k < kWaves; ++k) sum += sh[k][threadIdx.x];
        partials[(int64_t)I.out * kNrhs + threadIdx.x] = sum;
    }
}

// Per-system scalars, index s = variant * kNrhs + j
enum { B_RZ = 0, B_PQ, B_ALPHA, B_BETA, B_RR, B_RR0, B_IT, B_DONE, B_MAXIT, B_TOL2, B_N };

// Chunk reduction of the FP64 residual: each block owns rows [row0, row1) of
// one variant and accumulates, per rhs j, |r|^2 into partials[chunk][0][j].
__global__ __launch_bounds__(256) void k_chunk_rr64(const int32_t* __restrict__ chunk_row,
                                                    const double* __restrict__ a, double* __restrict__ partials) {
    __shared__ double sh[256];
    const int ch = blockIdx.x;
    const int j = threadIdx.x % kNrhs;
    const int64_t e0 = (int64_t)chunk_row[ch] * 3, e1 = (int64_t)chunk_row[ch + 1] * 3;
    double t = 0.0;
#pragma unroll 4
    for (int64_t e = e0 + threadIdx.x / kNrhs; e < e1; e += 256 / kNrhs) {
        const int64_t i = e * kNrhs + j;
        t += a[i] * a[i];
    }
    sh[threadIdx.x] = t;
    __syncthreads();
    for (int s = 128; s >= kNrhs; s >>= 1) {
        if (threadIdx.x < s) sh[threadIdx.x] += sh[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x < kNrhs) partials[(int64_t)ch * 2 * kNrhs + threadIdx.x] = sh[threadIdx.x];
}

// Sums of the NV values per system over the partials [c0, c1) of a variant, at
// most MAX of them, in the same order in every workgroup: load() has all of a
// thread's reads (two values each) in flight, finish() adds them up, res
// standing for all threads after the next barrier.
template <int NV, int MAX>
struct VarSums {
    static constexpr int kCols = NV * kNrhs, kPairs = kCols / 2, kLanes = 256 / kPairs, kReads = MAX / kLanes;
    static_assert(MAX % kLanes == 0, "whole reads");
    double2 v[kReads];
    __device__ __forceinline__ void load(const double* __restrict__ partials, int c0, int c1) {
        const int col = threadIdx.x % kPairs, q = threadIdx.x / kPairs;
#pragma unroll
        for (int k = 0; k < kReads; ++k) {
            const int c = c0 + q + k * kLanes;
            v[k] = *reinterpret_cast<const double2*>(partials + (int64_t)min(c, c1 - 1) * kCols + 2 * col);
            if (c >= c1) v[k].x = v[k].y = 0.0;
        }
    }
    // sh: [2 * 256]
    __device__ __forceinline__ void finish(double* sh, double (&res)[NV][kNrhs]) {
#pragma unroll
        for (int k = 1; k < kReads; ++k) {
            v[0].x += v[k].x;
            v[0].y += v[k].y;
        }
        reinterpret_cast<double2*>(sh)[threadIdx.x] = v[0];
        __syncthreads();
        if (threadIdx.x < kCols) {
            double t = 0.0;
#pragma unroll
            for (int k = 0; k < kLanes; ++k) t += sh[k * kCols + threadIdx.x];
            (&res[0][0])[threadIdx.x] = t;
        }
    }
};

// A workgroup's sums of threads' values for right-hand sides 4 (t % 4) + j to its
// partials (sh: no longer read by others).
template <int NV>
__device__ __forceinline__ void chunk_partials(double (&t)[NV][4], double* sh, double* __restrict__ out) {
#pragma unroll
    for (int m = 4; m < kWave; m <<= 1)
#pragma unroll
        for (int i = 0; i < NV; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) t[i][j] += __shfl_xor(t[i][j], m, kWave);
    if (threadIdx.x % kWave < 4)
#pragma unroll
        for (int i = 0; i < NV; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j)
                sh[((threadIdx.x / kWave) * NV + i) * kNrhs + 4 * (threadIdx.x % 4) + j] = t[i][j];
    __syncthreads();
    if (threadIdx.x < NV * kNrhs) {
        double sum = 0.0;
#pragma unroll
        for (int k = 0; k < 256 / kWave; ++k) sum += sh[k * NV * kNrhs + threadIdx.x];
        out[threadIdx.x] = sum;
    }
}

__device__ __forceinline__ void load4(const float4* __restrict__ a, int64_t i, float (&v)[4]) {
    const float4 f = a[i];
    v[0] = f.x, v[1] = f.y, v[2] = f.z, v[3] = f.w;
}

// p.r at the start and after a reliable update
__global__ __launch_bounds__(256) void k_chunk_pr(const int32_t* __restrict__ chunk_row, const float4* __restrict__ P,
                                                  const float4* __restrict__ R, double* __restrict__ partials) {
    __shared__ double sh[256];
    const int ch = blockIdx.x, jq = threadIdx.x % 4;
    double t[1][4] = {{0.0, 0.0, 0.0, 0.0}};
    const int64_t e0 = (int64_t)chunk_row[ch] * 3, e1 = (int64_t)chunk_row[ch + 1] * 3;
    for (int64_t e = e0 + threadIdx.x / 4; e < e1; e += 64) {
        float p[4], r[4];
        load4(P, e * 4 + jq, p);
        load4(R, e * 4 + jq, r);
#pragma unroll
        for (int j = 0; j < 4; ++j) t[0][j] += (double)p[j] * r[j];
    }
    chunk_partials<1>(t, sh, partials + (int64_t)ch * kNrhs);
}

// Rows of a chunk in registers at once: 6 DOFs a thread cover kChunkRows rows.  They
// are on their way while the sums before them are added.
constexpr int kAtOnce = 3 * kChunkRows / 64;

// alpha = p.r / p.q; r -= alpha q ; partials of (Dinv r).q and r.r (FP32 inner).
// out: the scalars with alpha, another slot than in (which other workgroups
// still read); going: the flags as this iteration finds them.  A thread takes
// four right-hand sides of a DOF.
// 56,512 rows: this and the solution's update 14.4 us, 10.7 us for the dots' pass
// and 4.4 us for the sums' launch; 9.9 us now.
__global__ __launch_bounds__(256) void k_chunk_update(const ChunkInfo* __restrict__ info,
                                                      const float* __restrict__ dinv, float4* __restrict__ R,
                                                      const float4* __restrict__ Q, const double* __restrict__ pq,
                                                      const double* __restrict__ pr, const double* __restrict__ in,
                                                      double* __restrict__ out, double* __restrict__ partials,
                                                      const uint8_t* __restrict__ active,
                                                      uint8_t* __restrict__ going) {
    __shared__ double sh[2][512], pqs[1][kNrhs], prs[1][kNrhs], sv[kNrhs * B_N];
    const ChunkInfo I = info[blockIdx.x];
    const bool lead = I.out == I.chunk0, go = active[I.seg] != 0;
    if (lead && threadIdx.x == 0) going[I.seg] = go;
    if (!go) return;
    const int jq = threadIdx.x % 4;
    const int64_t e1 = (int64_t)I.row1 * 3;
    int64_t e = (int64_t)I.row0 * 3 + threadIdx.x / 4;
    float r[kAtOnce][4], q[kAtOnce][4], di[kAtOnce];
    auto load = [&]() {
#pragma unroll
        for (int u = 0; u < kAtOnce; ++u) {
            const int64_t eu = min(e + 64 * u, e1 - 1), i = eu * (kNrhs / 4) + jq;
            load4(R, i, r[u]);
            load4(Q, i, q[u]);
            di[u] = dinv[eu];
        }
    };
    const int64_t base = (int64_t)I.seg * kNrhs * B_N;
    if (threadIdx.x < kNrhs * B_N) sv[threadIdx.x] = in[base + threadIdx.x];
    VarSums<1, kVarParts> sum_pq;
    VarSums<1, kVarChunks> sum_pr;
    sum_pq.load(pq, I.blk0, I.blk1);
    sum_pr.load(pr, I.chunk0, I.chunk1);
    load();
    sum_pq.finish(sh[0], pqs);
    sum_pr.finish(sh[1], prs);
    __syncthreads();
    if (threadIdx.x < kNrhs) {
        double* v = sv + threadIdx.x * B_N;
        if (v[B_DONE] == 0.0) {
            v[B_PQ] = pqs[0][threadIdx.x];
            v[B_ALPHA] = prs[0][threadIdx.x] / pqs[0][threadIdx.x];
        }
    }
    __syncthreads();
    if (lead && threadIdx.x < kNrhs * B_N) out[base + threadIdx.x] = sv[threadIdx.x];
    float alpha[4];
    bool on[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const double* v = sv + (4 * jq + j) * B_N;
        on[j] = v[B_DONE] == 0.0;
        alpha[j] = (float)v[B_ALPHA];
    }
    double t[2][4];
#pragma unroll
    for (int j = 0; j < 4; ++j) t[0][j] = t[1][j] = 0.0;
    for (;;) {
#pragma unroll
        for (int u = 0; u < kAtOnce; ++u) {
            if (e + 64 * u >= e1) break;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                if (!on[j]) continue;
                r[u][j] -= alpha[j] * q[u][j];
                t[0][j] += (double)(di[u] * r[u][j]) * q[u][j];
                t[1][j] += (double)r[u][j] * r[u][j];
            }
            R[(e + 64 * u) * (kNrhs / 4) + jq] = make_float4(r[u][0], r[u][1], r[u][2], r[u][3]);
        }
        e += 64 * kAtOnce;
        if (e >= e1) break;
        load();
    }
    chunk_partials<2>(t, sh[0], partials + (int64_t)I.out * 2 * kNrhs);
}

// x += alpha p; beta = -z.q / p.q, convergence of r.r, p = Dinv r + beta p and the
// partials of the new p.r; out: the scalars of the next iteration, active[v]: some
// system of the variant goes on.
// 56,512 rows: without the solution's update 11.0 us and 8 us for the sums' and the
// flags' launches; 9.8 us now.
__global__ __launch_bounds__(256) void k_chunk_dir(const ChunkInfo* __restrict__ info, const float* __restrict__ dinv,
                                                   const float4* __restrict__ R, float4* __restrict__ P,
                                                   float4* __restrict__ X, const double* __restrict__ partials,
                                                   const double* __restrict__ in, double* __restrict__ out,
                                                   double* __restrict__ pr, const uint8_t* __restrict__ going,
                                                   uint8_t* __restrict__ active) {
    __shared__ double sh[512], res[2][kNrhs], sv[kNrhs * B_N];
    const ChunkInfo I = info[blockIdx.x];
    if (!going[I.seg]) return;
    const int jq = threadIdx.x % 4;
    const int64_t e1 = (int64_t)I.row1 * 3;
    int64_t e = (int64_t)I.row0 * 3 + threadIdx.x / 4;
    float r[kAtOnce][4], p[kAtOnce][4], x[kAtOnce][4], di[kAtOnce];
    auto load = [&]() {
#pragma unroll
        for (int u = 0; u < kAtOnce; ++u) {
            const int64_t eu = min(e + 64 * u, e1 - 1), i = eu * (kNrhs / 4) + jq;
            load4(R, i, r[u]);
            load4(P, i, p[u]);
            load4(X, i, x[u]);
            di[u] = dinv[eu];
        }
    };
    const int64_t base = (int64_t)I.seg * kNrhs * B_N;
    if (threadIdx.x < kNrhs * B_N) sv[threadIdx.x] = in[base + threadIdx.x];
    VarSums<2, kVarChunks> sums;
    sums.load(partials, I.chunk0, I.chunk1);
    load();
    sums.finish(sh, res);
    __syncthreads();
    float alpha[4], beta[4];
    bool was[4], on[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const double* v = sv + (4 * jq + j) * B_N;
        was[j] = v[B_DONE] == 0.0;
        alpha[j] = (float)v[B_ALPHA];
    }
    __syncthreads();
    if (threadIdx.x < kNrhs) {
        double* v = sv + threadIdx.x * B_N;
        const double zq = res[0][threadIdx.x], rr = res[1][threadIdx.x];
        if (v[B_DONE] == 0.0) {
            v[B_BETA] = -zq / v[B_PQ];
            v[B_RR] = rr;
            v[B_IT] += 1.0;
            if (rr <= v[B_TOL2] * v[B_RR0] || v[B_IT] >= v[B_MAXIT] || !(rr == rr)) v[B_DONE] = 1.0;
        }
    }
    __syncthreads();
    if (I.out == I.chunk0) {
        if (threadIdx.x < kNrhs * B_N) out[base + threadIdx.x] = sv[threadIdx.x];
        if (threadIdx.x == 0) {
            uint8_t a = 0;
            for (int j = 0; j < kNrhs; ++j) a |= sv[j * B_N + B_DONE] == 0.0 ? 1 : 0;
            active[I.seg] = a;
        }
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const double* v = sv + (4 * jq + j) * B_N;
        on[j] = v[B_DONE] == 0.0;
        beta[j] = (float)v[B_BETA];
    }
    double t[1][4] = {{0.0, 0.0, 0.0, 0.0}};
    for (;;) {
#pragma unroll
        for (int u = 0; u < kAtOnce; ++u) {
            if (e + 64 * u >= e1) break;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                if (was[j]) x[u][j] += alpha[j] * p[u][j];
                if (!on[j]) continue;
                p[u][j] = di[u] * r[u][j] + beta[j] * p[u][j];
                t[0][j] += (double)p[u][j] * r[u][j];
            }
            const int64_t i = (e + 64 * u) * (kNrhs / 4) + jq;
            X[i] = make_float4(x[u][0], x[u][1], x[u][2], x[u][3]);
            P[i] = make_float4(p[u][0], p[u][1], p[u][2], p[u][3]);
        }
        e += 64 * kAtOnce;
        if (e >= e1) break;
        load();
    }
    chunk_partials<1>(t, sh, pr + (int64_t)I.out * kNrhs);
}

// r = b, x = 0, p = Dinv r; partials of r.z and r.r
__global__ __launch_bounds__(256) void k_chunk_init(const int32_t* __restrict__ chunk_row,
                                                    const float* __restrict__ dinv, const float* __restrict__ B,
                                                    float* __restrict__ X, float* __restrict__ R,
                                                    float* __restrict__ P, double* __restrict__ partials) {
    __shared__ double sh[2][256];
    const int ch = blockIdx.x;
    const int j = threadIdx.x % kNrhs;
    const int64_t e0 = (int64_t)chunk_row[ch] * 3, e1 = (int64_t)chunk_row[ch + 1] * 3;
    double t0 = 0.0, t1 = 0.0;
#pragma unroll 4
    for (int64_t e = e0 + threadIdx.x / kNrhs; e < e1; e += 256 / kNrhs) {
        const int64_t i = e * kNrhs + j;
        const float bi = B[i], zi = dinv[e] * bi;
        X[i] = 0.f;
        R[i] = bi;
        P[i] = zi;
        t0 += (double)bi * zi;
        t1 += (double)bi * bi;
    }
    sh[0][threadIdx.x] = t0;
    sh[1][threadIdx.x] = t1;
    __syncthreads();
    for (int k = 128; k >= kNrhs; k >>= 1) {
        if (threadIdx.x < k) {
            sh[0][threadIdx.x] += sh[0][threadIdx.x + k];
            sh[1][threadIdx.x] += sh[1][threadIdx.x + k];
        }
        __syncthreads();
    }
    if (threadIdx.x < kNrhs) {
        partials[(int64_t)ch * 2 * kNrhs + threadIdx.x] = sh[0][threadIdx.x];
        partials[(int64_t)ch * 2 * kNrhs + kNrhs + threadIdx.x] = sh[1][threadIdx.x];
    }
}

// partials of r.(Dinv r) and r.r (after a reliable update reloaded r)
__global__ __launch_bounds__(256) void k_chunk_rz(const int32_t* __restrict__ chunk_row,
                                                  const float* __restrict__ dinv, const float* __restrict__ R,
                                                  double* __restrict__ partials) {
    __shared__ double sh[2][256];
    const int ch = blockIdx.x;
    const int j = threadIdx.x % kNrhs;
    const int64_t e0 = (int64_t)chunk_row[ch] * 3, e1 = (int64_t)chunk_row[ch + 1] * 3;
    double t0 = 0.0, t1 = 0.0;
#pragma unroll 4
    for (int64_t e = e0 + threadIdx.x / kNrhs; e < e1; e += 256 / kNrhs) {
        const float ri = R[e * kNrhs + j];
        t0 += (double)ri * (dinv[e] * ri);
        t1 += (double)ri * ri;
    }
    sh[0][threadIdx.x] = t0;
    sh[1][threadIdx.x] = t1;
    __syncthreads();
    for (int k = 128; k >= kNrhs; k >>= 1) {
        if (threadIdx.x < k) {
            sh[0][threadIdx.x] += sh[0][threadIdx.x + k];
            sh[1][threadIdx.x] += sh[1][threadIdx.x + k];
        }
        __syncthreads();
    }
    if (threadIdx.x < kNrhs) {
        partials[(int64_t)ch * 2 * kNrhs + threadIdx.x] = sh[0][threadIdx.x];
        partials[(int64_t)ch * 2 * kNrhs + kNrhs + threadIdx.x] = sh[1][threadIdx.x];
    }
}

// Per-system finalize over the chunks of its variant: one workgroup per
// variant; the 256 / kNrhs lanes of each right-hand side add a strided share
// of the chunks, then a fixed-order tree over those lanes (deterministic).
// The inner solves are flexible CG (one truncation vector): alpha = p.r / p.q
// and beta = -z.q / p.q from fresh inner products, so a residual replaced by
// a reliable update needs no repair of the recurrence.
//   OP 0 (init):   rz, rr0 = rr, it = 0, done when rr0 = 0 or the system is frozen
//   OP 3 (|r|^2):  rr (FP64 residual norm) into out[s]
//   OP 4 (reliable update): rz, rr = rr0 of the reloaded residual, tol2 =
//                  out[s], the iteration count kept; done when frozen or r = 0
__global__ __launch_bounds__(256) void k_sys_fin(const int32_t* __restrict__ seg_chunk,
                                                 const double* __restrict__ partials, int op,
                                                 double* __restrict__ sv, const uint8_t* __restrict__ frozen,
                                                 double* __restrict__ out) {
    __shared__ double sh[2][256];
    const int seg = blockIdx.x;
    const int j = threadIdx.x % kNrhs, q = threadIdx.x / kNrhs;
    const int s = seg * kNrhs + j;
    double* v = sv + (int64_t)s * B_N;
    double t0 = 0.0, t1 = 0.0;
    for (int ch = seg_chunk[seg] + q; ch < seg_chunk[seg + 1]; ch += 256 / kNrhs) {
        t0 += partials[(int64_t)ch * 2 * kNrhs + j];
        t1 += partials[(int64_t)ch * 2 * kNrhs + kNrhs + j];
    }
    sh[0][threadIdx.x] = t0;
    sh[1][threadIdx.x] = t1;
    __syncthreads();
    for (int w = 128; w >= kNrhs; w >>= 1) {
        if (threadIdx.x < w) {
            sh[0][threadIdx.x] += sh[0][threadIdx.x + w];
            sh[1][threadIdx.x] += sh[1][threadIdx.x + w];
        }
        __syncthreads();
    }
    if (q != 0) return;
    t0 = sh[0][j];
    t1 = sh[1][j];
    if (op == 0) {
        v[B_RZ] = t0;
        v[B_RR] = t1;
        v[B_RR0] = t1;
        v[B_IT] = 0.0;
        v[B_DONE] = (frozen[s] || t1 == 0.0) ? 1.0 : 0.0;
    } else if (op == 4) {
        v[B_RZ] = t0;
        v[B_RR] = t1;
        v[B_RR0] = t1;
        v[B_TOL2] = out[s];
        v[B_DONE] = (frozen[s] || t1 == 0.0 || v[B_IT] >= v[B_MAXIT]) ? 1.0 : 0.0;
    } else {
        out[s] = t0;
    }
}

// active[v] = some system of variant v still iterating
__global__ void k_var_active(int n_var, const double* __restrict__ sv, uint8_t* __restrict__ active) {
    const int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= n_var) return;
    uint8_t a = 0;
    for (int j = 0; j < kNrhs; ++j) a |= (sv[(int64_t)(v * kNrhs + j) * B_N + B_DONE] == 0.0) ? 1 : 0;
    active[v] = a;
}

// FP64 residual -> FP32 inner right-hand side, scaled per system by 1/||r||
__global__ void k_mr_to_f32(int64_t n_elem, const double* __restrict__ R, const double* __restrict__ inv_norm,
                            const int32_t* __restrict__ seg_of_elem_row, float* __restrict__ R32) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n_elem;
         i += (int64_t)gridDim.x * blockDim.x) {
        const int64_t row = i / (3 * kNrhs);
        const int s = seg_of_elem_row[row] * kNrhs + (int)(i % kNrhs);
        R32[i] = (float)(R[i] * inv_norm[s]);
    }
}

// Reliable update of the search direction per system: P *= ratio[s] (the
// same direction in the new normalisation of its residual), or, where
// ratio[s] = 0, a restart P = Dinv R
__global__ void k_mr_scale(int64_t n_elem, const double* __restrict__ ratio, const int32_t* __restrict__ seg_of_elem_row,
                           const float* __restrict__ dinv, const float* __restrict__ R, float* __restrict__ P) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n_elem;
         i += (int64_t)gridDim.x * blockDim.x) {
        const int64_t row = i / (3 * kNrhs);
        const int s = seg_of_elem_row[row] * kNrhs + (int)(i % kNrhs);
        const double q = ratio[s];
        P[i] = q != 0.0 ? (float)(P[i] * q) : dinv[i / kNrhs] * R[i];
    }
}

// U += X / inv_norm (FP64 update of every system)
__global__ void k_mr_axpy(int64_t n_elem, const float* __restrict__ X, const double* __restrict__ inv_norm,
                          const int32_t* __restrict__ seg_of_elem_row, double* __restrict__ U) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n_elem;
         i += (int64_t)gridDim.x * blockDim.x) {
        const int64_t row = i / (3 * kNrhs);
        const int s = seg_of_elem_row[row] * kNrhs + (int)(i % kNrhs);
        const double w = inv_norm[s];
        if (w > 0.0) U[i] += (double)X[i] / w;
    }
}

// The batch's copy of one variant's operator: slice s of the batch's order takes the
// rows order[64 s ...] of the variant (-1: none), their blocks in the same slots;
// slots a row does not have are zero blocks on itself.  TOGETHER: a row's nine values of
// a slot one after another, else each component of the 64 rows.
template <typename T, bool TOGETHER>
__global__ __launch_bounds__(kBlock) void k_permute_sell(const int32_t* __restrict__ order,
                                                         const int32_t* __restrict__ inv,
                                                         const int32_t* __restrict__ sptr_old,
                                                         const int32_t* __restrict__ scol_old,
                                                         const T* __restrict__ val_old,
                                                         const int32_t* __restrict__ sptr, int slice0,
                                                         int32_t* __restrict__ scol, T* __restrict__ val) {
    const int s = blockIdx.x, lane = threadIdx.x % kWave;
    const int32_t row0 = kWave * slice0;
    const int r = order[(int64_t)s * kWave + lane];
    const int p0 = r >= 0 ? sptr_old[r / kWave] : 0, w = r >= 0 ? sptr_old[r / kWave + 1] - p0 : 0;
    const int k0 = sptr[slice0 + s], k1 = sptr[slice0 + s + 1];
    for (int k = threadIdx.x / kWave; k < k1 - k0; k += kBlock / kWave) {
        const int64_t dst = (int64_t)(k0 + k) * kWave + lane, src = (int64_t)(p0 + k) * kWave + r % kWave;
        const bool have = k < w;
        if (scol) scol[dst] = row0 + (have ? inv[scol_old[src]] : s * kWave + lane);
#pragma unroll
        for (int q = 0; q < 9; ++q)
            val[TOGETHER ? dst * 9 + q : ((int64_t)(k0 + k) * 9 + q) * kWave + lane] =
                have ? val_old[((int64_t)(p0 + k) * 9 + q) * kWave + r % kWave] : (T)0;
    }
}

__global__ void k_permute_dofs(int64_t n_rows, const int32_t* __restrict__ order, const float* __restrict__ a,
                               float* __restrict__ b) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= 3 * n_rows) return;
    const int r = order[i / 3];
    b[i] = r >= 0 ? a[3 * (int64_t)r + i % 3] : 0.f;
}

// Right-hand sides of one variant, [j][dof], into and out of the batch's
// [row][3][kNrhs]; those a variant does not have are zero.
__global__ void k_pack(int64_t n_rows, const int32_t* __restrict__ order, int nrhs, int64_t n_dof,
                       const double* __restrict__ a, double* __restrict__ F) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= 3 * n_rows * kNrhs) return;
    const int64_t e = i / kNrhs;
    const int j = (int)(i % kNrhs), r = order[e / 3];
    F[i] = (r >= 0 && j < nrhs) ? a[j * n_dof + 3 * (int64_t)r + e % 3] : 0.0;
}

__global__ void k_unpack(int64_t n_rows, const int32_t* __restrict__ order, int nrhs, int64_t n_dof,
                         const double* __restrict__ U, double* __restrict__ a) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= 3 * n_rows * kNrhs) return;
    const int64_t e = i / kNrhs;
    const int j = (int)(i % kNrhs), r = order[e / 3];
    if (r >= 0 && j < nrhs) a[j * n_dof + 3 * (int64_t)r + e % 3] = U[i];
}

int nbk(int64_t n) { return (int)std::min<int64_t>((n + 255) / 256, 8192); }

}  // namespace

struct Batch {
    std::string err;
    hipStream_t st = nullptr;
    int n_var = 0;
    std::vector<int64_t> n_rows, row_off;  // block rows of each variant and their offset
    int32_t* order = nullptr;              // variant's row of each of the batch's rows (-1: padding)
    int64_t rows_total = 0;                // padded to whole slices
    int n_slices = 0;
    int32_t *sptr = nullptr, *scol = nullptr;
    float* K32 = nullptr;
    double* K64 = nullptr;
    float* dinv = nullptr;
    // reduction chunks
    int n_chunks = 0;
    int32_t *chunk_row = nullptr, *seg_chunk = nullptr, *seg_of_row = nullptr;
    int n_blks = 0;  // workgroups of the product
    BlkInfo* blk_info = nullptr;
    ChunkInfo* chunk_info = nullptr;
    // per variant: some system still iterating; active as the iteration under way found it
    uint8_t *active = nullptr, *going = nullptr;
    // vectors [rows_total][3][kNrhs]
    double *F = nullptr, *U = nullptr, *R64 = nullptr;
    float *B32 = nullptr, *X = nullptr, *R = nullptr, *P = nullptr, *Q = nullptr;
    // scalars before an iteration and (sv_mid) before its direction; partials of the chunks and
    // (pq) of the product, (pr) of the new directions
    double *sv = nullptr, *sv_mid = nullptr, *partials = nullptr, *pq = nullptr, *pr = nullptr, *rr = nullptr, *inv_norm = nullptr, *ratio = nullptr, *tol2 = nullptr;
    uint8_t* frozen = nullptr;
    double* h_sv = nullptr;
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
};

namespace {

#define BCHK(expr)                                                       \
    do {                                                                 \
        hipError_t e_ = (expr);                                          \
        if (e_ != hipSuccess) {                                          \
            b->err = std::string(#expr) + ": " + hipGetErrorString(e_);  \
            return ASEND_ERR_HIP;                                        \
        }                                                                \
    } while (0)

template <typename T>
void bfree(T*& p) {
    if (p) (void)hipFree((void*)p);
    p = nullptr;
}

// FP64 residual R64 = F - K64 U for every system and its squared norm per system
void residual64(Batch* b) {
    const int nblk = (b->n_slices + kBlock / kWave - 1) / (kBlock / kWave);
    for (int j0 = 0; j0 < kNrhs; j0 += 8)
        hipLaunchKernelGGL(k_mrhs_residual, dim3(nblk), dim3(kBlock), 0, b->st, b->n_slices, b->sptr, b->scol, b->K64,
                           b->U, b->R64, b->F, j0);
    hipLaunchKernelGGL(k_chunk_rr64, dim3(b->n_chunks), dim3(256), 0, b->st, b->chunk_row, b->R64, b->partials);
    hipLaunchKernelGGL(k_sys_fin, dim3(b->n_var), dim3(256), 0, b->st,
                       b->seg_chunk, b->partials, 3, b->sv, b->frozen, b->rr);
}

// one lockstep iteration of every active system
void iterate(Batch* b) {
    hipLaunchKernelGGL(k_mrhs_dir_product, dim3(b->n_blks), dim3(kBlock), 0, b->st, b->blk_info, b->sptr, b->scol,
                       b->K32, b->P, b->Q, b->active, b->pq);
    hipLaunchKernelGGL(k_chunk_update, dim3(b->n_chunks), dim3(256), 0, b->st, b->chunk_info, b->dinv, (float4*)b->R,
                       (const float4*)b->Q, b->pq, b->pr, b->sv, b->sv_mid, b->partials, b->active, b->going);
    hipLaunchKernelGGL(k_chunk_dir, dim3(b->n_chunks), dim3(256), 0, b->st, b->chunk_info, b->dinv,
                       (const float4*)b->R, (float4*)b->P, (float4*)b->X, b->partials, b->sv_mid, b->sv, b->pr,
                       b->going, b->active);
}

// p.r of the directions and residuals an iteration starts from
void start_pr(Batch* b) {
    hipLaunchKernelGGL(k_chunk_pr, dim3(b->n_chunks), dim3(256), 0, b->st, b->chunk_row, (const float4*)b->P,
                       (const float4*)b->R, b->pr);
}

}  // namespace

// Which of n pieces workgroup k of a variant takes: the workgroups of an XCD (every
// kNumXcd-th) contiguous ones.
static int xcd_piece(int k, int n) {
    const int x = k % kNumXcd, per = n / kNumXcd, more = n % kNumXcd;
    return x * per + std::min(x, more) + k / kNumXcd;
}

// Rows by bricks of 4 x 4 x 4 nodes, from their coordinates and the mean reach of a
// row in each direction (on a lattice its spacing; on any mesh some order).  Sorted by
// digits of the key, whose fields are as wide as the mesh needs (two passes up to
// 22 bits); rows of one place stay in their order.  337,881 rows 17 ms on the host,
// 45 ms with std::sort on pairs; a batch's first creation over three meshes of 209,475
// rows 33 -> 15 ms.
std::vector<int32_t> batch_row_order(int64_t n, const int32_t* rp, const int32_t* bc, const double* xyz) {
    constexpr double kMaxCell = (1 << 20) - 1;
    double lo[3] = {xyz[0], xyz[1], xyz[2]}, h[3] = {0.0, 0.0, 0.0};
    for (int64_t r = 0; r < n; ++r)
        for (int a = 0; a < 3; ++a) lo[a] = std::min(lo[a], xyz[3 * r + a]);
    const int64_t step = std::max<int64_t>(1, n / 4096);
    int64_t cnt = 0;
    for (int64_t r = 0; r < n; r += step, ++cnt) {
        double d[3] = {0.0, 0.0, 0.0};
        for (int32_t k = rp[r]; k < rp[r + 1]; ++k)
            for (int a = 0; a < 3; ++a) d[a] = std::max(d[a], std::abs(xyz[3 * (int64_t)bc[k] + a] - xyz[3 * r + a]));
        for (int a = 0; a < 3; ++a) h[a] += d[a];
    }
    for (int a = 0; a < 3; ++a) h[a] /= cnt;
    std::vector<int32_t> cell(3 * n);
    int32_t top[3] = {0, 0, 0};
    for (int64_t r = 0; r < n; ++r)
        for (int a = 0; a < 3; ++a) {
            const double q = (xyz[3 * r + a] - lo[a]) / h[a] + 0.5;  // the cell is its floor
            const int32_t c = q > 0.0 ? (q < kMaxCell ? (int32_t)q : (int32_t)kMaxCell) : 0;
            cell[3 * r + a] = c;
            top[a] = std::max(top[a], c >> 2);
        }
    int width[3];
    for (int a = 0; a < 3; ++a)
        for (width[a] = 0; top[a] >> width[a]; ++width[a]) {
        }
    std::vector<uint64_t> key(n), key2(n);
    std::vector<int32_t> order(n), order2(n);
    for (int64_t r = 0; r < n; ++r) {
        uint64_t box = 0, in = 0;
        for (int a = 2; a >= 0; --a) {
            box = (box << width[a]) | (uint64_t)(cell[3 * r + a] >> 2);
            in = (in << 2) | (uint64_t)(cell[3 * r + a] & 3);
        }
        key[r] = (box << 6) | in;
        order[r] = (int32_t)r;
    }
    constexpr int kDigit = 11;
    for (int shift = 0; shift < width[0] + width[1] + width[2] + 6; shift += kDigit) {
        std::vector<int64_t> at((1 << kDigit) + 1, 0);
        auto digit = [&](uint64_t k) { return (k >> shift) & ((1 << kDigit) - 1); };
        for (int64_t i = 0; i < n; ++i) ++at[digit(key[i]) + 1];
        for (int d = 0; d < 1 << kDigit; ++d) at[d + 1] += at[d];
        for (int64_t i = 0; i < n; ++i) {
            const int64_t o = at[digit(key[i])]++;
            key2[o] = key[i];
            order2[o] = order[i];
        }
        key.swap(key2);
        order.swap(order2);
    }
    return order;
}

int batch_create(Batch** out, const std::vector<OperatorView>& ops) {
    Batch* b = new Batch();
    *out = b;
    b->n_var = (int)ops.size();
    if (b->n_var < 1) {
        b->err = "empty batch";
        return ASEND_ERR_ARG;
    }
    BCHK(hipStreamCreateWithFlags(&b->st, hipStreamNonBlocking));
    BCHK(hipEventCreate(&b->ev0));
    BCHK(hipEventCreate(&b->ev1));
    // layout: variant v owns slices [slice_off, slice_off + n_slices_v)
    std::vector<int32_t> slice_off(b->n_var + 1, 0);
    std::vector<int32_t> sptr(1, 0), order;
    for (int v = 0; v < b->n_var; ++v) {
        const OperatorView& o = ops[v];
        slice_off[v + 1] = slice_off[v] + o.n_slices;
        b->n_rows.push_back(o.n_rows);
        b->row_off.push_back((int64_t)kWave * slice_off[v]);
        for (int s = 0; s < o.n_slices; ++s) {
            int32_t w = 0;
            for (int l = 0; l < kWave; ++l) {
                const int64_t i = (int64_t)kWave * s + l;
                const int32_t r = i < o.n_rows ? o.order[i] : -1;
                order.push_back(r);
                if (r >= 0) w = std::max(w, o.h_rp[r + 1] - o.h_rp[r]);
            }
            if ((int64_t)sptr.back() + w > (1ll << 31) - 1) {
                b->err = "batch too large";
                return ASEND_ERR_UNSUPPORTED;
            }
            sptr.push_back(sptr.back() + w);
        }
    }
    b->n_slices = slice_off[b->n_var];
    b->rows_total = (int64_t)kWave * b->n_slices;
    const int64_t n_slots = sptr[b->n_slices];
    if (b->rows_total * 3 * kNrhs >= (1ll << 31) * 4 || b->rows_total >= (1ll << 31)) {
        b->err = "batch too large";
        return ASEND_ERR_UNSUPPORTED;
    }
    BCHK(hipMalloc((void**)&b->sptr, (b->n_slices + 1) * sizeof(int32_t)));
    BCHK(hipMalloc((void**)&b->scol, n_slots * kWave * sizeof(int32_t)));
    BCHK(hipMalloc((void**)&b->K32, n_slots * 9 * kWave * sizeof(float)));
    BCHK(hipMalloc((void**)&b->K64, n_slots * 9 * kWave * sizeof(double)));
    BCHK(hipMalloc((void**)&b->dinv, b->rows_total * 3 * sizeof(float)));
    BCHK(hipMalloc((void**)&b->order, order.size() * sizeof(int32_t)));
    BCHK(hipMemcpyAsync(b->order, order.data(), order.size() * 4, hipMemcpyHostToDevice, b->st));
    BCHK(hipMemcpyAsync(b->sptr, sptr.data(), sptr.size() * sizeof(int32_t), hipMemcpyHostToDevice, b->st));
    {
        // the variants' rows in the batch's order (scratch: row of each in it)
        std::vector<int32_t> inv(b->rows_total, 0);
        for (int v = 0; v < b->n_var; ++v)
            for (int64_t i = 0; i < ops[v].n_rows; ++i) inv[b->row_off[v] + ops[v].order[i]] = (int32_t)i;
        int32_t* d_inv = nullptr;
        BCHK(hipMalloc((void**)&d_inv, inv.size() * sizeof(int32_t)));
        hipError_t e = hipMemcpyAsync(d_inv, inv.data(), inv.size() * 4, hipMemcpyHostToDevice, b->st);
        for (int v = 0; v < b->n_var && e == hipSuccess; ++v) {
            const OperatorView& o = ops[v];
            const int64_t r0 = b->row_off[v], nr = (int64_t)kWave * o.n_slices;
            hipLaunchKernelGGL((k_permute_sell<float, true>), dim3(o.n_slices), dim3(kBlock), 0, b->st, b->order + r0,
                               d_inv + r0, o.sptr, o.scol, o.K32, b->sptr, slice_off[v], b->scol, b->K32);
            hipLaunchKernelGGL((k_permute_sell<double, false>), dim3(o.n_slices), dim3(kBlock), 0, b->st, b->order + r0,
                               d_inv + r0, o.sptr, o.scol, o.K64, b->sptr, slice_off[v], (int32_t*)nullptr, b->K64);
            hipLaunchKernelGGL(k_permute_dofs, dim3((unsigned)((3 * nr + 255) / 256)), dim3(256), 0, b->st, nr,
                               b->order + r0, o.dinv32, b->dinv + 3 * r0);
            e = hipGetLastError();
        }
        if (e == hipSuccess) e = hipStreamSynchronize(b->st);
        (void)hipFree(d_inv);
        BCHK(e);
    }
    // workgroups of the product: one slice each, or as many as keep a variant within kVarParts
    std::vector<int32_t> seg_blk(1, 0);
    {
        std::vector<BlkInfo> info;
        for (int v = 0; v < b->n_var; ++v) {
            const int n = ops[v].n_slices, per = (n + kVarParts - 1) / kVarParts, nb = (n + per - 1) / per;
            for (int k = 0; k < nb; ++k) {
                const int i = xcd_piece(k, nb);
                info.push_back({slice_off[v] + per * i, slice_off[v] + std::min(n, per * (i + 1)), v,
                                seg_blk.back() + i});
            }
            seg_blk.push_back((int32_t)info.size());
        }
        b->n_blks = (int)info.size();
        BCHK(hipMalloc((void**)&b->blk_info, info.size() * sizeof(BlkInfo)));
        BCHK(hipMalloc((void**)&b->active, b->n_var));
        BCHK(hipMalloc((void**)&b->going, b->n_var));
        BCHK(hipMemcpyAsync(b->blk_info, info.data(), info.size() * sizeof(BlkInfo), hipMemcpyHostToDevice, b->st));
        BCHK(hipStreamSynchronize(b->st));
    }
    // reduction chunks never span two variants
    std::vector<int32_t> crow, cseg, segc(b->n_var + 1, 0), seg_of_row(b->rows_total, 0);
    for (int v = 0; v < b->n_var; ++v) {
        const int64_t r0 = b->row_off[v], r1 = (v + 1 < b->n_var) ? b->row_off[v + 1] : b->rows_total;
        segc[v] = (int32_t)cseg.size();
        const int64_t even = ((r1 - r0 + kVarChunks - 1) / kVarChunks + kWave - 1) / kWave * kWave;
        const int64_t per = std::max<int64_t>(kChunkRows, even);
        for (int64_t r = r0; r < r1; r += per) {
            crow.push_back((int32_t)r);
            cseg.push_back(v);
        }
        for (int64_t r = r0; r < r1; ++r) seg_of_row[r] = v;
    }
    segc[b->n_var] = (int32_t)cseg.size();
    crow.push_back((int32_t)b->rows_total);
    b->n_chunks = (int)cseg.size();
    BCHK(hipMalloc((void**)&b->chunk_row, crow.size() * sizeof(int32_t)));
    std::vector<ChunkInfo> cinfo(b->n_chunks);
    for (int v = 0; v < b->n_var; ++v)
        for (int k = 0; k < segc[v + 1] - segc[v]; ++k) {
            const int ch = segc[v] + xcd_piece(k, segc[v + 1] - segc[v]);
            cinfo[segc[v] + k] = {crow[ch], crow[ch + 1], v, ch, segc[v], segc[v + 1], seg_blk[v], seg_blk[v + 1]};
        }
    BCHK(hipMalloc((void**)&b->chunk_info, cinfo.size() * sizeof(ChunkInfo)));
    BCHK(hipMalloc((void**)&b->seg_chunk, segc.size() * sizeof(int32_t)));
    BCHK(hipMalloc((void**)&b->seg_of_row, seg_of_row.size() * sizeof(int32_t)));
    BCHK(hipMemcpyAsync(b->chunk_row, crow.data(), crow.size() * 4, hipMemcpyHostToDevice, b->st));
    BCHK(hipMemcpyAsync(b->chunk_info, cinfo.data(), cinfo.size() * sizeof(ChunkInfo), hipMemcpyHostToDevice, b->st));
    BCHK(hipMemcpyAsync(b->seg_chunk, segc.data(), segc.size() * 4, hipMemcpyHostToDevice, b->st));
    BCHK(hipMemcpyAsync(b->seg_of_row, seg_of_row.data(), seg_of_row.size() * 4, hipMemcpyHostToDevice, b->st));
    const int64_t ne = b->rows_total * 3 * kNrhs;
    for (double** q : {&b->F, &b->U, &b->R64}) BCHK(hipMalloc((void**)q, ne * sizeof(double)));
    for (float** q : {&b->B32, &b->X, &b->R, &b->P, &b->Q}) BCHK(hipMalloc((void**)q, ne * sizeof(float)));
    const int n_sys = b->n_var * kNrhs;
    BCHK(hipMalloc((void**)&b->sv, (size_t)n_sys * B_N * sizeof(double)));
    BCHK(hipMalloc((void**)&b->sv_mid, (size_t)n_sys * B_N * sizeof(double)));
    BCHK(hipMalloc((void**)&b->partials, (size_t)b->n_chunks * 2 * kNrhs * sizeof(double)));
    BCHK(hipMalloc((void**)&b->pq, (size_t)b->n_blks * kNrhs * sizeof(double)));
    BCHK(hipMalloc((void**)&b->pr, (size_t)b->n_chunks * kNrhs * sizeof(double)));
    BCHK(hipMalloc((void**)&b->rr, n_sys * sizeof(double)));
    BCHK(hipMalloc((void**)&b->inv_norm, n_sys * sizeof(double)));
    BCHK(hipMalloc((void**)&b->ratio, n_sys * sizeof(double)));
    BCHK(hipMalloc((void**)&b->tol2, n_sys * sizeof(double)));
    BCHK(hipMalloc((void**)&b->frozen, n_sys));
    BCHK(hipHostMalloc((void**)&b->h_sv, (size_t)n_sys * B_N * sizeof(double), hipHostMallocDefault));
    BCHK(hipStreamSynchronize(b->st));
    return ASEND_OK;
}

void batch_destroy(Batch* b) {
    if (!b) return;
    if (b->st) (void)hipStreamSynchronize(b->st);
    bfree(b->sptr);
    bfree(b->scol);
    bfree(b->K32);
    bfree(b->K64);
    bfree(b->dinv);
    bfree(b->chunk_row);
    bfree(b->chunk_info);
    bfree(b->seg_chunk);
    bfree(b->seg_of_row);
    bfree(b->blk_info);
    bfree(b->order);
    bfree(b->active);
    bfree(b->going);
    for (double** q : {&b->F, &b->U, &b->R64, &b->sv, &b->sv_mid, &b->partials, &b->pq, &b->pr, &b->rr, &b->inv_norm, &b->ratio,
                       &b->tol2})
        bfree(*q);
    for (float** q : {&b->B32, &b->X, &b->R, &b->P, &b->Q}) bfree(*q);
    bfree(b->frozen);
    if (b->h_sv) (void)hipHostFree(b->h_sv);
    if (b->ev0) (void)hipEventDestroy(b->ev0);
    if (b->ev1) (void)hipEventDestroy(b->ev1);
    if (b->st) (void)hipStreamDestroy(b->st);
    delete b;
}

const char* batch_error(const Batch* b) { return b ? b->err.c_str() : ""; }

int batch_solve(Batch* b, const double* const* rhs, double* const* x, int nrhs, double tol, double inner_tol, int64_t max_it,
                int check_every, int verbose, BatchStats* stats) {
    if (nrhs < 1 || nrhs > kNrhs || !(tol > 0) || !(inner_tol > 0) || check_every < 1) {
        b->err = "bad batch solve arguments";
        return ASEND_ERR_ARG;
    }
    const int n_sys = b->n_var * kNrhs;
    const int64_t ne = b->rows_total * 3 * kNrhs;
    // the right-hand sides through R64, which the first residual overwrites
    auto padded_rows = [&](int v) { return ((v + 1 < b->n_var) ? b->row_off[v + 1] : b->rows_total) - b->row_off[v]; };
    for (int v = 0; v < b->n_var; ++v) {
        const int64_t r0 = b->row_off[v], nr = padded_rows(v), nd = 3 * b->n_rows[v];
        double* stage = b->R64 + r0 * 3 * kNrhs;
        BCHK(hipMemcpyAsync(stage, rhs[v], nrhs * nd * sizeof(double), hipMemcpyHostToDevice, b->st));
        hipLaunchKernelGGL(k_pack, dim3((unsigned)((3 * nr * kNrhs + 255) / 256)), dim3(256), 0, b->st, nr,
                           b->order + r0, nrhs, nd, stage, b->F + r0 * 3 * kNrhs);
    }
    BCHK(hipMemsetAsync(b->U, 0, ne * sizeof(double), b->st));
    BCHK(hipEventRecord(b->ev0, b->st));
    // ||f|| per system
    residual64(b);
    std::vector<double> ff(n_sys), rr(n_sys), invn(n_sys);
    BCHK(hipMemcpyAsync(ff.data(), b->rr, n_sys * sizeof(double), hipMemcpyDeviceToHost, b->st));
    BCHK(hipStreamSynchronize(b->st));
    rr = ff;
    // FP32 lockstep block-PCG with FP64 reliable updates.  Every system runs
    // one PCG whose residual is normalised at its last refresh; a refresh
    // (U += |r| X in FP64, the FP64 residual of every system, the converged
    // systems frozen, R = R64 / |R64|, P rescaled by |r_old| / |r_new|, rz and
    // |r|^2 recomputed) keeps every search direction.  It comes once every
    // active system has cut its recursive residual by inner_tol or claims
    // convergence; the FP64 residual alone decides convergence.
    std::vector<uint8_t> frozen(n_sys);
    std::vector<double> init((size_t)n_sys * B_N, 0.0), ratio(n_sys, 0.0), tol2(n_sys, 0.0), rr_prev(n_sys, 0.0);
    int64_t total_inner = 0, outer = 0;
    std::vector<int64_t> sys_it(n_sys, 0);
    const double ru2 = inner_tol * inner_tol;
    // next refresh targets and the refresh itself (host part)
    auto classify = [&]() {
        int active = 0;
        for (int s = 0; s < n_sys; ++s) {
            const bool conv = (s % kNrhs) >= nrhs || ff[s] == 0.0 || std::sqrt(rr[s] / ff[s]) <= tol;
            const double inv_old = invn[s];
            frozen[s] = conv ? 1 : 0;
            invn[s] = conv ? 0.0 : 1.0 / std::sqrt(rr[s]);
            // |r_old| / |r_new|: the factor that keeps P's direction in the new
            // normalisation; 0 (restart the direction) where the FP32
            // recursion drifted, i.e. the FP64 residual is more than twice the
            // recursive one: the old directions no longer fit the residual
            ratio[s] = (conv || inv_old == 0.0) ? 0.0 : 1.0 / (inv_old * std::sqrt(rr[s]));
            if (ratio[s] != 0.0) {
                const double rec = b->h_sv[(size_t)s * B_N + B_RR] * rr_prev[s];
                if (!(rec > 0.0) || rr[s] > 4.0 * rec) ratio[s] = 0.0;
            }
            // recursive convergence target of the renormalised system
            tol2[s] = conv ? 0.0 : tol * tol * ff[s] / rr[s];
            active += conv ? 0 : 1;
        }
        return active;
    };
    std::fill(invn.begin(), invn.end(), 0.0);
    int active = classify();
    for (int s = 0; s < n_sys; ++s) {
        init[(size_t)s * B_N + B_TOL2] = tol2[s];
        init[(size_t)s * B_N + B_MAXIT] = (double)max_it;
    }
    if (active) {
        BCHK(hipMemcpyAsync(b->frozen, frozen.data(), n_sys, hipMemcpyHostToDevice, b->st));
        BCHK(hipMemcpyAsync(b->inv_norm, invn.data(), n_sys * sizeof(double), hipMemcpyHostToDevice, b->st));
        std::memcpy(b->h_sv, init.data(), init.size() * sizeof(double));
        BCHK(hipMemcpyAsync(b->sv, b->h_sv, init.size() * sizeof(double), hipMemcpyHostToDevice, b->st));
        hipLaunchKernelGGL(k_mr_to_f32, dim3(nbk(ne)), dim3(256), 0, b->st, ne, b->R64, b->inv_norm, b->seg_of_row,
                           b->B32);
        hipLaunchKernelGGL(k_chunk_init, dim3(b->n_chunks), dim3(256), 0, b->st, b->chunk_row, b->dinv, b->B32, b->X,
                           b->R, b->P, b->partials);
        hipLaunchKernelGGL(k_sys_fin, dim3(b->n_var), dim3(256), 0, b->st, b->seg_chunk, b->partials, 0, b->sv,
                           b->frozen, (double*)nullptr);
        hipLaunchKernelGGL(k_var_active, dim3((b->n_var + 255) / 256), dim3(256), 0, b->st, b->n_var, b->sv,
                           b->active);
        start_pr(b);
    }
    while (active && outer < 200) {
        for (int k = 0; k < check_every; ++k) iterate(b);
        total_inner += check_every;
        BCHK(hipGetLastError());
        BCHK(hipMemcpyAsync(b->h_sv, b->sv, (size_t)n_sys * B_N * sizeof(double), hipMemcpyDeviceToHost, b->st));
        BCHK(hipStreamSynchronize(b->st));
        // refresh once every active system is done or has cut its residual by inner_tol
        bool refresh = true, stalled = true;
        for (int s = 0; s < n_sys && refresh; ++s) {
            if (frozen[s]) continue;
            const double* v = b->h_sv + (size_t)s * B_N;
            const bool done = v[B_DONE] != 0.0;
            refresh = done || v[B_RR] <= ru2 * v[B_RR0];
            stalled = stalled && done && v[B_IT] >= v[B_MAXIT];
        }
        if (!refresh) continue;
        ++outer;
        for (int s = 0; s < n_sys; ++s) sys_it[s] = (int64_t)b->h_sv[(size_t)s * B_N + B_IT];
        hipLaunchKernelGGL(k_mr_axpy, dim3(nbk(ne)), dim3(256), 0, b->st, ne, b->X, b->inv_norm, b->seg_of_row, b->U);
        BCHK(hipMemsetAsync(b->X, 0, ne * sizeof(float), b->st));
        residual64(b);
        rr_prev = rr;
        BCHK(hipMemcpyAsync(rr.data(), b->rr, n_sys * sizeof(double), hipMemcpyDeviceToHost, b->st));
        BCHK(hipStreamSynchronize(b->st));
        active = classify();
        if (verbose) {
            double worst = 0.0;
            for (int s = 0; s < n_sys; ++s)
                if ((s % kNrhs) < nrhs && ff[s] > 0.0) worst = std::max(worst, std::sqrt(rr[s] / ff[s]));
            std::fprintf(stderr, "[batch] refresh %lld: %d active systems, %lld lockstep iterations, worst residual %.2e\n",
                         (long long)outer, active, (long long)total_inner, worst);
        }
        if (!active || stalled) break;
        BCHK(hipMemcpyAsync(b->frozen, frozen.data(), n_sys, hipMemcpyHostToDevice, b->st));
        BCHK(hipMemcpyAsync(b->inv_norm, invn.data(), n_sys * sizeof(double), hipMemcpyHostToDevice, b->st));
        BCHK(hipMemcpyAsync(b->ratio, ratio.data(), n_sys * sizeof(double), hipMemcpyHostToDevice, b->st));
        BCHK(hipMemcpyAsync(b->tol2, tol2.data(), n_sys * sizeof(double), hipMemcpyHostToDevice, b->st));
        hipLaunchKernelGGL(k_mr_to_f32, dim3(nbk(ne)), dim3(256), 0, b->st, ne, b->R64, b->inv_norm, b->seg_of_row,
                           b->R);
        hipLaunchKernelGGL(k_mr_scale, dim3(nbk(ne)), dim3(256), 0, b->st, ne, b->ratio, b->seg_of_row, b->dinv, b->R,
                           b->P);
        hipLaunchKernelGGL(k_chunk_rz, dim3(b->n_chunks), dim3(256), 0, b->st, b->chunk_row, b->dinv, b->R,
                           b->partials);
        hipLaunchKernelGGL(k_sys_fin, dim3(b->n_var), dim3(256), 0, b->st, b->seg_chunk, b->partials, 4, b->sv,
                           b->frozen, b->tol2);
        hipLaunchKernelGGL(k_var_active, dim3((b->n_var + 255) / 256), dim3(256), 0, b->st, b->n_var, b->sv,
                           b->active);
        start_pr(b);
    }
    BCHK(hipEventRecord(b->ev1, b->st));
    BCHK(hipEventSynchronize(b->ev1));
    float ms = 0;
    BCHK(hipEventElapsedTime(&ms, b->ev0, b->ev1));
    for (int v = 0; v < b->n_var; ++v) {
        const int64_t r0 = b->row_off[v], nr = padded_rows(v), nd = 3 * b->n_rows[v];
        double* stage = b->R64 + r0 * 3 * kNrhs;
        hipLaunchKernelGGL(k_unpack, dim3((unsigned)((3 * nr * kNrhs + 255) / 256)), dim3(256), 0, b->st, nr,
                           b->order + r0, nrhs, nd, b->U + r0 * 3 * kNrhs, stage);
        BCHK(hipGetLastError());
        BCHK(hipMemcpyAsync(x[v], stage, nrhs * nd * sizeof(double), hipMemcpyDeviceToHost, b->st));
    }
    BCHK(hipStreamSynchronize(b->st));
    if (stats) {
        std::memset(stats, 0, sizeof(*stats));
        stats->outer_iterations = outer;
        stats->lockstep_iterations = total_inner;
        double worst = 0.0;
        int64_t nc = 0, sum_it = 0;
        for (int s = 0; s < n_sys; ++s) {
            if ((s % kNrhs) >= nrhs || ff[s] == 0.0) continue;
            const double rel = std::sqrt(rr[s] / ff[s]);
            worst = std::max(worst, rel);
            nc += rel <= tol ? 0 : 1;
            sum_it += sys_it[s];
        }
        stats->max_rel_residual = worst;
        stats->unconverged = nc;
        stats->system_iterations = sum_it;
        stats->device_ms = ms;
    }
    return ASEND_OK;
}

}  // namespace asend
