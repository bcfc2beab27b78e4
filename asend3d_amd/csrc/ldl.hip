// Device LDL^T of the operator over diagonal DOF blocks: the reference's
// LowerTriMat (S/lower_tri_mat_meth.rs:15-227) built for the GPU.
//
// The reference stores each row from its first column inside its block (the
// envelope) and factors column by column with scalar loops.  Inside the
// envelope the factor fills completely and outside it stays exactly zero, so
// the same factor is obtained from a uniform band of 64 x 64 tiles that
// covers the widest row: the factorization is then a blocked right-looking
// LDL^T whose steps are one diagonal-tile factorization, a panel of
// tile products with L_kk^-1 and a trailing update of tile products,
// all blocks of the numbering at once, followed by the inverses of
// the diagonal super-blocks of a few tiles.  The solve takes a super-block at
// a time: a product with its inverse and an update of the band it couples to.
#include "ldl.hpp"

#include <algorithm>
#include <cmath>

#include "device_common.hpp"

namespace asend {

namespace {

// Operator values inside each block's envelope into the banded tiles: one
// lane per block row (3 DOF rows) of a 64-row slice of the sliced-ELL FP64
// operator, every slot (3x3 block) of that row.
__global__ __launch_bounds__(kWave) void k_ldl_fill(LdlDesc d, int n_rows, const int32_t* __restrict__ sptr,
                                                    const int32_t* __restrict__ scol, const double* __restrict__ K,
                                                    double* __restrict__ L) {
    const int slice = blockIdx.x, lane = threadIdx.x;
    const int R = slice * kWave + lane;
    if (R >= n_rows) return;
    const int s0 = sptr[slice], ns = sptr[slice + 1] - s0;
    for (int k = 0; k < ns; ++k) {
        const int C = scol[(int64_t)kWave * (s0 + k) + lane];
        if (C < 0 || C > R) continue;  // upper blocks and padding
        for (int a = 0; a < 3; ++a) {
            const int64_t i = 3 * (int64_t)R + a;
            const int blk = (int)(i / d.bs);
            const int64_t b0 = (int64_t)blk * d.bs, li = i - b0;
            for (int c = 0; c < 3; ++c) {
                const int64_t j = 3 * (int64_t)C + c;
                if (j > i || j < b0) continue;
                const int64_t lj = j - b0;
                const int I = (int)(li / kLdlTile), J = (int)(lj / kLdlTile);
                if (I - J > d.wt) continue;
                const double v = K[((int64_t)9 * (s0 + k) + 3 * a + c) * kWave + lane];
                L[ldl_tile(d, blk, I, J) + (li % kLdlTile) * kLdlTile + lj % kLdlTile] += v;
            }
        }
    }
}

// Identity rows past the end of each block's last tile.
__global__ void k_ldl_pad(LdlDesc d, double* __restrict__ L) {
    const int blk = blockIdx.x;
    const int64_t s = (int64_t)blk * d.bs;
    const int64_t m = std::min(d.bs, d.n - s);
    const int nt = ldl_block_nt(d, blk);
    const int r = threadIdx.x;
    if ((int64_t)(nt - 1) * kLdlTile + r >= m) L[ldl_tile(d, blk, nt - 1, nt - 1) + r * kLdlTile + r] = 1.0;
}

typedef double d4v __attribute__((ext_vector_type(4)));
typedef double d2t __attribute__((ext_vector_type(2)));

// Matrix-core products of the factorization: v_mfma_f64_16x16x4_f64, one
// wavefront per 16 x 16 output.  Lane l holds A[l % 16][l / 16] and
// B[l / 16][l % 16] of a 4-deep step and rows 4 r + l / 16, column l % 16 of
// the output in register r, so an output is itself the B operand of the four
// steps of a following product.
__device__ __forceinline__ d4v mfma64(double a, double b, d4v c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// Tiles staged for the matrix-core products: rows 2 mod 32 doubles apart, so
// the 16 rows x 2 columns that half a wavefront reads fall in 64 different banks
// and rows stay 16-byte aligned for the staging stores.
constexpr int kLm = kLdlTile + 2;

// One 64 x 64 tile into registers: 256 threads, 16 doubles each, every load
// in flight before the first use.
__device__ __forceinline__ void load_tile(const double* __restrict__ g, d2t (&v)[8]) {
    const d2t* p = reinterpret_cast<const d2t*>(g);
#pragma unroll
    for (int h = 0; h < 8; ++h) v[h] = p[threadIdx.x + h * kBlock];
}

// Double pair e of a tile: row e / 32, columns 2 (e % 32) and the next.
__device__ __forceinline__ void store_tile(double* __restrict__ s, const d2t (&v)[8]) {
#pragma unroll
    for (int h = 0; h < 8; ++h) {
        const int e = threadIdx.x + h * kBlock;
        *reinterpret_cast<d2t*>(s + (e >> 5) * kLm + 2 * (e & 31)) = v[h];
    }
}

// value of lane l (a constant) of v in every lane
__device__ __forceinline__ double lane_value(double v, int l) {
    const long long b = __double_as_longlong(v);
    const unsigned lo = __builtin_amdgcn_readlane((unsigned)b, l);
    const unsigned hi = __builtin_amdgcn_readlane((unsigned)(b >> 32), l);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// 1 / v from the hardware estimate by two Newton steps (each doubles the
// correct bits): the pivot chain below waits for nothing else.
__device__ __forceinline__ double pivot_rcp(double v) {
    double r = __builtin_amdgcn_rcp(v);
    r = fma(fma(-v, r, 1.0), r, r);
    return fma(fma(-v, r, 1.0), r, r);
}

// LDS of a diagonal tile's factorization besides its two staged tiles
constexpr int kPivot = 16;          // pivot block edge
constexpr int kUs = kPivot + 2;     // row stride of U
struct DiagLds {
    double U[3 * kPivot * kUs];  // L D of the block column
    double d[kLdlTile];
};

// The staged tile A = L D L^T and the unit lower inverse L^-1, written to T as
// the diagonal tile (D on the diagonal, L^-1 below it, zeros above): the panel
// and the solves multiply by L^-1 and never need L.  256 threads; A is
// destroyed, Li is scratch, both in the staged layout.
//
// Bound by the chain of 64 dependent pivots, so everything but that chain is
// on the matrix cores: the tile is a 4 x 4 grid of 16 x 16 blocks; per block
// column wavefront 0 eliminates the 16 x 16 pivot block in registers (lane =
// row, pivot rows broadcast by readlane) and applies the same row operations
// to the identity, whose independent products fill the pivot chain's waits;
// then the block column below it is scaled and the trailing blocks updated by
// one wavefront per 16 x 16 product.  The inverse of the tile follows block
// diagonal by block diagonal, Li_IJ = -Li_II sum_M L_IM Li_MJ.
__device__ __forceinline__ void diag_factor(double* A, double* Li, DiagLds& S, double* T,
                                            int32_t* __restrict__ neg) {
    const int t = threadIdx.x, w = t >> 6, l = t & 63, c16 = l & 15, q4 = l >> 4;
    {
        const d2t z = {0.0, 0.0};
        const d2t v[8] = {z, z, z, z, z, z, z, z};
        store_tile(Li, v);
    }
    int n_neg = 0;
    for (int kb = 0; kb < 4; ++kb) {
        const int o = kPivot * kb;
        __syncthreads();
        if (w == 0) {
            double a[kPivot], v[kPivot];  // row c16 of the pivot block (lower part) and of its inverse factor
#pragma unroll
            for (int m = 0; m < kPivot; ++m) {
                a[m] = A[(o + c16) * kLm + o + m];
                v[m] = c16 == m ? 1.0 : 0.0;
            }
#pragma unroll
            for (int j = 0; j < kPivot; ++j) {
                const double dj = lane_value(a[j], j);
                n_neg += dj < 0.0 ? 1 : 0;
                const double lj = a[j] * pivot_rcp(dj);  // column j of L in the lanes below j
#pragma unroll
                for (int m = j + 1; m < kPivot; ++m) a[m] = fma(-a[j], lane_value(lj, m), a[m]);
                const double li = c16 > j ? lj : 0.0;
#pragma unroll
                for (int m = 0; m <= j; ++m) v[m] = fma(-li, lane_value(v[m], j), v[m]);
                if (l == j) S.d[o + j] = dj;
            }
            if (l < kPivot) {
#pragma unroll
                for (int m = 0; m < kPivot; ++m) Li[(o + c16) * kLm + o + m] = v[m];
            }
        }
        __syncthreads();
        // block column: U = A_ib,kb Li_kk^T (= L D), L = U D^-1
        if (w < 3 - kb) {
            const int ib = kb + 1 + w;
            const double inv = pivot_rcp(S.d[o + c16]);
            d4v acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
            for (int s = 0; s < 4; ++s)
                acc = mfma64(A[(kPivot * ib + c16) * kLm + o + 4 * s + q4], Li[(o + c16) * kLm + o + 4 * s + q4],
                             acc);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int i = 4 * r + q4;
                S.U[(kPivot * w + i) * kUs + c16] = acc[r];
                A[(kPivot * ib + i) * kLm + o + c16] = acc[r] * inv;
            }
        }
        __syncthreads();
        // trailing blocks (ib, jb), kb < jb <= ib: A -= L_ib U_jb^T
        const int nb = 3 - kb;
        for (int q = w; q < nb * (nb + 1) / 2; q += 4) {
            const int pi = q == 0 ? 0 : (q < 3 ? 1 : 2), pj = q - pi * (pi + 1) / 2;
            const int ib = kb + 1 + pi, jb = kb + 1 + pj;
            d4v acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
            for (int s = 0; s < 4; ++s)
                acc = mfma64(A[(kPivot * ib + c16) * kLm + o + 4 * s + q4],
                             S.U[(kPivot * pj + c16) * kUs + 4 * s + q4], acc);
#pragma unroll
            for (int r = 0; r < 4; ++r) A[(kPivot * ib + 4 * r + q4) * kLm + kPivot * jb + c16] -= acc[r];
        }
    }
    if (t == 0 && n_neg > 0) atomicAdd(neg, n_neg);
    for (int dist = 1; dist < 4; ++dist) {
        __syncthreads();
        if (w < 4 - dist) {
            const int J = w, I = w + dist;
            d4v acc = {0.0, 0.0, 0.0, 0.0};
            for (int M = J; M < I; ++M)
#pragma unroll
                for (int s = 0; s < 4; ++s)
                    acc = mfma64(A[(kPivot * I + c16) * kLm + kPivot * M + 4 * s + q4],
                                 Li[(kPivot * M + 4 * s + q4) * kLm + kPivot * J + c16], acc);
            d4v x = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
            for (int s = 0; s < 4; ++s)
                x = mfma64(-Li[(kPivot * I + c16) * kLm + kPivot * I + 4 * s + q4], acc[s], x);
#pragma unroll
            for (int r = 0; r < 4; ++r) Li[(kPivot * I + 4 * r + q4) * kLm + kPivot * J + c16] = x[r];
        }
    }
    __syncthreads();
    if (t < kLdlTile) Li[t * kLm + t] = S.d[t];
    __syncthreads();
    d2t* out = reinterpret_cast<d2t*>(T);
#pragma unroll
    for (int h = 0; h < 8; ++h) {
        const int e = t + h * kBlock;
        out[e] = *reinterpret_cast<const d2t*>(Li + (e >> 5) * kLm + 2 * (e & 31));
    }
}

// First diagonal tile of every block (the update of step k - 1 factors tile k).
__global__ __launch_bounds__(kBlock) void k_ldl_diag(LdlDesc d, double* __restrict__ L, int32_t* __restrict__ neg) {
    __shared__ __align__(16) double A[kLdlTile * kLm];
    __shared__ __align__(16) double Li[kLdlTile * kLm];
    __shared__ DiagLds S;
    double* T = L + ldl_tile(d, blockIdx.x, 0, 0);
    {
        d2t v[8];
        load_tile(T, v);
        store_tile(A, v);
    }
    diag_factor(A, Li, S, T, neg);
}

// 16 rows of a 64 x 64 product A B^T of two staged tiles: wavefront w takes
// rows 16 w.., acc[b] the columns 16 b.. .
__device__ __forceinline__ void tile_rows_abt(const double* __restrict__ sA, const double* __restrict__ sB,
                                              d4v (&acc)[4]) {
    const int l = threadIdx.x & 63, row = 16 * (threadIdx.x >> 6) + (l & 15), q4 = l >> 4;
#pragma unroll 4
    for (int s = 0; s < 16; ++s) {
        const double a = sA[row * kLm + 4 * s + q4];
#pragma unroll
        for (int b = 0; b < 4; ++b) acc[b] = mfma64(a, sB[(16 * b + (l & 15)) * kLm + 4 * s + q4], acc[b]);
    }
}

// Step k, panel: L_Ik = A_Ik L_kk^-T D_k^-1 for the tiles below the diagonal
// (blockIdx.y = I - k - 1).
//
// Panel and update are bound by the latency of one tile product per workgroup
// (a band of 9 tiles gives 9 and 45 of them): both operand tiles are loaded
// into registers at once (one exposed latency instead of one per loop turn)
// and multiplied on the matrix cores.
__global__ __launch_bounds__(kBlock) void k_ldl_panel(LdlDesc d, int k, double* __restrict__ L) {
    const int blk = blockIdx.x;
    const int I = k + 1 + blockIdx.y;
    if (I >= ldl_block_nt(d, blk)) return;
    __shared__ __align__(16) double sA[kLdlTile * kLm];
    __shared__ __align__(16) double sB[kLdlTile * kLm];
    __shared__ double si[kLdlTile];
    double* X = L + ldl_tile(d, blk, I, k);
    {
        d2t va[8], vb[8];
        load_tile(X, va);
        load_tile(L + ldl_tile(d, blk, k, k), vb);
        store_tile(sA, va);
        store_tile(sB, vb);
    }
    __syncthreads();
    if (threadIdx.x < kLdlTile) {
        si[threadIdx.x] = 1.0 / sB[threadIdx.x * (kLm + 1)];
        sB[threadIdx.x * (kLm + 1)] = 1.0;
    }
    __syncthreads();
    d4v acc[4] = {};
    tile_rows_abt(sA, sB, acc);
    const int l = threadIdx.x & 63, r0 = 16 * (threadIdx.x >> 6) + (l >> 4), c = l & 15;
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r) X[(r0 + 4 * r) * kLdlTile + 16 * b + c] = acc[b][r] * si[16 * b + c];
}

// Step k, trailing update of the band: A_IJ -= L_Ik D_k L_Jk^T for
// k < J <= I <= k + wt (blockIdx.y enumerates the pairs row by row).  The
// workgroup of the first pair holds the next diagonal tile once updated and
// factors it at once: one launch and one tile round trip less on the chain
// from a diagonal tile to the next.
//
// On a 552-wide band of 31,248 DOFs (489 steps, 9 tiles, MI355X): 30 us a
// step, panel 6.2 and update with the next diagonal tile 24.2, against 209 us
// with the tile eliminated element by element in LDS (177), and panel (14.5)
// and update (18) tiles staged one load at a time and multiplied on the VALU.
__global__ __launch_bounds__(kBlock) void k_ldl_update(LdlDesc d, int k, double* __restrict__ L,
                                                       int32_t* __restrict__ neg) {
    const int blk = blockIdx.x;
    const int q = blockIdx.y;
    int pi = (int)((std::sqrt(8.0 * q + 1.0) - 1.0) * 0.5);
    while ((pi + 1) * (pi + 2) / 2 <= q) ++pi;
    while (pi * (pi + 1) / 2 > q) --pi;
    const int pj = q - pi * (pi + 1) / 2;
    const int I = k + 1 + pi, J = k + 1 + pj;
    if (I >= ldl_block_nt(d, blk)) return;
    __shared__ __align__(16) double sA[kLdlTile * kLm];
    __shared__ __align__(16) double sB[kLdlTile * kLm];
    __shared__ DiagLds S;
    const double* Dk = L + ldl_tile(d, blk, k, k);
    double* C = L + ldl_tile(d, blk, I, J);
    const int l = threadIdx.x & 63, r0 = 16 * (threadIdx.x >> 6) + (l >> 4), c = l & 15;
    // the product is summed by itself and subtracted once: added to C term by
    // term it would be rounded at C's magnitude 16 times a step
    d4v acc[4] = {}, old[4];
    {
        d2t va[8], vb[8];
        load_tile(L + ldl_tile(d, blk, I, k), va);
        load_tile(L + ldl_tile(d, blk, J, k), vb);
        // the thread's two columns are the same in all of its rows
        const int m = 2 * (threadIdx.x & 31);
        const double d0 = Dk[m * (kLdlTile + 1)], d1 = Dk[(m + 1) * (kLdlTile + 1)];
#pragma unroll
        for (int b = 0; b < 4; ++b)
#pragma unroll
            for (int r = 0; r < 4; ++r) old[b][r] = C[(r0 + 4 * r) * kLdlTile + 16 * b + c];
        store_tile(sA, va);
#pragma unroll
        for (int h = 0; h < 8; ++h) {
            vb[h][0] *= d0;
            vb[h][1] *= d1;
        }
        store_tile(sB, vb);
    }
    __syncthreads();
    tile_rows_abt(sA, sB, acc);
#pragma unroll
    for (int b = 0; b < 4; ++b) acc[b] = old[b] - acc[b];
    if (q == 0) {
        __syncthreads();  // every wavefront is done with sA
#pragma unroll
        for (int b = 0; b < 4; ++b)
#pragma unroll
            for (int r = 0; r < 4; ++r) sA[(r0 + 4 * r) * kLm + 16 * b + c] = acc[b][r];
        diag_factor(sA, sB, S, C, neg);
        return;
    }
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r) C[(r0 + 4 * r) * kLdlTile + 16 * b + c] = acc[b][r];
}

// Inverses of the factor's diagonal super-blocks of S x S tiles, in place, by
// doubling: [[A, 0], [B, C]]^-1 = [[A^-1, 0], [-C^-1 B A^-1, C^-1]] for pairs
// of h-tile blocks, h = 1, 2, .. S / 2 (the tiles' own inverses are there).
// Pair q of a block covers tiles 2 h q ..; a first launch forms B A^-1 in
// scratch, a second -C^-1 times it over B.  One workgroup per output tile.
__device__ __forceinline__ void tile_rows_ab(const double* __restrict__ sA, const double* __restrict__ sB,
                                             d4v (&acc)[4]) {
    const int l = threadIdx.x & 63, row = 16 * (threadIdx.x >> 6) + (l & 15), q4 = l >> 4;
#pragma unroll 4
    for (int s = 0; s < 16; ++s) {
        const double a = sA[row * kLm + 4 * s + q4];
#pragma unroll
        for (int b = 0; b < 4; ++b) acc[b] = mfma64(a, sB[(4 * s + q4) * kLm + 16 * b + (l & 15)], acc[b]);
    }
}

__global__ __launch_bounds__(kBlock) void k_ldl_inv(LdlDesc d, int h, int pairs, int64_t pair0, int second,
                                                    double* __restrict__ L, double* __restrict__ tmp) {
    const int64_t q = pair0 + blockIdx.y;  // pair over all blocks
    const int blk = (int)(q / pairs), o = (int)(q % pairs) * 2 * h;
    const int nt = ldl_block_nt(d, blk);
    const int i = blockIdx.x / h, j = blockIdx.x % h;
    const int I = o + h + i, J = o + j;
    if (I >= nt) return;
    __shared__ __align__(16) double sA[kLdlTile * kLm];
    __shared__ __align__(16) double sB[kLdlTile * kLm];
    double* pair_tmp = tmp + (int64_t)blockIdx.y * h * h * kLdlTileElems;
    d4v acc[4] = {};
    const int m0 = second ? 0 : j, m1 = second ? i : h - 1;
    for (int m = m0; m <= m1; ++m) {
        // first: B_im A^-1_mj (m >= j); second: C^-1_im T_mj (m <= i)
        const double* pa = L + (second ? ldl_tile(d, blk, I, o + h + m) : ldl_tile(d, blk, I, o + m));
        const double* pb = second ? pair_tmp + (int64_t)(m * h + j) * kLdlTileElems : L + ldl_tile(d, blk, o + m, J);
        d2t va[8], vb[8];
        load_tile(pa, va);
        load_tile(pb, vb);
        __syncthreads();
        store_tile(sA, va);
        store_tile(sB, vb);
        __syncthreads();
        // a diagonal tile holds D where the inverse has ones
        const bool diag = second ? m == i : m == j;
        if (diag) {
            if (threadIdx.x < kLdlTile) (second ? sA : sB)[threadIdx.x * (kLm + 1)] = 1.0;
            __syncthreads();
        }
        tile_rows_ab(sA, sB, acc);
    }
    double* out = second ? L + ldl_tile(d, blk, I, J) : pair_tmp + (int64_t)(i * h + j) * kLdlTileElems;
    const int l = threadIdx.x & 63, r0 = 16 * (threadIdx.x >> 6) + (l >> 4), c = l & 15;
    const double sg = second ? -1.0 : 1.0;
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r) out[(r0 + 4 * r) * kLdlTile + 16 * b + c] = sg * acc[b][r];
}

// Sums of N values over the wavefront, N a power of two: the lanes first halve
// the number of values they hold at each exchange (N - 1 exchanges in all,
// against 6 N for N separate sums), then add within groups of 64 / N lanes.
// Lane l returns the total of a[l / (64 / N)].
template <int N>
__device__ __forceinline__ double rows_sum(double (&a)[N]) {
    const int l = threadIdx.x & 63;
    int o = kWave / 2;
#pragma unroll
    for (int m = N / 2; m >= 1; m >>= 1) {
        const bool up = (l & o) != 0;
#pragma unroll
        for (int i = 0; i < m; ++i) {
            const double give = up ? a[i] : a[i + m], keep = up ? a[i + m] : a[i];
            a[i] = keep + __shfl_xor(give, o, kWave);
        }
        o >>= 1;
    }
    double v = a[0];
#pragma unroll
    for (; o >= 1; o >>= 1) v += __shfl_xor(v, o, kWave);
    return v;
}

// x = L^-T D^-1 L^-1 b (ldl_solve, S/lower_tri_mat_meth.rs:194-227), S tile
// rows at a time: the diagonal super-blocks hold their inverses, so a block
// of S tile rows is two launches each way, a product with the inverse and the
// update of the rows (columns) the band couples it to, each spread over the
// chip; where one super-block covers a block it is one launch each way.
//   forward  z_s = Li_s y_s, w_s = z_s / d;  y_K -= sum_J L_KJ z_J below
//   backward x_s = Li_s^T w_s;               w_J -= sum_I L_IJ^T x_I above
// A workgroup of 4 wavefronts owns 16 rows (columns) of one tile row
// (column); the blocks are the grid's x, which takes any number of them (y ends at
// 65,536: one node a block reaches that on 65,537 nodes).  Every entry is written by one workgroup per launch and read by
// none of the same launch, so the result is deterministic.
//
// Bound by the factor's bytes, read twice, on many blocks and by the launches
// on few.  One CU streams tiles at only 20-45 GB/s here, so a step is spread
// over many workgroups: 58 blocks of 720 DOFs take 45 us a solve (6.6 TB/s of
// factor; 56 us with the blocks in the grid's y, a block's long and short rows
// dispatched together) against 118 us with one workgroup per block and 331 us
// with one launch per tile row and substitutions; one block of 31,248 DOFs, band 552,
// 1.28 ms in 245 launches against 13.5 ms in 978.

// Rows row0.. (4 of them) of tiles (I, ja..jb - 1) times the vector v (the
// block's, m entries): four tiles' loads in flight.
__device__ __forceinline__ void rows_dot(const LdlDesc& d, const double* __restrict__ L, int blk, int I, int ja,
                                         int jb, int row0, const double* __restrict__ v, int64_t m,
                                         double (&acc)[4]) {
    const int c = threadIdx.x & 63;
    for (int J = ja; J < jb; J += 4) {
        double a[4][4], x[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int Ju = J + u < jb ? J + u : jb - 1;
            const double* T = L + ldl_tile(d, blk, I, Ju) + row0 * kLdlTile + c;
#pragma unroll
            for (int p = 0; p < 4; ++p) a[u][p] = T[p * kLdlTile];
            const int64_t g = (int64_t)Ju * kLdlTile + c;
            x[u] = J + u < jb && g < m ? v[g] : 0.0;
        }
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int p = 0; p < 4; ++p) acc[p] = fma(a[u][p], x[u], acc[p]);
    }
}

// Columns c0.. (16 of them) of tiles (ia..ib - 1, J) transposed, times v: a
// lane takes column c0 + l % 16 of the rows 16 w + 4 u + l / 16.
__device__ __forceinline__ double cols_dot(const LdlDesc& d, const double* __restrict__ L, int blk, int J, int ia,
                                           int ib, int c0, const double* __restrict__ v, int64_t m) {
    const int l = threadIdx.x & 63, r0 = 16 * (threadIdx.x >> 6) + (l >> 4);
    double acc = 0.0;
    for (int I = ia; I < ib; I += 4) {
        double a[4][4], x[4][4];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const int It = I + t < ib ? I + t : ib - 1;
            const double* T = L + ldl_tile(d, blk, It, J) + r0 * kLdlTile + c0 + (l & 15);
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                a[t][u] = T[4 * u * kLdlTile];
                const int64_t g = (int64_t)It * kLdlTile + r0 + 4 * u;
                x[t][u] = I + t < ib && g < m ? v[g] : 0.0;
            }
        }
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int u = 0; u < 4; ++u) acc = fma(a[t][u], x[t][u], acc);
    }
    return acc;
}

// sum over the lanes of a column, then over the four wavefronts: the total of
// column c0 + t in threads t < 16
__device__ __forceinline__ double cols_total(double v) {
    __shared__ double red[4][16];
    const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
    v += __shfl_xor(v, 16, kWave);
    v += __shfl_xor(v, 32, kWave);
    if (l < 16) red[w][l] = v;
    __syncthreads();
    return threadIdx.x < 16 ? red[0][threadIdx.x] + red[1][threadIdx.x] + red[2][threadIdx.x] + red[3][threadIdx.x]
                            : 0.0;
}

// z_s = Li_s y_s and w_s = z_s / d over super-block sb (S tile rows)
__global__ __launch_bounds__(kBlock) void k_ldl_fwd_diag(LdlDesc d, const double* __restrict__ L, int S, int sb,
                                                         const double* __restrict__ y, double* __restrict__ z,
                                                         double* __restrict__ w, const int* __restrict__ done) {
    if (done && *done) return;
    const int blk = blockIdx.x, nt = ldl_block_nt(d, blk);
    const int I = sb * S + (blockIdx.y >> 2);
    if (I >= nt) return;
    const int64_t s = (int64_t)blk * d.bs, m = std::min(d.bs, d.n - s);
    const int c = threadIdx.x & 63, row0 = 16 * (blockIdx.y & 3) + 4 * (threadIdx.x >> 6);
    const double* TI = L + ldl_tile(d, blk, I, I);
    double li[4];
#pragma unroll
    for (int p = 0; p < 4; ++p) li[p] = TI[(row0 + p) * kLdlTile + c];
    const int row = row0 + (c >> 4);
    const double dr = TI[row * (kLdlTile + 1)];
    const int64_t gc = (int64_t)I * kLdlTile + c;
    const double yc = gc < m ? y[s + gc] : 0.0;
    double acc[4] = {};
    rows_dot(d, L, blk, I, sb * S, I, row0, y + s, m, acc);
#pragma unroll
    for (int p = 0; p < 4; ++p) acc[p] += c < row0 + p ? li[p] * yc : (c == row0 + p ? yc : 0.0);
    const double v = rows_sum<4>(acc);
    const int64_t g = (int64_t)I * kLdlTile + row;
    if ((c & 15) == 0 && g < m) {
        if (z) z[s + g] = v;
        w[s + g] = v / dr;
    }
}

// y_K -= sum over the super-block's tiles J of L_KJ z_J for the rows K below it
__global__ __launch_bounds__(kBlock) void k_ldl_fwd_band(LdlDesc d, const double* __restrict__ L, int S, int sb,
                                                         const double* __restrict__ z, double* __restrict__ y,
                                                         const int* __restrict__ done) {
    if (done && *done) return;
    const int blk = blockIdx.x, nt = ldl_block_nt(d, blk);
    const int K = (sb + 1) * S + (blockIdx.y >> 2);
    if (K >= nt) return;
    const int64_t s = (int64_t)blk * d.bs, m = std::min(d.bs, d.n - s);
    const int c = threadIdx.x & 63, row0 = 16 * (blockIdx.y & 3) + 4 * (threadIdx.x >> 6);
    double acc[4] = {};
    rows_dot(d, L, blk, K, max(sb * S, K - d.wt), (sb + 1) * S, row0, z + s, m, acc);
    const double v = rows_sum<4>(acc);
    const int64_t g = (int64_t)K * kLdlTile + row0 + (c >> 4);
    if ((c & 15) == 0 && g < m) y[s + g] -= v;
}

// x_s = Li_s^T w_s over super-block sb
__global__ __launch_bounds__(kBlock) void k_ldl_bwd_diag(LdlDesc d, const double* __restrict__ L, int S, int sb,
                                                         const double* __restrict__ w, double* __restrict__ x,
                                                         const int* __restrict__ done) {
    if (done && *done) return;
    const int blk = blockIdx.x, nt = ldl_block_nt(d, blk);
    const int J = sb * S + (blockIdx.y >> 2);
    if (J >= nt) return;
    const int64_t s = (int64_t)blk * d.bs, m = std::min(d.bs, d.n - s);
    const int l = threadIdx.x & 63, c0 = 16 * (blockIdx.y & 3), r0 = 16 * (threadIdx.x >> 6) + (l >> 4);
    const int col = c0 + (l & 15);
    // the diagonal tile: ones where it holds D
    double a[4], v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const int r = r0 + 4 * u;
        const int64_t g = (int64_t)J * kLdlTile + r;
        a[u] = L[ldl_tile(d, blk, J, J) + r * kLdlTile + col];
        v[u] = g < m ? w[s + g] : 0.0;
    }
    double acc = cols_dot(d, L, blk, J, J + 1, min((sb + 1) * S, nt), c0, w + s, m);
#pragma unroll
    for (int u = 0; u < 4; ++u) acc += r0 + 4 * u > col ? a[u] * v[u] : (r0 + 4 * u == col ? v[u] : 0.0);
    acc = cols_total(acc);
    const int64_t g = (int64_t)J * kLdlTile + c0 + threadIdx.x;
    if (threadIdx.x < 16 && g < m) x[s + g] = acc;
}

// w_J -= sum over the super-block's tiles I of L_IJ^T x_I for the columns J above it
__global__ __launch_bounds__(kBlock) void k_ldl_bwd_band(LdlDesc d, const double* __restrict__ L, int S, int sb,
                                                         const double* __restrict__ x, double* __restrict__ w,
                                                         const int* __restrict__ done) {
    if (done && *done) return;
    const int blk = blockIdx.x, nt = ldl_block_nt(d, blk);
    const int J = sb * S - 1 - (int)(blockIdx.y >> 2);
    if (J < 0 || sb * S >= nt) return;
    const int64_t s = (int64_t)blk * d.bs, m = std::min(d.bs, d.n - s);
    const int c0 = 16 * (blockIdx.y & 3);
    const int ib = min(min((sb + 1) * S, nt), J + d.wt + 1);
    const double v = cols_total(cols_dot(d, L, blk, J, sb * S, ib, c0, x + s, m));
    const int64_t g = (int64_t)J * kLdlTile + c0 + threadIdx.x;
    if (threadIdx.x < 16 && g < m) w[s + g] -= v;
}

__global__ __launch_bounds__(kBlock) void k_ldl_copy(int64_t n, const double* b, double* x, const int* done) {
    if (done && *done) return;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        x[i] = b[i];
}

}  // namespace

const char* ldl_plan(LdlDesc* d, int64_t* max_bw, int64_t n, int64_t block_dofs, const std::vector<int32_t>& h_rp,
                     const std::vector<int32_t>& h_bc) {
    if (n <= 0) return "empty operator";
    const int64_t n_rows = (int64_t)h_rp.size() - 1;
    if (3 * n_rows != n) return "operator rows are not 3-DOF block rows";
    const int64_t bs = (block_dofs <= 0 || block_dofs >= n) ? n : block_dofs;
    // envelope: first column of each row inside its block
    // (allocate_from_sparse_mat, S/lower_tri_mat_meth.rs:15-42)
    int64_t W = 1;
    for (int64_t R = 0; R < n_rows; ++R) {
        for (int a = 0; a < 3; ++a) {
            const int64_t i = 3 * R + a;
            const int64_t b0 = (i / bs) * bs;
            int64_t mc = i;
            for (int32_t k = h_rp[R]; k < h_rp[R + 1]; ++k) {
                const int64_t lo = 3 * (int64_t)h_bc[k], hi = lo + 2;
                if (hi < b0) continue;
                const int64_t cand = std::max(lo, b0);
                if (cand < mc) mc = cand;
            }
            W = std::max(W, i - mc + 1);
        }
    }
    d->n = n;
    d->bs = bs;
    d->n_blocks = (int)((n + bs - 1) / bs);
    d->nt_full = (int)((bs + kLdlTile - 1) / kLdlTile);
    d->wt = (int)std::min<int64_t>((W - 1 + kLdlTile - 1) / kLdlTile, d->nt_full - 1);
    if (d->wt > kLdlMaxWt) return "bandwidth exceeds the device solve's window (kLdlMaxWt tiles)";
    d->stride = ldl_row_off(d->nt_full, d->wt) * kLdlTileElems;
    *max_bw = W;
    return nullptr;
}

void ldl_fill(hipStream_t st, const LdlDesc& d, int n_rows, int n_slices, const int32_t* sptr, const int32_t* scol,
              const double* K, double* L) {
    (void)hipMemsetAsync(L, 0, (size_t)d.n_blocks * d.stride * sizeof(double), st);
    hipLaunchKernelGGL(k_ldl_fill, dim3(n_slices), dim3(kWave), 0, st, d, n_rows, sptr, scol, K, L);
    hipLaunchKernelGGL(k_ldl_pad, dim3(d.n_blocks), dim3(kLdlTile), 0, st, d, L);
}

static void ldl_invert_launch(hipStream_t st, const LdlDesc& d, double* L, double* tmp);

void ldl_factor_launch(hipStream_t st, const LdlDesc& d, double* L, double* tmp, int32_t* neg) {
    (void)hipMemsetAsync(neg, 0, sizeof(int32_t), st);
    hipLaunchKernelGGL(k_ldl_diag, dim3(d.n_blocks), dim3(kBlock), 0, st, d, L, neg);
    for (int k = 0; k < d.nt_full; ++k) {
        const int r = std::min(d.wt, d.nt_full - 1 - k);
        if (r <= 0) continue;
        hipLaunchKernelGGL(k_ldl_panel, dim3(d.n_blocks, r), dim3(kBlock), 0, st, d, k, L);
        hipLaunchKernelGGL(k_ldl_update, dim3(d.n_blocks, r * (r + 1) / 2), dim3(kBlock), 0, st, d, k, L, neg);
    }
    ldl_invert_launch(st, d, L, tmp);
}

int ldl_super(const LdlDesc& d) {
    int S = 1;
    if (d.nt_full <= kLdlWholeTiles && d.wt >= d.nt_full - 1) {
        while (S < d.nt_full) S *= 2;  // one super-block per block
    } else {
        while (2 * S <= kLdlSuperTiles && 2 * S <= d.wt + 1) S *= 2;
    }
    return S;
}

int64_t ldl_tmp_tiles(const LdlDesc& d) {
    const int S = ldl_super(d);
    if (S < 2) return 1;
    const int64_t pairs = (int64_t)d.n_blocks * ((d.nt_full + 1) / 2);
    // every pair of the first level or, for the wider ones, a share at a time
    return std::max<int64_t>((int64_t)(S / 2) * (S / 2), std::min<int64_t>(pairs * (S / 2), kLdlTmpTiles));
}

// super-block inverses over the finished factor (see k_ldl_inv)
static void ldl_invert_launch(hipStream_t st, const LdlDesc& d, double* L, double* tmp) {
    const int S = ldl_super(d);
    const int64_t room = ldl_tmp_tiles(d);
    for (int h = 1; h < S; h *= 2) {
        const int pairs = (d.nt_full + 2 * h - 1) / (2 * h);
        const int64_t all = (int64_t)pairs * d.n_blocks;
        const int64_t step = std::min<int64_t>(std::max<int64_t>(1, room / ((int64_t)h * h)), 65535);
        for (int64_t p0 = 0; p0 < all; p0 += step) {
            const dim3 grid(h * h, (unsigned)std::min(step, all - p0));
            hipLaunchKernelGGL(k_ldl_inv, grid, dim3(kBlock), 0, st, d, h, pairs, p0, 0, L, tmp);
            hipLaunchKernelGGL(k_ldl_inv, grid, dim3(kBlock), 0, st, d, h, pairs, p0, 1, L, tmp);
        }
    }
}

void ldl_solve_launch(hipStream_t st, const LdlDesc& d, const double* L, const double* b, double* x, double* work,
                      const int* done) {
    const int S = ldl_super(d);
    const int ns = (d.nt_full + S - 1) / S;
    double *w = work, *y = work + d.n, *z = work + 2 * d.n;
    const dim3 diag(d.n_blocks, 4 * S);
    if (ns == 1) {
        hipLaunchKernelGGL(k_ldl_fwd_diag, diag, dim3(kBlock), 0, st, d, L, S, 0, b, (double*)nullptr, w, done);
        hipLaunchKernelGGL(k_ldl_bwd_diag, diag, dim3(kBlock), 0, st, d, L, S, 0, w, x, done);
        return;
    }
    hipLaunchKernelGGL(k_ldl_copy, dim3(1024), dim3(kBlock), 0, st, d.n, b, y, done);
    for (int s = 0; s < ns; ++s) {
        hipLaunchKernelGGL(k_ldl_fwd_diag, diag, dim3(kBlock), 0, st, d, L, S, s, y, z, w, done);
        const int rows = std::min(d.wt, d.nt_full - (s + 1) * S);
        if (rows > 0)
            hipLaunchKernelGGL(k_ldl_fwd_band, dim3(d.n_blocks, 4 * rows), dim3(kBlock), 0, st, d, L, S, s, z, y,
                               done);
    }
    for (int s = ns - 1; s >= 0; --s) {
        hipLaunchKernelGGL(k_ldl_bwd_diag, diag, dim3(kBlock), 0, st, d, L, S, s, w, x, done);
        const int cols = std::min(d.wt, s * S);
        if (cols > 0)
            hipLaunchKernelGGL(k_ldl_bwd_band, dim3(d.n_blocks, 4 * cols), dim3(kBlock), 0, st, d, L, S, s, x, w,
                               done);
    }
}

}  // namespace asend
