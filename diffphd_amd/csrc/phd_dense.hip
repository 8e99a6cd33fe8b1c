// Dense SPD solve for the contact system: blocked right-looking Cholesky with
// the right-hand side as an extra block row, then blocked backward substitution.
#include "phd_dense.h"

#include <cstring>
#include <type_traits>

namespace phd {
namespace {

constexpr int CB = kCholBlock;

template <class TV, class TH>
__global__ void __launch_bounds__(256) k_chol_assemble(int nJ, int np, int64_t lda, const int* __restrict__ J,
                                                       const TH* __restrict__ H, int K, const double* __restrict__ nrm,
                                                       const double* __restrict__ om, const double* __restrict__ E,
                                                       const double* __restrict__ rhs, TV* __restrict__ M) {
    const int64_t rows = (int64_t)np + CB;
    const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= rows * np) return;
    const int r = (int)(idx % rows), c = (int)(idx / rows);
    double v;
    if (r < c) {
        v = 0.0;
    } else if (r >= np) {
        v = (r == np && c < nJ) ? rhs[c] : 0.0;
    } else if (r >= nJ || c >= nJ) {
        v = (r == c) ? 1.0 : 0.0;
    } else {
        const int i = J[r], j = J[c];
        const double nd = nrm ? nrm[3 * i] * nrm[3 * j] + nrm[3 * i + 1] * nrm[3 * j + 1] + nrm[3 * i + 2] * nrm[3 * j + 2]
                              : 1.0;
        // H is symmetric: read along its row j so that consecutive r stay close
        v = om[i] * nd * (double)H[(int64_t)j * K + i] * om[j];
        if (r == c) v += E[i];
    }
    M[r + (int64_t)c * lda] = (TV)v;
}

__device__ __forceinline__ float lane_bcast(float v, int l) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}
__device__ __forceinline__ double lane_bcast(double v, int l) {
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readlane((int)b, l), hi = __builtin_amdgcn_readlane((int)(b >> 32), l);
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

// 1 / sqrt(p) for the pivots: the hardware reciprocal square root (1 ulp in
// FP32); in FP64 refined by two Newton steps y <- y (3 - p y^2) / 2.
__device__ __forceinline__ float pivot_rsqrt(float p) { return __builtin_amdgcn_rsqf(p); }
__device__ __forceinline__ double pivot_rsqrt(double p) {
    double y = __builtin_amdgcn_rsq(p);
    const double h = 0.5 * p;
    y = y * (1.5 - h * y * y);
    y = y * (1.5 - h * y * y);
    return y;
}

template <class TV> struct V16;
template <> struct V16<float> { using type = float4; static constexpr int N = 4; };
template <> struct V16<double> { using type = double2; static constexpr int N = 2; };

constexpr int kTSB = CB + 4;             // row stride of the published L columns (16-byte aligned rows)

// ---- The FP32 panel in 16-column sub-blocks --------------------------------
// The diagonal wave (lane r holds row r of the diagonal block in z) factors
// sub-block SB's 16 columns with readlane pivots and rank-1 updates restricted
// to those columns, so a step waits on register broadcasts only; L(r, j)
// replaces z[j] (0 above the diagonal) and inv[jj] = 1 / L(j, j).
template <class TV, int SB>
__device__ __forceinline__ void diag_chain(TV (&z)[CB], int r, bool& bad_any, TV& inv_mine) {
#pragma unroll
    for (int jj = 0; jj < 16; ++jj) {
        const int j = 16 * SB + jj;
        const TV p = lane_bcast(z[j], j);
        const bool bad = !(p > TV(0));
        bad_any |= bad;
        const TV iv = bad ? TV(1) : pivot_rsqrt(p);
        if (r == j) inv_mine = iv;
        const TV l = (r > j) ? z[j] * iv : (r == j ? p * iv : TV(0));
        z[j] = l;
#pragma unroll
        for (int m = j + 1; m < 16 * SB + 16; ++m) z[m] -= l * lane_bcast(l, m);
    }
}

// Sub-block SB of L through LDS: Lt[j][m] = L(m, j), invp[j] = 1 / L(j, j)
// (lane j holds its own pivot's inverse).
template <class TV, int SB>
__device__ __forceinline__ void diag_publish(const TV (&z)[CB], int r, TV inv_mine, TV (*Lt)[kTSB], TV* invp) {
#pragma unroll
    for (int jj = 0; jj < 16; ++jj) Lt[16 * SB + jj][r] = z[16 * SB + jj];
    if (r >= 16 * SB && r < 16 * SB + 16) invp[r] = inv_mine;
}

__device__ __forceinline__ float vget(const float4& t, int e) { return e == 0 ? t.x : e == 1 ? t.y : e == 2 ? t.z : t.w; }
__device__ __forceinline__ double vget(const double2& t, int e) { return e == 0 ? t.x : t.y; }

// The block-row wave's forward substitution on sub-block SB: X(r, j) =
// (B(r, j) - sum_{i<j} X(r, i) L(j, i)) / L(j, j), right-looking within the
// sub-block; X is written to out (column-major, out_ld).
template <class TV, int SB>
__device__ __forceinline__ void row_solve(TV (&z)[CB], const TV (*Lt)[kTSB], const TV* invp, int r, TV* out,
                                          int64_t out_ld) {
    using VT = typename V16<TV>::type;
    constexpr int VN = V16<TV>::N, NV = 16 / VN, j0 = 16 * SB;
    // the sub-block's pivot inverses and L row j + 1 are read while row j is
    // applied, so each step waits on registers, not on LDS
    VT ip[NV], cur[NV], nxt[NV];
#pragma unroll
    for (int e = 0; e < NV; ++e) {
        ip[e] = reinterpret_cast<const VT*>(invp + j0)[e];
        cur[e] = reinterpret_cast<const VT*>(&Lt[j0][j0])[e];
    }
#pragma unroll
    for (int jj = 0; jj < 16; ++jj) {
        const int j = j0 + jj;
        if (jj + 1 < 16) {
#pragma unroll
            for (int e = 0; e < NV; ++e) nxt[e] = reinterpret_cast<const VT*>(&Lt[j + 1][j0])[e];
        }
        const TV x = z[j] * vget(ip[jj / VN], jj % VN);
        z[j] = x;
        out[r + (int64_t)j * out_ld] = x;
#pragma unroll
        for (int m = jj + 1; m < 16; ++m) z[j0 + m] -= x * vget(cur[m / VN], m % VN);
#pragma unroll
        for (int e = 0; e < NV; ++e) cur[e] = nxt[e];
    }
}

constexpr int kTS = CB + 4;  // LDS tile row stride (16-byte aligned rows)

// The 64 x 64 block at (r0, c0) into registers (256 threads, all loads in flight), and
// from there into LDS as S[l][row] = M(r0 + row, c0 + l).
template <class TV>
__device__ __forceinline__ void load_block(const TV* __restrict__ M, int64_t lda, int64_t r0, int64_t c0,
                                           TV (&v)[CB * CB / 256]) {
#pragma unroll
    for (int u = 0; u < CB * CB / 256; ++u) {
        const int e = (int)threadIdx.x + 256 * u;
        v[u] = M[r0 + e % CB + (c0 + e / CB) * lda];
    }
}
template <class TV>
__device__ __forceinline__ void store_block(const TV (&v)[CB * CB / 256], TV (*S)[kTS]) {
#pragma unroll
    for (int u = 0; u < CB * CB / 256; ++u) {
        const int e = (int)threadIdx.x + 256 * u;
        S[e / CB][e % CB] = v[u];
    }
}

template <class TV>
__device__ __forceinline__ void stage_block(const TV* __restrict__ M, int64_t lda, int64_t r0, int64_t c0,
                                            TV (*S)[kTS]) {
    TV v[CB * CB / 256];
    load_block<TV>(M, lda, r0, c0, v);
    store_block<TV>(v, S);
}

// FP64 rank-64 tile product: acc[u][v] = sum_l A[l][4 tx + u] B[l][4 ty + v], l
// ascending; thread (tx, ty) of 16 x 16. Four by four outputs per thread take four
// 16-byte LDS reads for 16 FMAs (a row of 16 columns per thread took nine).
__device__ __forceinline__ void tile_product(const double (*A)[kTS], const double (*B)[kTS], int tx, int ty,
                                             double (&acc)[4][4]) {
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int v = 0; v < 4; ++v) acc[u][v] = 0;
#pragma unroll 4
    for (int l = 0; l < CB; ++l) {
        double a[4], b[4];
        memcpy(a, &A[l][4 * tx], sizeof(a));
        memcpy(b, &B[l][4 * ty], sizeof(b));
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int v = 0; v < 4; ++v) acc[u][v] += a[u] * b[v];
    }
}

// FP32 rank-64 tile product on the matrix cores: C(row, col) = sum_l
// A[l][row] B[l][col], wave w owning rows 32 (w / 2) .. and columns
// 32 (w % 2) .. of the 64 x 64 tile. v_mfma_f32_32x32x2f32 is fed the
// transposed product D = C^T block (operand A lane i + 32 h = B[l][32 wj + i],
// operand B lane j + 32 h = A[l][32 wi + j], l = 2 s + h at step s), so that
// result register v of lane L holds C(32 wi + (L % 32), 32 wj + mfma_col(v, L)):
// the 32 lanes of a half-wave hold 32 consecutive rows of one column of the
// column-major matrix.
typedef float f32x16 __attribute__((ext_vector_type(16)));

__device__ __forceinline__ int mfma_col(int v, int lane) { return (v & 3) + 4 * (lane >> 5) + 8 * (v >> 2); }

__device__ __forceinline__ f32x16 tile_product_mfma(const float (*A)[kTS], const float (*B)[kTS], int wave, int lane) {
    const int wi = wave >> 1, wj = wave & 1, i = lane & 31, h = lane >> 5;
    // two accumulation chains (steps st and st + CB / 4) so that consecutive
    // MFMAs do not wait on each other's results
    f32x16 acc0, acc1;
#pragma unroll
    for (int v = 0; v < 16; ++v) acc0[v] = acc1[v] = 0.f;
#pragma unroll 4
    for (int st = 0; st < CB / 4; ++st) {
        const int l0 = 2 * st + h, l1 = CB / 2 + 2 * st + h;
        acc0 = __builtin_amdgcn_mfma_f32_32x32x2f32(B[l0][32 * wj + i], A[l0][32 * wi + i], acc0, 0, 0, 0);
        acc1 = __builtin_amdgcn_mfma_f32_32x32x2f32(B[l1][32 * wj + i], A[l1][32 * wi + i], acc1, 0, 0, 0);
    }
    return acc0 + acc1;
}

// Exchange of the upper half-wave of x with the lower half-wave of y
// (v_permlane32_swap_b32): x <- [x.lo, y.lo], y <- [x.hi, y.hi].
__device__ __forceinline__ void swap_halves(float& x, float& y) {
    const auto p = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(y), false, false);
    x = __uint_as_float(p[0]);
    y = __uint_as_float(p[1]);
}

// z[m] -= C(r, m) for the columns m >= M0 of column tile TJ (m = 32 TJ ..
// 32 TJ + 31), given the tile's two row halves in the MFMA result layout (lo:
// rows 0..31, hi: rows 32..63; register v of lane L holds row 32 t + L % 32,
// column 32 TJ + mfma_col(v, L)). One half-wave swap per register pair puts
// row r in lane r: afterwards x holds column 32 TJ + c and y column 32 TJ + c + 4.
template <int TJ, int M0>
__device__ __forceinline__ void trail_apply(float (&z)[CB], const f32x16& lo, const f32x16& hi) {
#pragma unroll
    for (int v = 0; v < 16; ++v) {
        const int c = 32 * TJ + (v & 3) + 8 * (v >> 2);
        if (c + 4 < M0) continue;
        float x = lo[v], y = hi[v];
        swap_halves(x, y);
        if (c >= M0) z[c] -= x;
        z[c + 4] -= y;
    }
}

// The panel's rank-16 updates on the matrix cores, C(r, m) = sum_j P(r, j)
// L(m, j) over sub-block SB's columns j for the columns m right of it, as
// 32 x 32 tiles of v_mfma_f32_32x32x2f32 (step s covers j = 16 SB + 2 s + h,
// h the half-wave). Operand lane i + 32 h of a row tile t is P(32 t + i, j):
// the half-wave swap of the register pair (z[j0 + 2 s], z[j0 + 2 s + 1]) gives
// both row tiles of step s at once.
// Diagonal wave: P = L (its own rows), only the lower part m <= r matters, so
// the column tile 32..63 needs only the row tile 32..63.
template <int SB>
__device__ __forceinline__ void diag_trail_mfma(float (&z)[CB]) {
    constexpr int j0 = 16 * SB, M0 = 16 * (SB + 1);
    float p0[8], p1[8];
#pragma unroll
    for (int s = 0; s < 8; ++s) {
        p0[s] = z[j0 + 2 * s];
        p1[s] = z[j0 + 2 * s + 1];
        swap_halves(p0[s], p1[s]);
    }
    f32x16 zero;
#pragma unroll
    for (int v = 0; v < 16; ++v) zero[v] = 0.f;
    if constexpr (M0 < 32) {
        f32x16 a0 = zero, a1 = zero;
#pragma unroll
        for (int s = 0; s < 8; ++s) {
            a0 = __builtin_amdgcn_mfma_f32_32x32x2f32(p0[s], p0[s], a0, 0, 0, 0);
            a1 = __builtin_amdgcn_mfma_f32_32x32x2f32(p0[s], p1[s], a1, 0, 0, 0);
        }
        trail_apply<0, M0>(z, a0, a1);
    }
    f32x16 a1 = zero;
#pragma unroll
    for (int s = 0; s < 8; ++s) a1 = __builtin_amdgcn_mfma_f32_32x32x2f32(p1[s], p1[s], a1, 0, 0, 0);
    trail_apply<1, M0>(z, zero, a1);
}

// Block-row wave: P = X (its rows of the solved block row), L(m, j) read from
// the published columns, Lt[j][m] = L(m, j), one 4-byte read per lane and step.
template <int SB>
__device__ __forceinline__ void row_trail_mfma(float (&z)[CB], const float (*Lt)[kTSB], int lane) {
    constexpr int j0 = 16 * SB, M0 = 16 * (SB + 1);
    const int i = lane & 31, h = lane >> 5;
    float p0[8], p1[8];
#pragma unroll
    for (int s = 0; s < 8; ++s) {
        p0[s] = z[j0 + 2 * s];
        p1[s] = z[j0 + 2 * s + 1];
        swap_halves(p0[s], p1[s]);
    }
    f32x16 zero;
#pragma unroll
    for (int v = 0; v < 16; ++v) zero[v] = 0.f;
#pragma unroll
    for (int tj = M0 / 32; tj < 2; ++tj) {
        float l[8];
#pragma unroll
        for (int s = 0; s < 8; ++s) l[s] = Lt[j0 + 2 * s + h][32 * tj + i];
        f32x16 a0 = zero, a1 = zero;
#pragma unroll
        for (int s = 0; s < 8; ++s) {
            a0 = __builtin_amdgcn_mfma_f32_32x32x2f32(l[s], p0[s], a0, 0, 0, 0);
            a1 = __builtin_amdgcn_mfma_f32_32x32x2f32(l[s], p1[s], a1, 0, 0, 0);
        }
        if (tj == 0) trail_apply<0, M0>(z, a0, a1);
        else trail_apply<1, M0>(z, a0, a1);
    }
}

// Updates of steps kp0 .. kp1 - 1 on block (ib, jb), in step order: A_ij -= L_{i,kp}
// L_{j,kp}^T (256 threads; the staging tiles are S0 and S1). The block is read and
// written once for all of them. FP64, with two workgroups per CU, loads the next
// step's operands during the product; FP32 has four to overlap and no registers left.
template <class TV>
__device__ __forceinline__ void update_block(TV* __restrict__ M, int64_t lda, int kp0, int kp1, int ib, int jb, TV (*S0)[kTS],
                                             TV (*S1)[kTS]) {
    const int t = threadIdx.x;
    const int64_t ri = (int64_t)ib * CB, rj = (int64_t)jb * CB;
    if constexpr (std::is_same<TV, float>::value) {
        const int lane = t % 64, wave = t / 64;
        float* dst = M + ri + 32 * (wave >> 1) + (lane & 31) + (rj + 32 * (wave & 1)) * lda;
        float val[16];
#pragma unroll
        for (int v = 0; v < 16; ++v) val[v] = dst[mfma_col(v, lane) * lda];
#pragma unroll 1
        for (int kp = kp0; kp < kp1; ++kp) {
            stage_block<TV>(M, lda, ri, (int64_t)kp * CB, S0);
            stage_block<TV>(M, lda, rj, (int64_t)kp * CB, S1);
            __syncthreads();
            const f32x16 acc = tile_product_mfma(S0, S1, wave, lane);
#pragma unroll
            for (int v = 0; v < 16; ++v) val[v] -= acc[v];
            if (kp + 1 < kp1) __syncthreads();
        }
#pragma unroll
        for (int v = 0; v < 16; ++v) dst[mfma_col(v, lane) * lda] = val[v];
    } else {
        const int tx = t % 16, ty = t / 16;
        TV a[CB * CB / 256], b[CB * CB / 256];
        load_block<TV>(M, lda, ri, (int64_t)kp0 * CB, a);
        load_block<TV>(M, lda, rj, (int64_t)kp0 * CB, b);
        TV* dst = M + ri + 4 * tx + (rj + 4 * ty) * lda;
        TV val[4][4], acc[4][4];
#pragma unroll
        for (int v = 0; v < 4; ++v)
#pragma unroll
            for (int u = 0; u < 4; ++u) val[u][v] = dst[u + v * lda];
#pragma unroll 1
        for (int kp = kp0; kp < kp1; ++kp) {
            store_block<TV>(a, S0);
            store_block<TV>(b, S1);
            __syncthreads();
            if (kp + 1 < kp1) {
                load_block<TV>(M, lda, ri, (int64_t)(kp + 1) * CB, a);
                load_block<TV>(M, lda, rj, (int64_t)(kp + 1) * CB, b);
            }
            tile_product(S0, S1, tx, ty, acc);
#pragma unroll
            for (int v = 0; v < 4; ++v)
#pragma unroll
                for (int u = 0; u < 4; ++u) val[u][v] -= acc[u][v];
            if (kp + 1 < kp1) __syncthreads();
        }
#pragma unroll
        for (int v = 0; v < 4; ++v)
#pragma unroll
            for (int u = 0; u < 4; ++u) dst[u + v * lda] = val[u][v];
    }
}

// The rows below the matrix (block rows T, T + 1, ...) are either one right-hand-side
// block row, or (INV) the identity, one block row per block column: L^-1 rhs and
// Y = L^-T come out of the factorization there. Block row T + i of Y starts at
// column i, so the updates of steps up to kp reach kp + 1 of its block rows.
//
// Trailing updates of one launch. Every block (i, j) takes the steps 0 .. j - 2 in
// order before the panel of column j (which applies step j - 1 itself). They come in
// groups of kGroup steps, so that a trailing block is read and written once per group
// and not once per step (which bound the launches with many blocks: 45 us against the
// panel's 14 at 95 block columns in FP32). Launch k = g + r, g the group's first step:
//  * due now: r = 0: the previous group's steps on the columns g + 1 .. g + kGroup;
//    r > 0: the steps g .. k - 1 on column k + 1;
//  * due before launch g + kGroup: the previous group's steps on the columns beyond,
//    the r-th of kGroup equal shares.
constexpr int kGroup = 4;

struct TrailPart {
    int ndue, nlazy, lazy0;  // blocks due now, blocks of this launch's share and the first of them
};
// blocks of the columns j0 <= j < j1: rows j .. T - 1 and `extra` rows below
__host__ __device__ inline int column_blocks(int T, int extra, int j0, int j1) {
    return j1 <= j0 ? 0 : (j1 - j0) * (T + extra) - (j0 + j1 - 1) * (j1 - j0) / 2;
}
template <bool INV>
__host__ __device__ inline TrailPart trail_part(int k, int T) {
    const int r = k % kGroup, g = k - r;
    TrailPart p{0, 0, 0};
    if (r > 0) p.ndue = k + 1 < T ? column_blocks(T, INV ? k : 1, k + 1, k + 2) : 0;
    else if (k > 0) p.ndue = column_blocks(T, INV ? g : 1, k + 1, k + 1 + kGroup < T ? k + 1 + kGroup : T);
    if (g > 0) {
        const int n = column_blocks(T, INV ? g : 1, g + kGroup + 1, T);
        p.lazy0 = (int)((int64_t)n * r / kGroup);
        p.nlazy = (int)((int64_t)n * (r + 1) / kGroup) - p.lazy0;
    }
    return p;
}

// The FP64 panel in LDS: D the diagonal block, R the block row (or the identity), both
// [row][column]. Stage s: wave 0 factors the 16 columns of sub-block s in registers
// (readlane broadcasts), wave 1 solves the block row against sub-block s - 1; then all
// four waves apply both rank-16 updates to the columns on the right, 4 x 4 entries per
// thread, j ascending (each entry sees the operations of one rank-1 update per column
// in column order). A row of the block in registers (64 doubles) would leave two waves
// idle and spills; one pivot per barrier took 38 us a step, this takes 17 us.
constexpr int kLS = 18;  // row stride of a published 16 x 16 diagonal sub-block

__device__ __forceinline__ void panel64(double (*D)[kTS], double (*R)[kTS], double (*Ls)[16][kLS], double* invp, int w,
                                        double* out, int64_t out_ld, int* __restrict__ fail) {
    const int t = threadIdx.x, wave = t / 64, r = t % 64;
    bool bad_any = false;
#pragma unroll 1
    for (int s = 0; s <= 4; ++s) {
        const int q = s - 1;
        if (wave == 0 && s < 4) {
            double z[16], inv = 1.0;
            memcpy(z, &D[r][16 * s], sizeof(z));
#pragma unroll
            for (int jj = 0; jj < 16; ++jj) {
                const int j = 16 * s + jj;
                const double p = lane_bcast(z[jj], j);
                const bool bad = !(p > 0.0);
                bad_any |= bad;
                const double iv = bad ? 1.0 : pivot_rsqrt(p);
                if (r == j) inv = iv;
                const double l = (r > j) ? z[jj] * iv : (r == j ? p * iv : 0.0);
                z[jj] = l;
#pragma unroll
                for (int m = jj + 1; m < 16; ++m) z[m] -= l * lane_bcast(l, 16 * s + m);
            }
            memcpy(&D[r][16 * s], z, sizeof(z));
            if (r / 16 == s) {
                invp[r] = inv;
#pragma unroll
                for (int jj = 0; jj < 16; ++jj) Ls[s & 1][jj][r % 16] = z[jj];
            }
        } else if (wave == 1 && s > 0) {
            double z[16];
            memcpy(z, &R[r][16 * q], sizeof(z));
#pragma unroll
            for (int jj = 0; jj < 16; ++jj) {
                const double x = z[jj] * invp[16 * q + jj];
                z[jj] = x;
                out[r + (int64_t)(16 * q + jj) * out_ld] = x;
#pragma unroll
                for (int m = jj + 1; m < 16; ++m) z[m] -= x * Ls[q & 1][jj][m];
            }
            memcpy(&R[r][16 * q], z, sizeof(z));
        }
        if (s == 4) break;
        __syncthreads();
        const int cd = 4 * (3 - s), cr = s > 0 ? 4 * (4 - s) : 0;  // column groups right of s / of q
        for (int tile = t; tile < 16 * (cd + cr); tile += 256) {
            const int tx = tile % 16, g = tile / 16;
            const bool diag = g < cd;
            double (*A)[kTS] = diag ? D : R;
            const int j0 = diag ? 16 * s : 16 * q, c0 = 16 * s + (diag ? 16 + 4 * g : 4 * (g - cd));
            double acc[4][4];
#pragma unroll
            for (int u = 0; u < 4; ++u) memcpy(acc[u], &A[tx + 16 * u][c0], sizeof(acc[u]));
#pragma unroll 4
            for (int j = 0; j < 16; j += 2) {
                double a[4][2], b[4][2];
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    memcpy(a[u], &A[tx + 16 * u][j0 + j], sizeof(a[u]));
                    memcpy(b[u], &D[c0 + u][j0 + j], sizeof(b[u]));
                }
#pragma unroll
                for (int e = 0; e < 2; ++e)
#pragma unroll
                    for (int u = 0; u < 4; ++u)
#pragma unroll
                        for (int v = 0; v < 4; ++v) acc[u][v] -= a[u][e] * b[v][e];
            }
#pragma unroll
            for (int u = 0; u < 4; ++u) memcpy(&A[tx + 16 * u][c0], acc[u], sizeof(acc[u]));
        }
        __syncthreads();
    }
    if (wave == 0 && bad_any && w == 0 && r == 0) fail[0] = 1;
}

// Step k of the factorization, one launch of 256-thread workgroups in two parts
// that touch disjoint blocks, so the panel of step k runs next to trailing updates
// of earlier steps:
//  * workgroups w < T - k + 1, INV w < T (panel of block column k): the rank-64 update of
//    step k - 1 is applied here, in LDS, to the two blocks the workgroup
//    reads: the diagonal block (k, k) (every workgroup repeats it) and block
//    (k + 1 + w, k); w = T - k - 1 is the right-hand-side block row and
//    w = T - k the identity. Then wave 0 factors the diagonal block and
//    wave 1 solves X L_kk^T = B, writing L(k + 1 + w, k) into M, or
//    Xinv_k = L_kk^-T (column-major 64 x 64) for the identity. Both work in
//    16-column sub-blocks: wave 0 runs each sub-block's pivot chain on
//    readlane broadcasts and publishes its columns through LDS, wave 1
//    solves against them one sub-block behind, and the rank-16 update of the
//    columns to the right follows (FP32 as MFMA tiles of the same two waves,
//    FP64 see panel64);
//  * the remaining workgroups apply trailing updates (trail_part), none of them of
//    step k or to column k.
// Four workgroups per CU in FP32 (the MFMA accumulators stay in VGPRs, so the
// update workgroups of a step run at four waves per SIMD), two in FP64, whose staging
// tiles allow no more.
template <class TV, bool INV>
__global__ void __launch_bounds__(256, sizeof(TV) == 8 ? 2 : 4) k_chol_step(int k, int T, int64_t lda, TV* __restrict__ M,
                                                   TV* __restrict__ Xinv, int* __restrict__ fail) {
    __shared__ __align__(16) TV S0[CB][kTS];
    __shared__ __align__(16) TV S1[CB][kTS];
    __shared__ __align__(16) TV invp[CB];
    __shared__ __align__(16) TV Ls[sizeof(TV) == 8 ? 2 : 1][16][kLS];  // FP64 only
    const int t = threadIdx.x;
    const int NP = INV ? T : T - k + 1;
    const int kp = k - 1;
    if ((int)blockIdx.x >= NP) {
        const TrailPart p = trail_part<INV>(k, T);
        const int rr = k % kGroup, g = k - rr;
        int u = (int)blockIdx.x - NP, jb, kp0 = g - kGroup, kp1 = g;
        if (u < p.ndue) {
            jb = k + 1;
            if (rr > 0) { kp0 = g; kp1 = k; }
        } else {
            u += p.lazy0 - p.ndue;
            jb = g + kGroup + 1;
        }
        const int extra = INV ? kp1 : 1;
        for (int cnt = T - jb + extra; u >= cnt; cnt = T - jb + extra) { u -= cnt; ++jb; }
        // a block row of Y takes no part in the steps before its first column
        if (INV && jb + u >= T) kp0 = max(kp0, jb + u - T);
        update_block<TV>(M, lda, kp0, kp1, jb + u, jb, S0, S1);
        return;
    }
    const int w = blockIdx.x;
    const int wave = t / 64, r = t % 64;
    const int role = wave < 2 ? wave : 2;
    // block row k + 1 + w of M, which INV continues with the first k + 1 of Y; without
    // INV the last workgroup has the identity instead
    const bool has_row = INV || w < T - k;
    const int64_t c0 = (int64_t)k * CB, i0 = (int64_t)(k + 1 + w) * CB;
    if constexpr (std::is_same<TV, double>::value) {
        const int ux = t % 16, uy = t / 16;
        TV aD[4][4], aR[4][4];
#pragma unroll
        for (int v = 0; v < 4; ++v)
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int64_t off = 4 * ux + u + (c0 + 4 * uy + v) * lda;
                aD[u][v] = M[c0 + off];
                aR[u][v] = has_row ? M[i0 + off] : (u + 4 * ux == v + 4 * uy ? TV(1) : TV(0));
            }
        if (k > 0) {
            TV accD[4][4], accR[4][4];
            stage_block<TV>(M, lda, c0, (int64_t)kp * CB, S0);
            if (has_row) stage_block<TV>(M, lda, i0, (int64_t)kp * CB, S1);
            __syncthreads();
            tile_product(S0, S0, ux, uy, accD);
            if (has_row) tile_product(S1, S0, ux, uy, accR);
            __syncthreads();
#pragma unroll
            for (int u = 0; u < 4; ++u)
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    aD[u][v] -= accD[u][v];
                    if (has_row) aR[u][v] -= accR[u][v];
                }
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            memcpy(&S0[4 * ux + u][4 * uy], aD[u], sizeof(aD[u]));
            memcpy(&S1[4 * ux + u][4 * uy], aR[u], sizeof(aR[u]));
        }
        __syncthreads();
        panel64(S0, S1, Ls, invp, w, has_row ? M + i0 + c0 * lda : Xinv + (int64_t)k * CB * CB, has_row ? lda : CB, fail);
        return;
    } else {
    TV z[CB];
    using VT = typename V16<TV>::type;
    constexpr int VN = V16<TV>::N;
    if (k > 0) {
        // FP32: the two target blocks are read together with the staging loads
        const int row = 32 * (wave >> 1) + (r & 31);
        float aD[16], aR[16];
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            const int64_t off = row + (c0 + 32 * (wave & 1) + mfma_col(v, r)) * lda;
            aD[v] = M[c0 + off];
            aR[v] = has_row ? M[i0 + off] : 0.f;
        }
        stage_block<TV>(M, lda, c0, (int64_t)kp * CB, S0);
        if (has_row) stage_block<TV>(M, lda, i0, (int64_t)kp * CB, S1);
        __syncthreads();
        const f32x16 accD = tile_product_mfma(S0, S0, wave, r);
        f32x16 accR;
        if (has_row) accR = tile_product_mfma(S1, S0, wave, r);
        __syncthreads();
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            const int col = 32 * (wave & 1) + mfma_col(v, r);
            S0[row][col] = aD[v] - accD[v];
            if (has_row) S1[row][col] = aR[v] - accR[v];
        }
        __syncthreads();
        if (role == 0) {
#pragma unroll
            for (int q = 0; q < CB / VN; ++q) {
                const VT t4 = reinterpret_cast<const VT*>(&S0[r][0])[q];
#pragma unroll
                for (int e = 0; e < VN; ++e) z[VN * q + e] = vget(t4, e);
            }
        } else if (role == 1) {
#pragma unroll
            for (int q = 0; q < CB / VN; ++q) {
                const VT t4 = has_row ? reinterpret_cast<const VT*>(&S1[r][0])[q] : VT{};
#pragma unroll
                for (int e = 0; e < VN; ++e) z[VN * q + e] = has_row ? vget(t4, e) : (VN * q + e == r ? TV(1) : TV(0));
            }
        }
    } else if (role == 0) {
#pragma unroll
        for (int c = 0; c < CB; ++c) z[c] = M[c0 + r + (c0 + c) * lda];
    } else if (role == 1) {
#pragma unroll
        for (int c = 0; c < CB; ++c) z[c] = has_row ? M[i0 + r + (c0 + c) * lda] : (c == r ? TV(1) : TV(0));
    }
    TV* out = nullptr;
    int64_t out_ld = 0;
    if (role == 1) {
        out = has_row ? M + i0 + c0 * lda : Xinv + (int64_t)k * CB * CB;
        out_ld = has_row ? lda : CB;
    }
    bool bad_any = false;
    __syncthreads();  // every wave holds its rows: S0 now carries the published L columns
    TV (*Lt)[kTSB] = reinterpret_cast<TV (*)[kTSB]>(&S0[0][0]);
    TV inv = TV(1);
    // the diagonal wave runs one sub-block ahead of the block-row wave
    if (role == 0) { diag_chain<TV, 0>(z, r, bad_any, inv); diag_publish<TV, 0>(z, r, inv, Lt, invp); }
    __syncthreads();
    if (role == 0) {
        diag_trail_mfma<0>(z);
        diag_chain<TV, 1>(z, r, bad_any, inv);
        diag_publish<TV, 1>(z, r, inv, Lt, invp);
    } else if (role == 1) {
        row_solve<TV, 0>(z, Lt, invp, r, out, out_ld);
        row_trail_mfma<0>(z, Lt, r);
    }
    __syncthreads();
    if (role == 0) {
        diag_trail_mfma<1>(z);
        diag_chain<TV, 2>(z, r, bad_any, inv);
        diag_publish<TV, 2>(z, r, inv, Lt, invp);
    } else if (role == 1) {
        row_solve<TV, 1>(z, Lt, invp, r, out, out_ld);
        row_trail_mfma<1>(z, Lt, r);
    }
    __syncthreads();
    if (role == 0) {
        diag_trail_mfma<2>(z);
        diag_chain<TV, 3>(z, r, bad_any, inv);
        diag_publish<TV, 3>(z, r, inv, Lt, invp);
    } else if (role == 1) {
        row_solve<TV, 2>(z, Lt, invp, r, out, out_ld);
        row_trail_mfma<2>(z, Lt, r);
    }
    __syncthreads();
    if (role == 1) row_solve<TV, 3>(z, Lt, invp, r, out, out_ld);
    if (role == 0 && bad_any && w == 0) fail[0] = 1;
    }
}

// y = row np of the layout (L^-1 rhs after the factorization).
template <class TV>
__global__ void k_chol_gety(int np, int64_t lda, const TV* __restrict__ M, TV* __restrict__ y) {
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c < np) y[c] = M[np + (int64_t)c * lda];
}

// Backward substitution over the group of blocks b0 .. b0 + 3 (those below T),
// with Xinv_b = L_bb^-T (column-major). Wave w owns block b0 + w. Every
// workgroup solves the group: from the top block down, x_i = Xinv_i y_i, then
// y_w -= L_{i,w}^T x_i for the group's blocks w < i. Workgroup b0 stores the
// group's x; workgroup a < b0 updates y_a -= sum_i L_{b0+i,a}^T x_i. Four
// blocks per launch cut the number of dependent launches by four.
constexpr int kBsGroup = 4;

template <class TV>
__global__ void __launch_bounds__(256) k_chol_bsolve(int b0, int T, int64_t lda, const TV* __restrict__ M,
                                                     const TV* __restrict__ Xinv, TV* __restrict__ y, TV* __restrict__ x) {
    __shared__ TV ys[kBsGroup][CB];
    __shared__ TV xs[kBsGroup][CB];
    __shared__ TV part[kBsGroup][CB];
    const int t = threadIdx.x, w = t / CB, r = t % CB;
    const int a = blockIdx.x;
    const int G = min(kBsGroup, T - b0);
    const int64_t bw = (int64_t)b0 + w;
    const bool valid = w < G;
    TV X[CB];  // X[c] = Xinv_bw(r, c)
    if (valid) {
        const TV* Xb = Xinv + bw * CB * CB;
#pragma unroll
        for (int c = 0; c < CB; ++c) X[c] = Xb[c * CB + r];
        ys[w][r] = y[bw * CB + r];
    }
    __syncthreads();
    for (int i = G - 1; i >= 0; --i) {
        TV Lv[CB];  // Lv[l] = L(64 (b0 + i) + l, 64 (b0 + w) + r)
        if (w < i) {
            const TV* Lc = M + ((int64_t)b0 + i) * CB + (bw * CB + r) * lda;
#pragma unroll
            for (int l = 0; l < CB; ++l) Lv[l] = Lc[l];
        }
        if (w == i) {
            TV s = 0;
#pragma unroll
            for (int c = 0; c < CB; ++c) s += X[c] * ys[i][c];
            xs[i][r] = s;
        }
        __syncthreads();
        if (w < i) {
            TV s = 0;
#pragma unroll
            for (int l = 0; l < CB; ++l) s += Lv[l] * xs[i][l];
            ys[w][r] -= s;
        }
        __syncthreads();
    }
    if (a == b0) {
        if (valid) x[bw * CB + r] = xs[w][r];
        return;
    }
    TV s = 0;
    if (valid) {
        const TV* Lc = M + bw * CB + ((int64_t)a * CB + r) * lda;
        TV U[CB];
#pragma unroll
        for (int l = 0; l < CB; ++l) U[l] = Lc[l];
#pragma unroll
        for (int l = 0; l < CB; ++l) s += U[l] * xs[w][l];
    }
    part[w][r] = s;
    __syncthreads();
    if (w == 0) y[(int64_t)a * CB + r] -= (part[0][r] + part[1][r]) + (part[2][r] + part[3][r]);
}

__global__ void k_clear_flag(int* f) {
    if (threadIdx.x == 0) f[0] = 0;
}

}  // namespace

template <class TV, class TH>
void launch_chol_assemble(hipStream_t s, int nJ, const int* J, const TH* H, int K, const double* nrm,
                          const double* om, const double* E, const double* rhs, TV* M) {
    const int np = chol_padded(nJ);
    const int64_t lda = chol_lda(nJ);
    const int64_t total = lda * np;
    hipLaunchKernelGGL((k_chol_assemble<TV, TH>), dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s, nJ, np, lda, J, H,
                       K, nrm, om, E, rhs, M);
}

template <class TV>
void launch_chol_solve(hipStream_t s, int n, TV* M, TV* work, TV* x, int* fail) {
    const int np = chol_padded(n);
    const int64_t lda = chol_lda(n);
    const int T = np / CB;
    TV* y = work;
    TV* Xinv = work + np;
    for (int k = 0; k < T; ++k) {
        const TrailPart p = trail_part<false>(k, T);
        hipLaunchKernelGGL((k_chol_step<TV, false>), dim3(T - k + 1 + p.ndue + p.nlazy), dim3(256), 0, s, k, T, lda, M, Xinv, fail);
    }
    hipLaunchKernelGGL(k_chol_gety<TV>, dim3((np + 255) / 256), dim3(256), 0, s, np, lda, (const TV*)M, y);
    for (int b0 = kBsGroup * ((T - 1) / kBsGroup); b0 >= 0; b0 -= kBsGroup)
        hipLaunchKernelGGL(k_chol_bsolve<TV>, dim3(b0 + 1), dim3(256), 0, s, b0, T, lda, (const TV*)M, (const TV*)Xinv, y,
                           x);
}

// Gs = Y Y^T (both triangles, zero past n) from the factor's rows [np, 2 np): block
// (i, j), i >= j, is the sum over the block columns k >= i, one workgroup each. The
// blocks of small i have the longest sums and come first. At 6,339 rows in FP32 the
// factorization takes 3.4 ms and this product 1.0 (85 TFLOP/s), where the library's
// factorization and inversion took 30.
template <class TV, class TS>
__global__ void __launch_bounds__(256, sizeof(TV) == 8 ? 2 : 4) k_chol_inverse_product(int n, int T, int64_t lda,
                                                                                       const TV* __restrict__ M,
                                                                                       TS* __restrict__ Gs) {
    __shared__ __align__(16) TV S0[CB][kTS];
    __shared__ __align__(16) TV S1[CB][kTS];
    int ib = 0, jb = blockIdx.x;
    // row of the packed lower triangle: ib (ib + 1) / 2 <= blockIdx.x
    ib = (int)((sqrt(8.0 * jb + 1.0) - 1.0) * 0.5);
    while ((int64_t)ib * (ib + 1) / 2 > jb) --ib;
    while ((int64_t)(ib + 1) * (ib + 2) / 2 <= jb) ++ib;
    jb -= (int)((int64_t)ib * (ib + 1) / 2);
    const int t = threadIdx.x;
    const int64_t yi = (int64_t)(T + ib) * CB, yj = (int64_t)(T + jb) * CB;
    if constexpr (std::is_same<TV, float>::value) {
        const int lane = t % 64, wave = t / 64;
        float val[16];
#pragma unroll
        for (int v = 0; v < 16; ++v) val[v] = 0.f;
#pragma unroll 1
        for (int kp = ib; kp < T; ++kp) {
            stage_block<TV>(M, lda, yi, (int64_t)kp * CB, S0);
            stage_block<TV>(M, lda, yj, (int64_t)kp * CB, S1);
            __syncthreads();
            const f32x16 acc = tile_product_mfma(S0, S1, wave, lane);
#pragma unroll
            for (int v = 0; v < 16; ++v) val[v] += acc[v];
            __syncthreads();
        }
#pragma unroll
        for (int v = 0; v < 16; ++v) S0[32 * (wave >> 1) + (lane & 31)][32 * (wave & 1) + mfma_col(v, lane)] = val[v];
    } else {
        const int tx = t % 16, ty = t / 16;
        TV val[4][4], acc[4][4];
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int v = 0; v < 4; ++v) val[u][v] = TV(0);
#pragma unroll 1
        for (int kp = ib; kp < T; ++kp) {
            stage_block<TV>(M, lda, yi, (int64_t)kp * CB, S0);
            stage_block<TV>(M, lda, yj, (int64_t)kp * CB, S1);
            __syncthreads();
            tile_product(S0, S1, tx, ty, acc);
#pragma unroll
            for (int u = 0; u < 4; ++u)
#pragma unroll
                for (int v = 0; v < 4; ++v) val[u][v] += acc[u][v];
            __syncthreads();
        }
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int v = 0; v < 4; ++v) S0[4 * tx + u][4 * ty + v] = val[u][v];
    }
    __syncthreads();
    const int64_t ld = (int64_t)T * CB;
    const int r = t % CB;
    for (int c = t / CB; c < CB; c += 256 / CB) {
        const int64_t ri = (int64_t)ib * CB, rj = (int64_t)jb * CB;
        Gs[ri + r + (rj + c) * ld] = ri + r < n && rj + c < n ? (TS)S0[r][c] : TS(0);
        if (ib != jb) Gs[rj + r + (ri + c) * ld] = rj + r < n && ri + c < n ? (TS)S0[c][r] : TS(0);
    }
}

template <class TV, class TS>
void launch_chol_inverse(hipStream_t s, int n, TV* M, TS* Gs, int* fail) {
    const int T = chol_padded(n) / CB;
    const int64_t lda = chol_inv_lda(n);
    for (int k = 0; k < T; ++k) {
        const TrailPart p = trail_part<true>(k, T);
        hipLaunchKernelGGL((k_chol_step<TV, true>), dim3(T + p.ndue + p.nlazy), dim3(256), 0, s, k, T, lda, M, (TV*)nullptr,
                           fail);
    }
    hipLaunchKernelGGL((k_chol_inverse_product<TV, TS>), dim3(T * (T + 1) / 2), dim3(256), 0, s, n, T, lda, M, Gs);
}
template void launch_chol_inverse<float, float>(hipStream_t, int, float*, float*, int*);
template void launch_chol_inverse<double, float>(hipStream_t, int, double*, float*, int*);
template void launch_chol_inverse<double, double>(hipStream_t, int, double*, double*, int*);

// M_ab = (d_a . d_b) H[cidx_a][cidx_b] in the layout of launch_chol_inverse
template <class TV>
__global__ void __launch_bounds__(256) k_gram_assemble(int nb, int np, int64_t lda, const int* __restrict__ cidx,
                                                       const double* __restrict__ dirs, const double* __restrict__ H, int K,
                                                       TV* __restrict__ M) {
    const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (idx >= lda * np) return;
    const int r = (int)(idx % lda), c = (int)(idx / lda);
    double v;
    if (r < c) {
        v = 0.0;
    } else if (r >= np) {
        v = r - np == c ? 1.0 : 0.0;
    } else if (r >= nb) {
        v = r == c ? 1.0 : 0.0;
    } else {
        const double dd = dirs[3 * c] * dirs[3 * r] + dirs[3 * c + 1] * dirs[3 * r + 1] + dirs[3 * c + 2] * dirs[3 * r + 2];
        v = dd * H[(int64_t)cidx[c] * K + cidx[r]];
    }
    M[idx] = (TV)v;
}

template <class TV>
void launch_gram_assemble(hipStream_t s, int nb, const int* cidx, const double* dirs, const double* H, int K, TV* M) {
    const int np = chol_padded(nb);
    const int64_t lda = chol_inv_lda(nb), total = lda * np;
    hipLaunchKernelGGL(k_gram_assemble<TV>, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s, nb, np, lda, cidx, dirs, H,
                       K, M);
}
template void launch_gram_assemble<float>(hipStream_t, int, const int*, const double*, const double*, int, float*);
template void launch_gram_assemble<double>(hipStream_t, int, const int*, const double*, const double*, int, double*);

void launch_clear_flag(hipStream_t s, int* flag) { hipLaunchKernelGGL(k_clear_flag, dim3(1), dim3(64), 0, s, flag); }

template void launch_chol_assemble<float, double>(hipStream_t, int, const int*, const double*, int, const double*,
                                                  const double*, const double*, const double*, float*);
template void launch_chol_assemble<float, float>(hipStream_t, int, const int*, const float*, int, const double*,
                                                 const double*, const double*, const double*, float*);
template void launch_chol_assemble<double, double>(hipStream_t, int, const int*, const double*, int, const double*,
                                                   const double*, const double*, const double*, double*);
template void launch_chol_solve<float>(hipStream_t, int, float*, float*, float*, int*);
template void launch_chol_solve<double>(hipStream_t, int, double*, double*, double*, int*);

}  // namespace phd
