// Kernels (gfx950) of the explicit inverse of small systems: A^-1 = S^T S as a
// full matrix in vertex order, and its products.
//
// The two products with S are four dependent launches (chunk partials, their sums,
// column-tile partials, their sums). One product with the full inverse is one launch
// without a chain (4 us at 425 vertices in FP64, 14 us at 2,673 in FP32), at the price of
// n^2 values; Body::kDenseMaxVertices states up to which n that pays, with both sides.
#include <hip/hip_runtime.h>

#include "phd_kernels.h"

namespace phd {

namespace {

constexpr int WAVE = 64;

__device__ inline double wave_sum(double v) {
#pragma unroll
    for (int off = WAVE / 2; off > 0; off /= 2) v += __shfl_xor(v, off, WAVE);
    return v;
}

// Tile (a, b), a <= b, of A^-1: sum over the rows k of S that cross both column
// tiles, which are among tile b's rows (its own and the ancestors of its last
// column; items[i0 .. i1)). 64 x 64 outputs per workgroup, 4 x 4 per thread,
// 16 rows of S staged at a time. Runs once per body.
template <class TV>
__global__ void __launch_bounds__(256) k_dense_inverse(int n, int ld, const int* __restrict__ items,
                                                       const int* __restrict__ item_ptr, const int* __restrict__ fd,
                                                       const int64_t* __restrict__ base, const double* __restrict__ V,
                                                       const int* __restrict__ perm, TV* __restrict__ out) {
    constexpr int KB = 16;
    __shared__ double As[KB][64], Bs[KB][64];
    const int ta = blockIdx.x, tb = blockIdx.y;
    if (ta > tb) return;
    const int tx = threadIdx.x % 16, ty = threadIdx.x / 16;
    const int i0 = item_ptr[tb], i1 = item_ptr[tb + 1];
    double acc[4][4] = {};
    for (int r0 = i0; r0 < i1; r0 += KB) {
        for (int t = threadIdx.x; t < KB * 64; t += 256) {
            const int r = r0 + t / 64, c = t % 64;
            double va = 0, vb = 0;
            if (r < i1) {
                const int k = items[r], f = fd[k];
                const int ja = 64 * ta + c, jb = 64 * tb + c;
                if (ja >= f && ja <= k) va = V[base[k] + ja];
                if (jb >= f && jb <= k) vb = V[base[k] + jb];
            }
            As[t / 64][c] = va;
            Bs[t / 64][c] = vb;
        }
        __syncthreads();
#pragma unroll
        for (int r = 0; r < KB; ++r) {
            double x[4], y[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) { x[u] = As[r][tx + 16 * u]; y[u] = Bs[r][ty + 16 * u]; }
#pragma unroll
            for (int u = 0; u < 4; ++u)
#pragma unroll
                for (int v = 0; v < 4; ++v) acc[u][v] += x[u] * y[v];
        }
        __syncthreads();
    }
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int i = 64 * ta + tx + 16 * u, j = 64 * tb + ty + 16 * v;
            if (i >= n || j >= n) continue;
            const int64_t pi = perm[i], pj = perm[j];
            out[pi * ld + pj] = (TV)acc[u][v];
            out[pj * ld + pi] = (TV)acc[u][v];
        }
}

template <class TV>
__global__ void k_dense_columns(int n, int ld, int K, int ldk, const int* __restrict__ cand, const TV* __restrict__ inv,
                                TV* __restrict__ out) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (int64_t)n * ldk) return;
    const int v = (int)(t / ldk), c = (int)(t % ldk);
    out[t] = c < K ? inv[(int64_t)v * ld + cand[c]] : TV(0);
}

// out[3v + d] = add[3v + d] + sum_j M[v][j] x[3j + d] (M: n rows of ncol values,
// row stride ld, a multiple of 4 with zeros past ncol; x: 3 ncol values, FP64
// products and sums in both precisions; add may be out). Vertices of dmask (may be
// null) get dval (0 when dval is null). uC (may be null): the sum alone at the
// vertex's candidate. R rows per workgroup, whose four waves take every fourth
// 16-byte vector of each row and add up through LDS: the product is bound by the
// loads in flight, and one wave per four rows left the chip at 0.65 waves per SIMD
// (17 us for the 28.6 MB of 2,673 vertices in FP32, 1.7 TB/s; now 13.6 us, 2.1 TB/s).
template <class TV, int R>
__global__ void __launch_bounds__(256) k_dense_apply(int n, int ncol, int ld, const TV* __restrict__ M,
                                                     const double* __restrict__ x, const double* add,
                                                     const unsigned char* __restrict__ dmask,
                                                     const double* __restrict__ dval, const int* __restrict__ vcand,
                                                     double* __restrict__ uC, double* out) {
    constexpr int VN = 16 / sizeof(TV);
    __shared__ double part[4][3 * R];
    const int lane = threadIdx.x % WAVE, wave = threadIdx.x / WAVE;
    const int v0 = R * blockIdx.x;
    double s[R][3] = {};
#pragma unroll 2
    for (int j = VN * (int)threadIdx.x; j < ncol; j += VN * 256) {
        TV m[R][VN];
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int v = min(v0 + r, n - 1);
            __builtin_memcpy(m[r], __builtin_assume_aligned(M + (int64_t)v * ld + j, 16), 16);
        }
#pragma unroll
        for (int e = 0; e < VN; ++e) {
            // columns past ncol are zeros of M; x is not read there
            const bool in = j + e < ncol;
            const double x0 = in ? x[3 * (j + e)] : 0.0, x1 = in ? x[3 * (j + e) + 1] : 0.0, x2 = in ? x[3 * (j + e) + 2] : 0.0;
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const double a = (double)m[r][e];
                s[r][0] += a * x0;
                s[r][1] += a * x1;
                s[r][2] += a * x2;
            }
        }
    }
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            const double t = wave_sum(s[r][d]);
            if (lane == 0) part[wave][3 * r + d] = t;
        }
    __syncthreads();
    const int k = threadIdx.x, v = v0 + k / 3, d = k % 3;
    if (k >= 3 * R || v >= n) return;
    const double t = ((part[0][k] + part[1][k]) + part[2][k]) + part[3][k];
    const int i = 3 * v + d;
    if (uC) {
        const int c = vcand[v];
        if (c >= 0) uC[3 * c + d] = t;
    }
    out[i] = dmask && dmask[v] ? (dval ? dval[i] : 0.0) : (add ? add[i] + t : t);
}

}  // namespace

template <class TV>
void launch_dense_inverse(hipStream_t s, int n, int ld, const int* items, const int* item_ptr, const int* fd,
                          const int64_t* base, const double* V, const int* perm, TV* out) {
    const int T = (n + 63) / 64;
    hipLaunchKernelGGL(k_dense_inverse<TV>, dim3(T, T), dim3(256), 0, s, n, ld, items, item_ptr, fd, base, V, perm, out);
}
template void launch_dense_inverse<float>(hipStream_t, int, int, const int*, const int*, const int*, const int64_t*,
                                          const double*, const int*, float*);
template void launch_dense_inverse<double>(hipStream_t, int, int, const int*, const int*, const int*, const int64_t*,
                                           const double*, const int*, double*);

template <class TV>
void launch_dense_columns(hipStream_t s, int n, int ld, int K, int ldk, const int* cand, const TV* inv, TV* out) {
    const int64_t m = (int64_t)n * ldk;
    hipLaunchKernelGGL(k_dense_columns<TV>, dim3((unsigned)((m + 255) / 256)), dim3(256), 0, s, n, ld, K, ldk, cand, inv, out);
}
template void launch_dense_columns<float>(hipStream_t, int, int, int, int, const int*, const float*, float*);
template void launch_dense_columns<double>(hipStream_t, int, int, int, int, const int*, const double*, double*);

template <class TV>
void launch_dense_apply(hipStream_t s, int n, int ncol, int ld, const TV* M, const double* x, const double* add,
                        const unsigned char* dmask, const double* dval, const int* vcand, double* uC, double* out) {
    // four rows read x once between them; under 1,024 rows that would leave fewer
    // than one workgroup per CU
    if (n >= 1024)
        hipLaunchKernelGGL((k_dense_apply<TV, 4>), dim3((n + 3) / 4), dim3(256), 0, s, n, ncol, ld, M, x, add, dmask, dval,
                           vcand, uC, out);
    else
        hipLaunchKernelGGL((k_dense_apply<TV, 1>), dim3(n), dim3(256), 0, s, n, ncol, ld, M, x, add, dmask, dval, vcand, uC,
                           out);
}
template void launch_dense_apply<float>(hipStream_t, int, int, int, const float*, const double*, const double*,
                                        const unsigned char*, const double*, const int*, double*, double*);
template void launch_dense_apply<double>(hipStream_t, int, int, int, const double*, const double*, const double*,
                                         const unsigned char*, const double*, const int*, double*, double*);

}  // namespace phd
