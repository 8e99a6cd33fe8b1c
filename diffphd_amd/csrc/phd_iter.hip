// Kernels (gfx950) of one PD / adjoint iteration between the local step and the
// global solve, and after it: the right-hand side with its residual, and the
// Anderson step with the convergence sums.
//
// An iteration of a small body is a chain of dependent launches, each bound by
// its latency (a few microseconds), so what counts is how many there are and
// how often the host waits. Three kernels take the place of about fifteen
// launches and two host round trips:
//  * k_iter_residual: gather of the element contributions, right-hand side,
//    residual of the global system, contact impulses, previous iterate, and the
//    permuted input of the S product;
//  * k_iter_push: the newest Anderson difference pair and its dot products;
//  * k_iter_combine: the regularized least squares on the device, the combined
//    iterate and the sums of the convergence test, which go to pinned host memory.
// Partial sums of a kernel are added by every block of the next one, in a fixed
// order, so no launch is spent on a final reduction and results do not depend
// on scheduling.
#include <hip/hip_runtime.h>

#include <cfloat>

#include "phd_kernels.h"

namespace phd {

namespace {

constexpr int WAVE = 64;
constexpr int NT = 256;

// the sum lies in lane 0
__device__ inline double wave_sum(double v) {
#pragma unroll
    for (int off = WAVE / 2; off > 0; off /= 2) v += __shfl_down(v, off, WAVE);
    return v;
}

// -----------------------------------------------------------------------------
// b = inv_h2m q~ + sum of the element contributions - c_dir (FWD), or rhs + the
// contributions; r = b - A x, plus the contact impulses F of the vertex. One thread
// per DOF: the three of a vertex read the same entries of A, and a body of 2,700
// vertices has 32 blocks in flight instead of 11. Each sum runs in the order of
// its list, as the frictional iteration amplifies round-off.
// -----------------------------------------------------------------------------
template <bool FWD, class TV>
__global__ void __launch_bounds__(NT) k_iter_residual(IterResidual a, TV* __restrict__ w, int ldw) {
    const int i = blockIdx.x * NT + threadIdx.x;
    if (i >= 3 * a.nv) return;
    const int v = i / 3, d = i - 3 * v;
    double s = 0;
    const int p1 = a.inc_ptr[v + 1];
#pragma unroll 8
    for (int p = a.inc_ptr[v]; p < p1; ++p) s += a.elem[3 * (int64_t)a.inc_idx[p] + d];
    double b;
    if (FWD) {
        s -= a.c_dir[i];
        a.pd_rhs[i] = s;
        b = a.inv_h2m * a.rhs[i] + s;
    } else {
        b = a.rhs[i] + s;
    }
    a.x_prev[i] = a.x[i];
    double r = 0.0;
    if (!a.dmask[v] && !(a.pmask && a.pmask[i])) {
        r = b;
        if (a.pmask) {
            // per-DOF Dirichlet: axis d of the matrix drops the couplings to the
            // DOFs fixed on axis d
            for (int j = 0; j < a.width; ++j) {
                const int c = 3 * a.Ai[(int64_t)j * a.nv + v] + d;
                if (!a.pmask[c]) r -= a.Ax[(int64_t)j * a.nv + v] * a.x[c];
            }
        } else {
#pragma unroll 9
            for (int j = 0; j < a.width; ++j)
                r -= a.Ax[(int64_t)j * a.nv + v] * a.x[3 * a.Ai[(int64_t)j * a.nv + v] + d];
        }
    }
    if (a.F) {
        const int c = a.vcand[v];
        if (c >= 0) r += a.F[3 * c + d];
    }
    w[a.ipos ? (int64_t)d * ldw + a.ipos[v] : i] = (TV)r;
}

// x <- 0 where it is not finite; block sums of x.x
__global__ void __launch_bounds__(NT) k_iter_norm(int n, double* __restrict__ x, double* __restrict__ part) {
    __shared__ double sh[NT / WAVE];
    double s = 0;
    for (int i = blockIdx.x * NT + threadIdx.x; i < n; i += gridDim.x * NT) {
        double t = x[i];
        if (!isfinite(t)) { t = 0.0; x[i] = t; }
        s += t * t;
    }
    s = wave_sum(s);
    if (threadIdx.x % WAVE == 0) sh[threadIdx.x / WAVE] = s;
    __syncthreads();
    if (threadIdx.x == 0) part[blockIdx.x] = ((sh[0] + sh[1]) + sh[2]) + sh[3];
}

// sum of `rows` (at most kIterRows) block partials by one wave, in a fixed order;
// every lane gets it
__device__ inline double sum_rows(const double* __restrict__ p, int rows) {
    const int lane = threadIdx.x % WAVE;
    double t[kIterRows / WAVE], s = 0;
#pragma unroll
    for (int u = 0; u < kIterRows / WAVE; ++u) t[u] = lane + u * WAVE < rows ? p[lane + u * WAVE] : 0.0;
#pragma unroll
    for (int u = 0; u < kIterRows / WAVE; ++u) s += t[u];
    return __shfl(wave_sum(s), 0, WAVE);
}

// With g = x - x_prev: the newest difference pair (x_prev - x_last, g - g_last)
// and the new last iterate, and block sums of dG_a . dG_new, dG_a . g (a < m) and
// g . g. norm_rows > 0: x is first scaled to the clip norm (x.x from k_iter_norm).
__global__ void __launch_bounds__(NT) k_iter_push(int n, AAHist h, double* __restrict__ x, const double* __restrict__ x_prev,
                                                  double clip, const double* __restrict__ norm_part, int norm_rows,
                                                  double* __restrict__ part) {
    __shared__ double sh[NT / WAVE][2 * kAAMax + 1];
    double scale = 1.0;
    if (norm_rows > 0) {
        const double nn = sqrt(sum_rows(norm_part, norm_rows));
        if (isfinite(nn) && nn > clip) scale = clip / nn;
    }
    double acc[2 * kAAMax + 1];
#pragma unroll
    for (int k = 0; k <= 2 * kAAMax; ++k) acc[k] = 0.0;
    for (int i = blockIdx.x * NT + threadIdx.x; i < n; i += gridDim.x * NT) {
        const double xp = x_prev[i];
        double xi = x[i];
        if (scale != 1.0) { xi *= scale; x[i] = xi; }
        const double g = xi - xp;
        if (h.push) {
            double dg = 0.0;
            if (h.m > 0) {
                h.dq[i] = xp - h.x_last[i];
                dg = g - h.g_last[i];
                h.dg[i] = dg;
            }
            h.x_last[i] = xp;
            h.g_last[i] = g;
#pragma unroll
            for (int a = 0; a < kAAMax; ++a)
                if (a < h.m) {
                    const double ga = a == h.m - 1 ? dg : h.G[a][i];
                    acc[a] += ga * dg;
                    acc[kAAMax + a] += ga * g;
                }
        }
        acc[2 * kAAMax] += g * g;
    }
    const int lane = threadIdx.x % WAVE, wid = threadIdx.x / WAVE;
#pragma unroll
    for (int k = 0; k <= 2 * kAAMax; ++k) {
        if (k < 2 * kAAMax && k % kAAMax >= h.m) continue;
        const double s = wave_sum(acc[k]);
        if (lane == 0) sh[wid][k] = s;
    }
    __syncthreads();
    const int k = threadIdx.x;
    if (k <= 2 * kAAMax && (k == 2 * kAAMax || k % kAAMax < h.m))
        part[k * kIterRows + blockIdx.x] = ((sh[0][k] + sh[1][k]) + sh[2][k]) + sh[3][k];
}

// Solves M x = x by LDL^T for the leading N x N block (N at compile time, so that
// everything stays in registers), without fused operations: the host's arithmetic.
template <int N>
__device__ __forceinline__ void small_ldlt(double (&M)[kAAMax][kAAMax], double (&x)[kAAMax]) {
#pragma clang fp contract(off)
    double d[N];
#pragma unroll
    for (int j = 0; j < N; ++j) {
        double djj = M[j][j];
#pragma unroll
        for (int k = 0; k < j; ++k) djj -= M[j][k] * M[j][k] * d[k];
        d[j] = djj;
#pragma unroll
        for (int i = j + 1; i < N; ++i) {
            double s = M[i][j];
#pragma unroll
            for (int k = 0; k < j; ++k) s -= M[i][k] * M[j][k] * d[k];
            M[i][j] = djj != 0 ? s / djj : 0;
        }
    }
#pragma unroll
    for (int i = 0; i < N; ++i)
#pragma unroll
        for (int k = 0; k < i; ++k) x[i] -= M[i][k] * x[k];
#pragma unroll
    for (int i = 0; i < N; ++i) x[i] = d[i] != 0 ? x[i] / d[i] : 0;
#pragma unroll
    for (int i = N - 1; i >= 0; --i)
#pragma unroll
        for (int k = i + 1; k < N; ++k) x[i] -= M[k][i] * x[k];
}

// gamma of (M + reg) gamma = rr into gam; returns |gamma|
template <int N>
__device__ __forceinline__ double aa_solve(const double (*M)[kAAMax], double* gam, int replay) {
#pragma clang fp contract(off)
    double R[kAAMax][kAAMax], rr[kAAMax], sq = 0;
#pragma unroll
    for (int a = 0; a < N; ++a) {
#pragma unroll
        for (int b = 0; b < N; ++b) R[a][b] = M[a][b];
        rr[a] = gam[a];
        sq += R[a][a];
    }
    const double reg = replay ? 1e-10 * fmax(sq / N, 1.0) : fmax(1e-6 * sq / N, 1e-12);
#pragma unroll
    for (int a = 0; a < N; ++a) R[a][a] += reg;
    small_ldlt<N>(R, rr);
    double g2 = 0;
#pragma unroll
    for (int a = 0; a < N; ++a) { gam[a] = rr[a]; g2 += rr[a] * rr[a]; }
    return sqrt(g2);
}

// Every block adds the partial sums of k_iter_push and solves the small least
// squares; then x <- x_prev + g - sum gamma_a (dQ_a + dG_a) with the Dirichlet
// values put back (FWD) or non-finite entries cleared. With |gamma| >= 10 (and
// h.restart) x stays and the host drops the history. out (pinned host memory):
// [0] 1 when x was combined, [1] g.g, then block sums (kIterRows each): FWD
// |x - x_prev|^2, |x_prev|^2, |pd_rhs - pd_prev|^2, |pd_prev|^2, else x.x.
template <bool FWD>
__global__ void __launch_bounds__(NT) k_iter_combine(int n, AAHist h, const double* __restrict__ part, int rows,
                                                     const double* __restrict__ gram_in, double* __restrict__ gram_out,
                                                     const double* __restrict__ x_prev, double* __restrict__ x,
                                                     const unsigned char* __restrict__ fix, const double* __restrict__ fixval,
                                                     const double* __restrict__ pd_rhs, double* __restrict__ pd_prev,
                                                     double* __restrict__ out) {
    __shared__ double sum[2 * kAAMax + 1];
    __shared__ double M[kAAMax][kAAMax], gam[kAAMax];
    __shared__ int use;
    __shared__ double sh[NT / WAVE][4];
    const int lane = threadIdx.x % WAVE, wid = threadIdx.x / WAVE;
    for (int k = wid; k <= 2 * kAAMax; k += NT / WAVE) {
        if (k < 2 * kAAMax && k % kAAMax >= h.m) continue;
        const double s = sum_rows(part + k * kIterRows, rows);
        if (lane == 0) sum[k] = s;
    }
    __syncthreads();
    const int m = h.m;
    if (threadIdx.x < kAAMax * kAAMax) {
        const int a = threadIdx.x / kAAMax, b = threadIdx.x % kAAMax;
        if (a < m && b < m) {
            const int nw = m - 1;
            M[a][b] = a == nw ? sum[b] : b == nw ? sum[a] : gram_in[h.slot[a] * kAASlots + h.slot[b]];
        }
        if (a == 0 && b < m) gam[b] = sum[kAAMax + b];
    }
    if (blockIdx.x == 0 && m > 0 && threadIdx.x < kAASlots * kAASlots) {
        // the Gram matrix by pool slot, with the newest difference's row and column
        const int a = threadIdx.x / kAASlots, b = threadIdx.x % kAASlots, nw = h.slot[m - 1];
        double t = gram_in[threadIdx.x];
        for (int c = 0; c < m; ++c) {
            if (a == nw && b == h.slot[c]) t = sum[c];
            if (b == nw && a == h.slot[c]) t = sum[c];
        }
        gram_out[threadIdx.x] = t;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        double gn = 0;
        switch (m) {
            case 1: gn = aa_solve<1>(M, gam, h.replay); break;
            case 2: gn = aa_solve<2>(M, gam, h.replay); break;
            case 3: gn = aa_solve<3>(M, gam, h.replay); break;
            case 4: gn = aa_solve<4>(M, gam, h.replay); break;
            case 5: gn = aa_solve<5>(M, gam, h.replay); break;
            case 6: gn = aa_solve<6>(M, gam, h.replay); break;
        }
        const int ok = m > 0 && (h.replay || !(gn >= 10.0));
        use = ok;
        if (blockIdx.x == 0) { out[0] = ok; out[1] = sum[2 * kAAMax]; }
    }
    __syncthreads();
    const bool ok = use != 0;
    double e0 = 0, e1 = 0, e2 = 0, e3 = 0;
    for (int i = blockIdx.x * NT + threadIdx.x; i < n; i += gridDim.x * NT) {
        const double xp = x_prev[i];
        double c = x[i];
        if (ok) {
            c = xp + (c - xp);
#pragma unroll
            for (int a = 0; a < kAAMax; ++a)
                if (a < m) c -= (h.Q[a][i] + h.G[a][i]) * gam[a];
            if (FWD) { if (fix && fix[i]) c = fixval[i]; }
            else if (!isfinite(c)) c = 0.0;
            x[i] = c;
        }
        if (FWD) {
            const double p = pd_rhs[i], pp = pd_prev[i];
            pd_prev[i] = p;
            e0 += (c - xp) * (c - xp);
            e1 += xp * xp;
            e2 += (p - pp) * (p - pp);
            e3 += pp * pp;
        } else {
            e0 += c * c;
        }
    }
    e0 = wave_sum(e0);
    if (FWD) { e1 = wave_sum(e1); e2 = wave_sum(e2); e3 = wave_sum(e3); }
    if (lane == 0) { sh[wid][0] = e0; sh[wid][1] = e1; sh[wid][2] = e2; sh[wid][3] = e3; }
    __syncthreads();
    if (threadIdx.x < (FWD ? 4 : 1)) {
        const int k = threadIdx.x;
        out[kIterHead + k * kIterRows + blockIdx.x] = ((sh[0][k] + sh[1][k]) + sh[2][k]) + sh[3][k];
    }
}

// -----------------------------------------------------------------------------
// The two loops of L-BFGS (h: pairs oldest first) in one workgroup each: every step
// needs the previous one's dot product, which as launches with a host round trip each
// took about 20 us; here it is a barrier. A thread owns its entries throughout.
// -----------------------------------------------------------------------------
constexpr int NL = 1024;

// sum over the workgroup of two values; sh alternates between two buffers, so one
// barrier per call is enough
__device__ inline void block_sum2(double& a, double& b, double (*sh)[2]) {
    a = wave_sum(a);
    b = wave_sum(b);
    if (threadIdx.x % WAVE == 0) { sh[threadIdx.x / WAVE][0] = a; sh[threadIdx.x / WAVE][1] = b; }
    __syncthreads();
    a = b = 0;
#pragma unroll
    for (int w = 0; w < NL / WAVE; ++w) { a += sh[w][0]; b += sh[w][1]; }
}

// q = g, then from the newest pair to the oldest alpha_k = rho_k s_k . q and
// q -= alpha_k y_k; coef: alpha, then rho (kLbfgsMax each)
__global__ void __launch_bounds__(NL) k_lbfgs_first(int n, LbfgsHist h, const double* __restrict__ g, double* __restrict__ q,
                                                    double* __restrict__ coef) {
    __shared__ double sh[2][NL / WAVE][2];
    for (int k = h.m - 1; k >= 0; --k) {
        const double *s = h.S[k], *y = h.Y[k];
        double ys = 0, sq = 0;
        for (int i = threadIdx.x; i < n; i += NL) {
            ys += y[i] * s[i];
            sq += s[i] * (k == h.m - 1 ? g[i] : q[i]);
        }
        block_sum2(ys, sq, sh[k & 1]);
        const double rho = 1 / ys, alpha = rho * sq;
        for (int i = threadIdx.x; i < n; i += NL) q[i] = (k == h.m - 1 ? g[i] : q[i]) - alpha * y[i];
        if (threadIdx.x == 0) { coef[k] = alpha; coef[kLbfgsMax + k] = rho; }
    }
}

// from the oldest pair to the newest: d += (alpha_k - rho_k y_k . d) s_k
__global__ void __launch_bounds__(NL) k_lbfgs_second(int n, LbfgsHist h, const double* __restrict__ coef,
                                                     double* __restrict__ d) {
    __shared__ double sh[2][NL / WAVE][2];
    for (int k = 0; k < h.m; ++k) {
        const double *s = h.S[k], *y = h.Y[k];
        double yd = 0, unused = 0;
        for (int i = threadIdx.x; i < n; i += NL) yd += y[i] * d[i];
        block_sum2(yd, unused, sh[k & 1]);
        const double c = coef[k] - coef[kLbfgsMax + k] * yd;
        for (int i = threadIdx.x; i < n; i += NL) d[i] += c * s[i];
    }
}

}  // namespace

int iter_rows(int n) { return std::max(1, std::min(kIterRows, (n + NT - 1) / NT)); }

template <class TV>
void launch_iter_residual(hipStream_t s, const IterResidual& a, bool fwd, TV* w, int ldw) {
    const dim3 grid((unsigned)((3 * (int64_t)a.nv + NT - 1) / NT)), block(NT);
    if (fwd) hipLaunchKernelGGL((k_iter_residual<true, TV>), grid, block, 0, s, a, w, ldw);
    else hipLaunchKernelGGL((k_iter_residual<false, TV>), grid, block, 0, s, a, w, ldw);
}
template void launch_iter_residual<float>(hipStream_t, const IterResidual&, bool, float*, int);
template void launch_iter_residual<double>(hipStream_t, const IterResidual&, bool, double*, int);

void launch_lbfgs_first(hipStream_t s, int n, const LbfgsHist& h, const double* g, double* q, double* coef) {
    hipLaunchKernelGGL(k_lbfgs_first, dim3(1), dim3(NL), 0, s, n, h, g, q, coef);
}
void launch_lbfgs_second(hipStream_t s, int n, const LbfgsHist& h, const double* coef, double* d) {
    hipLaunchKernelGGL(k_lbfgs_second, dim3(1), dim3(NL), 0, s, n, h, coef, d);
}

void launch_iter_norm(hipStream_t s, int n, double* x, double* part) {
    hipLaunchKernelGGL(k_iter_norm, dim3(iter_rows(n)), dim3(NT), 0, s, n, x, part);
}

void launch_iter_push(hipStream_t s, int n, const AAHist& h, double* x, const double* x_prev, double clip,
                      const double* norm_part, double* part) {
    hipLaunchKernelGGL(k_iter_push, dim3(iter_rows(n)), dim3(NT), 0, s, n, h, x, x_prev, clip, norm_part,
                       norm_part ? iter_rows(n) : 0, part);
}

void launch_iter_combine(hipStream_t s, int n, bool fwd, const AAHist& h, const double* part, const double* gram_in,
                         double* gram_out, const double* x_prev, double* x, const unsigned char* fix, const double* fixval,
                         const double* pd_rhs, double* pd_prev, double* out) {
    const dim3 grid(iter_rows(n)), block(NT);
    if (fwd)
        hipLaunchKernelGGL(k_iter_combine<true>, grid, block, 0, s, n, h, part, iter_rows(n), gram_in, gram_out, x_prev, x,
                           fix, fixval, pd_rhs, pd_prev, out);
    else
        hipLaunchKernelGGL(k_iter_combine<false>, grid, block, 0, s, n, h, part, iter_rows(n), gram_in, gram_out, x_prev, x,
                           fix, fixval, pd_rhs, pd_prev, out);
}

}  // namespace phd
