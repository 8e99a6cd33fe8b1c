// Launchers for the HIP kernels of the PD time step (phd_kernels.hip).
// All pointers are device pointers; every launcher enqueues on `stream`.
#pragma once
#include <hip/hip_runtime.h>
#include <cstdint>

namespace phd {

// Per-element material description of the merged PD energies.
struct DevMaterials {
    int ne = 0, edim = 8, samples = 8;
    const int* elems = nullptr;   // SoA: elems[k * ne + e]
    const double* G = nullptr;    // grad_undeformed_sample_weight rows (edim x 3, row-major) per sample
    int g_stride = 0;             // doubles per element (0: shared by all elements)
    const double* wc = nullptr;   // corotated weight * vol / samples (nullptr: none)
    const double* wv = nullptr;   // volume weight * vol / samples
    int n_nh = 0;
    const double* wn[4] = {nullptr, nullptr, nullptr, nullptr};
    double nh_mu[4] = {0, 0, 0, 0}, nh_la[4] = {0, 0, 0, 0}, nh_k[4] = {0, 0, 0, 0};
    // muscle fibers (PdMuscleEnergy), at most one per element: weight
    // stiffness * vol / samples (0: none), unit fiber direction (SoA, 3 ne) and
    // actuation level; mw == nullptr when the body has no muscles
    const double* mw = nullptr;
    const double* mfib = nullptr;
    const double* mact = nullptr;
};

struct DotArgs {
    int m = 0;
    const double* a[32];
    const double* b[32];
};

// Boundary (frictional obstacle) description for the contact kernels.
struct DevBoundary {
    int type = 0;                 // 1 planar, 2 spherical, 3 heightfield, 4 press, 5 mesh
    double n[3] = {0, 0, 1}, off = 0;
    double c[3] = {0, 0, 0}, r = 0;
    double z0 = 0, plane_z = 0;
    int nwaves = 0;
    const double* waves = nullptr;  // device (amp, kx, ky, phase) quadruples
    // mesh: two triangle sets of the body itself (left, then right: 3 vertex
    // indices each); a vertex below `split` queries the right set, any other
    // the left set, at the body's current positions
    int split = 0, nfl = 0, nfr = 0;
    const int* faces = nullptr;
    double radius = 0;
};

// Axis stride of the S-product input w (3 axes): 64-aligned with room for the
// 16-byte vector loads past the last column.
__host__ __device__ inline int spmv_ldw(int n) { return ((n + 64 + 63) / 64) * 64; }
// Tail padding (elements) of the factor arrays V64 / V32 for the same loads.
constexpr int kVPad = 64;

// ---- factor expansion and the S / S^T products --------------------------------
// chain[i] = 1 when parent(i) == i + 1 and pattern(i) = {i} + pattern(i + 1).
void launch_expand_s(hipStream_t s, int n, int t_begin, int t_end, const int64_t* Lp, const int* Li, const double* Lx,
                     const int* parent, const int* depth, const int* fd, const int64_t* base, const unsigned char* chain,
                     double* ws, int64_t ws_stride, double* V64, float* V32);

// S w by (row_group-row group, chunk_w-column chunk) units with w staged in LDS; the
// per-(row, chunk) partials are then summed per row (plan: SpmvPlan::gu_*, rbase,
// built for the same chunk_w, one of kSpmvChunks).
constexpr int kSpmvChunks[3] = {512, 1024, 2048};
template <class TV>
void launch_spmv_rows_grp(hipStream_t s, int nunits, int row_group, const int* gu_group, const int* gu_chunk, const int* fd,
                          const int64_t* base, const int* rbase, const TV* V, const TV* w, int n, TV* pslot, int chunk_w);
template <class TV>
void launch_spmv_rows_slots(hipStream_t s, int n, const int* rbase, const TV* pslot, TV* y);
template <class TV>
void launch_spmv_cols(hipStream_t s, int nunits, const int* cu_tile, const int* cu_i0, const int* cu_i1, const int* items,
                      const int* fd, const int64_t* base, const TV* V, const TV* y, int n, TV* xpart);
// out[3 perm[j] + d] = (add ? add[...] : 0) + sum of tile partials; vertices with dmask set keep dval.
// fine: the partials of the fine units, which are many per tile.
template <class TV>
void launch_spmv_cols_fin(hipStream_t s, int n, const int* tile_unit_ptr, const TV* xpart, const int* perm,
                          const double* add, const unsigned char* dmask, const double* dval, double* out, bool fine = false);
// w[d * n + j] = r[3 perm[j] + d] (SoA, postorder), zero at dmask vertices.
template <class TV>
void launch_perm_in(hipStream_t s, int n, const int* perm, const double* r, const unsigned char* dmask, TV* w);

// ---- local step, gather, residual --------------------------------------------
// fp32: the SVD and the projections in FP32 (F and the sums in FP64); samples: one
// thread per sample of a hex (another order of the sums)
void launch_local_step(hipStream_t s, const DevMaterials& m, const double* q, double* elem_out, int block, bool fp32,
                       bool samples);
// pd_rhs = sum of element contributions - c_dir; b = inv_h2m * q_tilde + pd_rhs
void launch_gather_rhs(hipStream_t s, int nv, const int* inc_ptr, const int* inc_idx, const double* elem_out,
                       const double* c_dir, const double* q_tilde, double inv_h2m, double* pd_rhs, double* b);
// Per-DOF Dirichlet (the bordered correction of a global solve on the shared
// factor; PdirAxes: axis d's fixed vertices are fv[off[d] .. off[d + 1]) and
// its G_d^-1 starts at ginv + goff[d]).
struct PdirAxes {
    int off[4];
    long long goff[3];
};
void launch_pdir_coef(hipStream_t s, int np, const PdirAxes& ax, const int* map, const int* fv, const double* ginv,
                      const double* y, const double* t, double* coef);
void launch_pdir_apply(hipStream_t s, int nv, int np, const double* Z, const double* coef, const unsigned char* pmask,
                       const double* o, double* y);
void launch_pdir_columns(hipStream_t s, int nv, int p0, int na, const double* x, double* Z);
void launch_pdir_gather(hipStream_t s, int np, int nv, const int* pv, const double* Z, double* out);
// r = b - A q for the three axes (AoS); A in ELL form (entry j of row v at
// j * nv + v, width entries per row); dmask: whole-vertex Dirichlet rows
// (r = 0); pmask (per DOF, may be null): DOFs fixed on their own (r = 0, and
// their couplings are left out on that axis)
void launch_residual(hipStream_t s, int nv, int width, const int* Ai, const double* Ax, const double* b, const double* q,
                     const unsigned char* dmask, double* r,
                     const unsigned char* pmask = nullptr);
void launch_gather_vertex(hipStream_t s, int nv, const int* inc_ptr, const int* inc_idx, const double* elem_out, double* out);

// ---- reductions and vector updates -------------------------------------------
void launch_dots(hipStream_t s, int n, const DotArgs& args, double* partial, double* out);
int dots_partial_size();
// out = x + alpha * (y - z) ... generic axpby: out = a*x + b*y (+ c*z)
void launch_axpbypcz(hipStream_t s, int n, double a, const double* x, double b, const double* y, double c,
                     const double* z, double* out);
void launch_set_dirichlet(hipStream_t s, int nd, const int* ddof, const double* dval, double* q);
void launch_zero_dirichlet(hipStream_t s, int nd, const int* ddof, double* q);
void launch_scale(hipStream_t s, int n, double a, double* x);

// ---- one iteration around the global solve (phd_iter.hip) ---------------------
constexpr int kAAMax = 6;       // Anderson differences combined at once (aa_window <= 6)
constexpr int kAASlots = 7;     // difference buffers of the pool
constexpr int kIterRows = 512;  // most block partials per sum
constexpr int kIterHead = 8;    // doubles before the block sums of launch_iter_combine's output
constexpr int kIterPartials = (2 * kAAMax + 1) * kIterRows;
constexpr int kIterOut = kIterHead + 4 * kIterRows;
int iter_rows(int n);  // block partials of a vector of n entries
// The Anderson history as the kernels see it: m differences (oldest first, the
// newest last: dq / dg, also Q[m - 1] / G[m - 1]), their pool slots, the last iterate.
struct AAHist {
    int m = 0, push = 0, replay = 0;
    int slot[kAAMax] = {};
    const double* Q[kAAMax] = {};
    const double* G[kAAMax] = {};
    double *dq = nullptr, *dg = nullptr, *x_last = nullptr, *g_last = nullptr;
};
// Right-hand side and residual of one iteration (see k_iter_residual); F and
// vcand (candidate of a vertex or -1) may be null, pmask as in launch_residual.
struct IterResidual {
    int nv = 0, width = 0;
    const int *inc_ptr = nullptr, *inc_idx = nullptr, *Ai = nullptr, *ipos = nullptr, *vcand = nullptr;
    const double *elem = nullptr, *c_dir = nullptr, *rhs = nullptr, *Ax = nullptr, *x = nullptr, *F = nullptr;
    const unsigned char *dmask = nullptr, *pmask = nullptr;
    double inv_h2m = 0;
    double *pd_rhs = nullptr, *x_prev = nullptr;
};
// fwd: rhs is q~ and pd_rhs, c_dir are used; else b = rhs + the contributions.
// w[d * ldw + ipos[v]] = the residual (the S product's input), or w[3 v + d] when
// ipos is null; x_prev = x.
template <class TV>
void launch_iter_residual(hipStream_t s, const IterResidual& a, bool fwd, TV* w, int ldw);
// x <- 0 where not finite; part[0 .. iter_rows(n)) = block sums of x.x
void launch_iter_norm(hipStream_t s, int n, double* x, double* part);
// norm_part (may be null): x is first scaled to |x| <= clip; part: kIterPartials doubles
void launch_iter_push(hipStream_t s, int n, const AAHist& h, double* x, const double* x_prev, double clip,
                      const double* norm_part, double* part);
// out: kIterOut doubles of pinned host memory; gram_in / gram_out (kAASlots^2
// doubles each, not the same array): the Gram matrix before and after this step
void launch_iter_combine(hipStream_t s, int n, bool fwd, const AAHist& h, const double* part, const double* gram_in,
                         double* gram_out, const double* x_prev, double* x, const unsigned char* fix, const double* fixval,
                         const double* pd_rhs, double* pd_prev, double* out);

// L-BFGS direction of the baseline in one workgroup per loop, for vectors of up to
// kLbfgsEntries and kLbfgsMax pairs (oldest first): beyond about 32,000 entries one
// CU's reads of the pairs cost what the launches and round trips of many blocks do.
// coef: 2 kLbfgsMax doubles carried from the first loop to the second.
constexpr int kLbfgsMax = 32;
constexpr int kLbfgsEntries = 32768;
struct LbfgsHist {
    int m = 0;
    const double* S[kLbfgsMax] = {};
    const double* Y[kLbfgsMax] = {};
};
void launch_lbfgs_first(hipStream_t s, int n, const LbfgsHist& h, const double* g, double* q, double* coef);
void launch_lbfgs_second(hipStream_t s, int n, const LbfgsHist& h, const double* coef, double* d);

// ---- explicit inverse of small systems (phd_small.hip) -------------------------
// out (n x ld, zero-filled by the caller past column n) = S^T S in vertex order;
// items[item_ptr[t] .. item_ptr[t + 1]): the rows of S that cross column tile t
template <class TV>
void launch_dense_inverse(hipStream_t s, int n, int ld, const int* items, const int* item_ptr, const int* fd,
                          const int64_t* base, const double* V, const int* perm, TV* out);
// out (n x ldk) = the candidate columns of inv (n x ld), zeros past column K
template <class TV>
void launch_dense_columns(hipStream_t s, int n, int ld, int K, int ldk, const int* cand, const TV* inv, TV* out);
// out = add + M x on the three axes (see k_dense_apply)
template <class TV>
void launch_dense_apply(hipStream_t s, int n, int ncol, int ld, const TV* M, const double* x, const double* add,
                        const unsigned char* dmask, const double* dval, const int* vcand, double* uC, double* out);

// ---- contact -----------------------------------------------------------------
// normals / tangents at the frame-start positions (GetLocalFrame)
// Mesh boundary (type 5): the frames are anchored at the closest point of the
// opposite triangle set at q (normal (p - closest) / |p - closest|, tangents by
// Gram-Schmidt from the axis least parallel to it), and enabled_out[c] marks
// the candidates within 5 contact radii of that set; the distance is the
// projection of p - closest on the frame-start normal refn minus the radius.
void launch_contact_frames(hipStream_t s, int K, const DevBoundary& b, const int* nodes, const double* q, double* nrm,
                           double* t1, double* t2, unsigned char* enabled_out = nullptr);
void launch_contact_distance(hipStream_t s, int K, const DevBoundary& b, const int* nodes, const double* q, double* delta,
                             const double* refn = nullptr);
// Lists (candidate paths, or rows crossed by paths) cut into pieces of at most
// kContactPiece entries: piece q covers entries [b[q], e[q]) and the pieces of
// list l are [ptr[l], ptr[l + 1]) (device arrays).
constexpr int kContactPiece = 1024;
struct ContactPieces {
    int nlists = 0, npieces = 0;
    const int* b = nullptr;
    const int* e = nullptr;
    const int* ptr = nullptr;
};
// u[c] = sum_p val[p] * y[d * n + row[p]] for the three axes: out[3c + d]
// (part: 3 doubles per piece of scratch)
template <class TV>
void launch_contact_gather(hipStream_t s, const ContactPieces& pc, const int* cp_row, const TV* cp_val, const TV* y, int n,
                           double* part, double* out);
// y[d * n + row] += sum over the row's contacts of val * f[3c + d]
template <class TV>
void launch_contact_scatter(hipStream_t s, const ContactPieces& pc, const int* rc_row, const int* rc_c, const TV* rc_val,
                            const double* f, double* part, int n, TV* y);

void launch_gather_vals(hipStream_t s, int64_t m, const int* rows, const int* cols, const int64_t* base,
                        const double* V64, double* o64, float* o32);
void launch_scatter_dense(hipStream_t s, int64_t m, const int* ridx, const int* cidx, const double* val, int K, double* D);
// mirrors the lower triangle (column-major, as written by rocblas_dsyrk) into the upper one
void launch_symmetrize_lower(hipStream_t s, int K, double* H);

void launch_gather_nodes(hipStream_t s, int K, const int* nodes, const double* q, double* out);
// ub[a] = dirs_a . u[cidx[a]] (3-vectors per candidate)
// ub[a] = d_a . (u + u2)_{c_a} (u2 may be null)
void launch_basis_project(hipStream_t s, int nb, const int* cidx, const double* dirs, const double* u, const double* u2,
                          double* ub);
// F[3c + d] = -sum over the basis rows a of candidate c (clist[cptr[c] .. cptr[c+1]), increasing a) of g[a] dirs_a[d]
void launch_basis_expand(hipStream_t s, int K, const int* cptr, const int* clist, const double* dirs, const double* g,
                         double* F);
// y = Gs x for the full symmetric Gs above.
template <class TV>
void launch_gemv_sym(hipStream_t s, int n, int64_t ld, const TV* Gs, const double* x, double* y);

// out[3a + d] = sum_b H[rows[a]][cols[b]] f[3 cols[b] + d]
// ---- NCP iteration on the device (forward_gpu.cpp:1149-1302) ----
// flag bits of a candidate: in J (omega != 0), carries an impulse (F != 0),
// carries an impulse of g (omega lambda != 0 or friction), in P (J or F);
// friction sets: lambda > 0, omega lambda != 0
constexpr int kNcpJ = 1, kNcpF = 2, kNcpG = 4, kNcpP = 8, kNcpL = 1, kNcpN = 2;
// enabled (may be null): candidates outside the set take no part (omega 0, no impulse)
void launch_ncp_sets(hipStream_t s, int K, const unsigned char* enabled, const double* delta, const double* lambda,
                     const double* rprec, const double* nrm, const double* t1, const double* t2, const double* qC, double* uC,
                     const double* F, const double* lt1, const double* lt2, int do_fric, double* om, double* E, double* hvec,
                     double* Fg, unsigned char* flags);
// lists (nl <= 4, K entries each) of the candidates whose flags contain masks[i];
// counts[i] their sizes; pos[c] = position of c in list 0 or -1
void launch_ncp_compact(hipStream_t s, int K, const unsigned char* flags, int nl, const int* masks, int* lists, int* counts,
                        int* pos);
void launch_ncp_rhs(hipStream_t s, int nP, const int* P, const double* hprev, const int* posJ, const double* hg,
                    const double* hvec, const double* om, const double* nrm, double* uC, double* rJ);
template <class TV>
void launch_ncp_lambda(hipStream_t s, int K, const int* posJ, const TV* x, const double* hvec, const double* E,
                       const double* om, double lam_max, double* lambda);
void launch_fric_sets(hipStream_t s, int K, const double* lambda, const double* om, const double* nrm, double* Fn,
                      unsigned char* flags);
void launch_fric_coulomb(hipStream_t s, int K, const double* lambda, const int* posL, const double* hn, const double* uC,
                         const double* qframe, const double* nrm, const double* t1, const double* t2, const double* Hdiag,
                         double fmu, double* lt1, double* lt2);
void launch_ncp_impulses(hipStream_t s, int K, const double* om, const double* lambda, const double* nrm, const double* lt1,
                         const double* lt2, const double* t1, const double* t2, int do_fric, double* F, double* dF);
// H_rows,cols f with both counts read on the device; grid for max_rows rows.
// TH: the stored precision of H (FP64, or its FP32 copy), sums in FP64.
template <class TH>
void launch_h_apply_idx_dev(hipStream_t s, int max_rows, const int* nr_dev, const int* rows, const int* nc_dev,
                            const int* cols, const TH* H, int K, const double* f, double* out);
template <class TH>
void launch_h_apply_idx(hipStream_t s, int nr, const int* rows, int nc, const int* cols, const TH* H, int K,
                        const double* f, double* out);
void launch_to_float(hipStream_t s, int64_t n, const double* a, float* b);

// streaming copy of n16 16-byte words (byte-counter calibration)
void launch_copy(hipStream_t s, int64_t n16, const void* a, void* b);

// ---- backward ----------------------------------------------------------------
// per-sample 9x9 proximal-map Jacobians weighted by the K_pd weights
template <class TW>
// filter != 0: each sample block's eigenvalues mu (relative to the sample's
// weight in A) above 1 move to 1 + theta (mu - 1), then up to lo; filter = 0
// keeps the reference's K_pd. nfilt (may be null) counts the samples whose
// block moved by more than 1e-9.
void launch_kpd_build(hipStream_t s, const DevMaterials& m, const double* kc, const double* kv, const double* const* kn,
                      const double* q, int filter, double theta, double lo, int* nfilt, TW* W);
template <class TW>
void launch_kpd_apply(hipStream_t s, const DevMaterials& m, const TW* W, const double* dq, double* elem_out);
// g[type][e]: z_e^T (-(vol/s) sum_s A_s^T vec(P_s / stiffness)) per merged energy type
void launch_dmatw(hipStream_t s, const DevMaterials& m, const double* q, const double* z, double vol_over_s, double* g_cor,
                  double* g_vol, double* g_nh);
// the baseline forward's per-element PD + muscle energy and element forces
void launch_pd_energy_force(hipStream_t s, const DevMaterials& m, const double* kc, const double* kv, const double* q,
                            double* energy, double* elem_out);
// x += Z[zcol[c]] mu[c] per axis over the nc frozen nodes; dst = src on the nodes
void launch_frozen_apply(hipStream_t s, int nv, int nc, const double* Z, const int* zcol, const double* mu, double* x);
void launch_copy_nodes(hipStream_t s, int nc, const int* nodes, const double* src, double* dst);
// G[i nc + j] = Z[zcol[j]][nodes[i]]
void launch_gather_z(hipStream_t s, int nc, int nv, const int* nodes, const int* zcol, const double* Z, double* G);
// per muscle element (m.mw != nullptr): g_da[e] = z^T df/da, g_dw[e] = z^T df/d(act_w) (0 elsewhere)
void launch_dact(hipStream_t s, const DevMaterials& m, const double* q, const double* z, double vol_over_s, double* g_da,
                 double* g_dw);

}  // namespace phd
