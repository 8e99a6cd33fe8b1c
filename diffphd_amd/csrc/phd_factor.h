// Host-side construction of the sparse-inverse factor S with S^T S = A^-1.
//
// The reference (deformable_projective_dynamics_forward_gpu.cpp:600-647 with
// RealSim SparseLDLT.cpp:226-431) builds S = D^-1/2 L^-1 P from a METIS-ordered
// LDL^T and stores it as an FP64 CSR of S^T. Here the ordering is a nested
// dissection by recursive coordinate bisection, the numeric factorization is a
// multifrontal FP64 Cholesky A = P^T L L^T P (so S = L^-1 P, identical to
// D^-1/2 L_unit^-1 P), and S is stored index-free: with the elimination tree
// postordered, row k of L^-1 is exactly the subtree of k, i.e. the contiguous
// column range [fd(k), k]. Value (k, j) lives at V[base[k] + j].
#pragma once
#include <cstdint>
#include <vector>

namespace phd {

struct Factor {
    int n = 0;
    std::vector<int> perm;    // perm[new] = old vertex
    std::vector<int> iperm;   // iperm[old] = new
    std::vector<int> parent;  // elimination tree (new indices), -1 for roots
    std::vector<int> fd;      // first descendant (postorder) of each node
    std::vector<int> depth;   // root depth 0
    // Cholesky factor L (new indices), CSC, diagonal first in each column.
    std::vector<int64_t> Lp;
    std::vector<int> Li;
    std::vector<double> Lx;
    // Index-free layout of S = L^-1 (rows = new indices).
    std::vector<int64_t> base;  // V[base[k] + j] = S(k, j) for fd[k] <= j <= k
    int64_t v_len = 0;          // padded length of V
    int64_t nnz = 0;            // sum of subtree sizes
    int max_depth = 0;
    double factor_seconds = 0, order_seconds = 0;

    // Builds the factor of the symmetric matrix given in full CSR (scalar,
    // n x n) with vertex coordinates X (3n) used by the bisection.
    void build(int n_, const std::vector<int>& Ap, const std::vector<int>& Ai, const std::vector<double>& Ax,
               const std::vector<double>& X, int threads);
};

// Work units of the two SpMVs over the S layout.
//  * rows (y = S w): units of (group of row_group consecutive rows, chunk of
//    chunk_w columns), see below.
//  * cols (x = S^T y): tile t = columns [64t, 64t+63]; its items are the rows
//    intersecting the tile (the tile's own rows then the ancestors of its last
//    column), split into units of at most `unit_items` rows.
struct SpmvPlan {
    // cols
    std::vector<int> items;         // concatenated per tile
    std::vector<int> cu_tile, cu_i0, cu_i1;  // unit -> tile, item range
    std::vector<int> tile_unit_ptr;          // units of tile t
    // The same items in shorter units, for the solves whose summation order is free
    // (the adjoint and bodies without a frictional boundary; the frictional forward
    // iteration amplifies round-off and keeps the order above): halved until they give
    // every CU 16 waves or have 64 rows, one batch. Empty where the units above are
    // that many or that short. A unit of 512 rows is walked by one wave while most of the
    // chip is idle: 66 us at 5,040 vertices in FP64 and 35 us at 9,261 in FP32, with units
    // of 64 rows 15 and 10 us; 56 and 52 us at 35,301 in FP32.
    std::vector<int> fu_tile, fu_i0, fu_i1, tile_fine_ptr;
    // S w by units of (group of row_group consecutive rows, chunk of chunk_w
    // columns): each unit stages w[chunk] once for all rows of the group that
    // cross it. Row k's partial for chunk c sits in slot rbase[k] + c - fd(k) / chunk_w.
    // Rows per group: 64 where that gives every CU eight units (w is staged once for
    // 64 rows); fewer on smaller factors, whose four waves a unit would each walk 16
    // rows in a row while most of the chip is idle (21 us at 242 vertices, 31 us at
    // 5,040 in FP64). A row's partial is the same wherever its unit ends.
    int row_group = 64;
    int chunk_w = 1024;
    std::vector<int> gu_group, gu_chunk, rbase;
    // min_fine_items, fine_units: the fewest rows of a shorter unit, and the units that are enough
    void build(const Factor& f, int unit_items, int group_chunk_w = 1024, int min_fine_items = 64, size_t fine_units = 4096);
};

void host_factor_check(int n, const std::vector<int>& Ap, const std::vector<int>& Ai, const std::vector<double>& Ax,
                       const std::vector<double>& X, double* out);

}  // namespace phd
