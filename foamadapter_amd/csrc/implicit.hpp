// implicit.hpp -- sparsity pattern and linear system handles.
#pragma once

#include "mesh.hpp"

#include <memory>

// The rows of other tiles that the persistent solvers' tiles of a pattern refer to, and the
// columns that refer to them (cgpersist.hpp).
struct fv_ghost_plan {
    fvhip::DBuf<uint32_t> words;
    fvhip::DBuf<int32_t> ghosts, count;
    int stride = -1;  // ghosts of a tile at most (-1: not counted yet)
};

// la::SparsityPattern (expression.hpp:35; test_sparsityPattern.cpp:36-62):
// CSR of the face graph, columns ascending per row; row c is
// [lower neighbours | c | upper neighbours] in the cell's stencil order.
struct fv_sparsity {
    fv_mesh* mesh = nullptr;
    int32_t nRows = 0;
    int64_t nnz = 0;
    fvhip::DBuf<int32_t> rowOffs, colIdxs, diagOffset, ownerOffset, neighbourOffset;
    // per stencil entry k (cell->face stencil of the mesh): CSR slot of the entry's
    // coefficient in the cell's row (-1 for boundary entries)
    fvhip::DBuf<int32_t> entrySlot;
    // sliced-ELL copy of the off-diagonal structure for the solvers' SpMVs,
    // whose scaled matrices have a unit diagonal (slices of 64 rows, one
    // wavefront each; entry k of row 64s+l at sellOff[s] + 64k + l): column and
    // source CSR index (-1 for padding)
    static constexpr int kSlice = 64;
    int64_t sellTotal = 0;
    fvhip::DBuf<int64_t> sellOff;
    fvhip::DBuf<int32_t> sellCol, sellSrc;
    // The persistent solvers read slices of one width, 4 or 6 (sellWidth; 0: a row has more
    // off-diagonal entries, or there are more rows than they take), without their offsets:
    // entry k of row i at (i / 64) * 64 w + 64 k + i % 64.  Where that makes the slices no
    // more than 5 % larger (hexahedra: those at the mesh's sides), all slices have that
    // width.  Else (triangles 3 of 4, prisms 5 of 6) they are as wide as their longest row,
    // for the solvers that stream them, and the first persistent solver makes these
    // (uniform_sell).
    static constexpr int64_t kUniformRows = 1 << 21;
    int32_t sellWidth = 0;
    bool sellUniform = false;
    fvhip::DBuf<int64_t> uniOff;
    fvhip::DBuf<int32_t> uniCol;
    int64_t uniTotal() const { return ((int64_t)nRows + kSlice - 1) / kSlice * kSlice * sellWidth; }
    fv_ghost_plan ghostPlan[2];  // for FP64, FP32: made by the first solver that uses it
};

// Solver workspace kept with a linear system between solves (one per precision).
struct fv_solver_cache {
    virtual ~fv_solver_cache() = default;
};

// Launches of a system's persistent solver, and the mishap the next ones are to have
// (fv_linsys_persist_fault).
struct fv_persist_log {
    int64_t launches = 0, apart = 0, refused = 0, lost = 0;
    int fault = 0, after = 0, exchange = 0;
    // the fault of the launch at hand
    int take() {
        if (!fault || after-- > 0) return 0;
        const int f = fault;
        fault = 0;
        return f;
    }
};

// la::LinearSystem<scalar, localIdx>: values[nnz], rhs[N] (FP64), with the
// convention A.x - b = (operator applied to x) * V.
struct fv_linsys {
    fv_sparsity* sp = nullptr;
    fvhip::DBuf<double> values, rhs;
    // boundary coefficients of the assembled laplacian terms, per boundary face:
    // the face flux is bRhs - bMat * x_P (NeoN's la::BoundaryCoefficients,
    // read by updateFaceVelocity, pressureVelocityCoupling.cpp:180-192)
    fvhip::DBuf<double> bMat, bRhs;
    fv_persist_log persistLog[3];
    std::unique_ptr<fv_solver_cache> cg[3];  // FP64 CG, FP32 CG in FP64 refinement, BiCGStab
};

namespace fvhip {
// Makes what the systems of a pattern share for fv_solve_cg in a mode (FV_SOLVE_*), for
// owners that keep patterns and account for their memory; the bytes a system's solver needs
// beside its vectors and its scaled matrix.
void cg_prepare(fv_sparsity* sp, int mode);
// The slices of width sellWidth (> 0), made on first use unless the others are such.
void uniform_sell(fv_sparsity* sp);
size_t cg_extra_bytes();
}  // namespace fvhip

#ifdef __HIPCC__
namespace fvhip {

// CSR rows by blocks of 256 rows and 256 threads: the block's entries are one
// contiguous range, read with consecutive lanes on consecutive entries (a thread
// that walks its own row reads every 56 bytes, and a wave's loads of one entry
// touch 28 lines), and handed to the rows through LDS.  kCsrLds entries fit (8 per
// row); a block with more walks its rows.  150x140x130 cells, FP64: A x - b 166 ->
// 63 us (305 MB: 4.9 TB/s), rAU and HbyA 225 -> 117.
constexpr int kCsrBlock = 256;
constexpr int kCsrU = 8;  // entries per thread
constexpr int kCsrLds = kCsrU * kCsrBlock;

// prod[k - ro[i0]] = va[k] * x[ci[k]] for the entries of rows [i0, i1); false (and
// nothing done) if they do not fit.  The caller's barrier comes before the rows read.
__device__ __forceinline__ bool csr_products(const int32_t* __restrict__ ro,
                                             const int32_t* __restrict__ ci,
                                             const double* __restrict__ va,
                                             const double* __restrict__ x, int i0, int i1,
                                             double* prod) {
    const int b = ro[i0], n = ro[i1] - b;
    if (n > kCsrLds) return false;
    double v[kCsrU], xg[kCsrU];
    int c[kCsrU];
    const int t = (int)threadIdx.x;
    const int last = n - 1;  // every lane loads (n > 0: a row holds its diagonal)
#pragma unroll
    for (int u = 0; u < kCsrU; ++u) {
        const int k = b + min(t + u * kCsrBlock, last);
        v[u] = va[k];
        c[u] = ci[k];
    }
#pragma unroll
    for (int u = 0; u < kCsrU; ++u) xg[u] = x[c[u]];
#pragma unroll
    for (int u = 0; u < kCsrU; ++u)
        if (t + u * kCsrBlock < n) prod[t + u * kCsrBlock] = v[u] * xg[u];
    return true;
}

}  // namespace fvhip
#endif
