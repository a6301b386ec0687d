// Launchers of the implicit-step kernels (afx_implicit.hip), FP64.
#pragma once
#include "afx_kernels.hpp"

namespace afx {

hipError_t launch_face_jacobian(hipStream_t s, CellsT<double> C, FacesT<double> F, const double* q, const double* gx,
                                const double* gy, GasT<double> g, int viscous, double* Jf);
// the Spalart-Allmaras model's 5x5 face blocks (q, gx, gy: 5 planes)
hipError_t launch_face_jacobian_sa(hipStream_t s, CellsT<double> C, FacesT<double> F, const double* q, const double* gx,
                                   const double* gy, GasT<double> g, double* Jf);
// the source row of the Spalart-Allmaras diagonal blocks (q null: none)
struct SaSource {
    const double* q;    // 5 planes
    const double* gx;   // unlimited cell gradients, 5 planes
    const double* gy;
    const double* wd;   // wall distance
    GasT<double> g;
};
// nv: block size, 4 or 5 (Spalart-Allmaras).  With E non-null also writes the
// ELL copy of the matrix for launch_lhs_apply: E 4 nv^2 nC off-diagonal blocks
// by slot, Ds nv^2 nC diagonal blocks, nbr 4 nC neighbour indices (-1: none),
// all slot/entry-major over the real cells
hipError_t launch_assemble_diag(hipStream_t s, int nv, CellsT<double> C, FacesT<double> F, const double* dt,
                                const double* Jf, SaSource src, double* D, double* Dinv, double* E, double* Ds,
                                int32_t* nbr, int* bad);
// y = LHS x from the ELL copy.  active: a device flag (nullable); the kernel
// does nothing while it reads 0
hipError_t launch_lhs_apply(hipStream_t s, int nv, int32_t nC, int32_t nT, const double* Ds, const double* E,
                            const int32_t* nbr, const double* x, double* y, const int* active = nullptr);
hipError_t launch_block_jacobi(hipStream_t s, int nv, int32_t nC, int32_t nT, const double* Dinv, const double* x,
                               double* z, const int* active = nullptr);
// Multicolour block DILU.  The colour order of the real cells: the colour of
// each, the cells listed colour by colour (cells[off[c] .. off[c+1]), off on
// the host) and pos, the inverse list (the position of each real cell).
struct ColourOrder {
    const uint8_t* colour;
    const int32_t* cells;
    const int32_t* pos;
    const int32_t* off;   // ncolours + 1, host
    int ncolours;
};
// The matrix by position p: E 4 nv^2 nC off-diagonal blocks by slot, nbr 4 nC
// neighbour codes (q + 1 for the neighbour at position q of an earlier colour,
// -(q + 1) of a later one, 0 none), Dti and D nv^2 nC diagonal blocks (Dt^-1
// of the preconditioner, and the matrix's own).  Vectors that the sweeps and
// the product work on are nv planes of nC by position.
struct ColourMatrix {
    double* E;
    int32_t* nbr;
    double* Dti;
    double* D;
};
hipError_t launch_dilu_setup(hipStream_t s, int nv, CellsT<double> C, FacesT<double> F, const ColourOrder& O,
                             const double* D, const double* Jf, double* Dti, const ColourMatrix& M, int* bad);
// y = M^-1 in; y = A x; both by position
hipError_t launch_dilu_apply(hipStream_t s, int nv, const ColourOrder& O, const ColourMatrix& M, const double* in,
                             double* y);
hipError_t launch_colour_apply(hipStream_t s, int nv, const ColourOrder& O, const ColourMatrix& M, const double* x,
                               double* y);
// how a kernel's blocks share the positions 0 .. off[colours]: each XCD takes
// per[c] tiles of 64 of colour c, per_xcd in all
struct Span {
    int32_t off[7];   // a cell has at most four neighbours: at most five colours
    int32_t per[6];
    int32_t per_xcd;
};
// out = b - w by position from b in cell order (w null: b); z in cell order
// from y by position, ghost rows from x; the end of a cycle (k_colour_update)
hipError_t launch_to_colour(hipStream_t s, int nv, int32_t nT, const ColourOrder& O, const double* b, const double* w,
                            double* out);
hipError_t launch_from_colour(hipStream_t s, int nv, int32_t nT, const ColourOrder& O, const double* y, const double* x,
                              double* z);
hipError_t launch_colour_update(hipStream_t s, int nv, int32_t nT, const ColourOrder& O, int first, double relax,
                                const double* z, double* x, double* dq, double* q, const int* converged);

// device-resident restarted GMRES state (m <= 32)
constexpr int kGsBlocks = 1024;                        // most blocks of a reduction
constexpr size_t kGsSums = 2 * 33 * (size_t)kGsBlocks;   // doubles of GmDev::sums
struct GmDev {
    double* hdr;    // [0] beta0, [1] beta of the cycle, [2] scale of the next basis vector
    int* flags;     // [0] Arnoldi active, [1] converged, [2] total iterations, [3] columns of the cycle (jend)
    int* seen;      // the flags where the host reads them, in pinned memory (nullable)
    double* sums;   // block sums of the two Gram-Schmidt passes (kGsSums)
    double* H;      // (m + 1) x m, row-major
    double *cs, *sn, *g, *y;
    double *h1, *h2;   // Gram-Schmidt coefficients of the two passes (m + 1 each)
    double tol;     // converged when |g_{j+1}| <= tol beta0
    int m, maxit;
};
// doubles of the basis V for vectors of nv rows of len positions (layout: basis_at)
inline size_t basis_doubles(size_t len, int nv, int m) { return (len + 63) / 64 * 64 * (size_t)nv * (size_t)(m + 1); }
// The parts of Arnoldi step j (afx_implicit.hip); all do nothing once the
// process is inactive; n is the vectors' length.
// With DILU: column cols of V from w, y = M^-1 of it; then w = A y and the
// first pass's block sums (their number in *nblk)
hipError_t launch_dilu_apply_next(hipStream_t s, int nv, const ColourOrder& O, const ColourMatrix& M, const GmDev& G,
                                  const double* w, double* V, int cols, double* y);
hipError_t launch_colour_apply_dots(hipStream_t s, int nv, const ColourOrder& O, const ColourMatrix& M,
                                    const GmDev& G, const double* x, double* y, const double* V, int cols, int* nblk);
// otherwise: the vector (also as v, which may be w), and the first pass after
// w = A M^-1 v
hipError_t launch_next_vector(hipStream_t s, const GmDev& G, const double* w, double* V, int cols, double* v,
                              int64_t n);
hipError_t launch_gs_dots(hipStream_t s, const GmDev& G, const double* V, int64_t n, int m, const double* w, int* nblk);
// both: the second pass and the Givens step (O: vectors of nv planes in the
// colour order, null: of n entries; show: the host reads the flags next)
hipError_t launch_gm_step(hipStream_t s, const GmDev& G, const ColourOrder* O, int nv, const double* V, int64_t n, int j,
                          bool show, double* w, int nblk1);
// y = M^-1 sum_{k < jend} y_k V_k, the end of a cycle
hipError_t launch_dilu_apply_sum(hipStream_t s, int nv, const ColourOrder& O, const ColourMatrix& M, const GmDev& G,
                                 double* V, double* y);
// a cycle's set-up from its start vector r
hipError_t launch_gm_begin(hipStream_t s, const GmDev& G, const double* r, int64_t n, int first);
hipError_t launch_gm_solve(hipStream_t s, const GmDev& G);
// x = sum_{k < jend} y_k V_k
hipError_t launch_lincomb(hipStream_t s, const GmDev& G, const double* V, double* x, int64_t n);
hipError_t launch_sub(hipStream_t s, const double* b, const double* w, double* r, int64_t n);
hipError_t launch_axpy(hipStream_t s, double a, const double* x, double* y, int64_t n);
// matrix-free operator of the RANS_MATRIX_FREE build (ransMatrix.h:138-178)
hipError_t launch_mf_base(hipStream_t s, CellsT<double> C, FacesT<double> F, const double* q, GasT<double> g,
                          int viscous, double* Fb);
hipError_t launch_mf_apply(hipStream_t s, CellsT<double> C, FacesT<double> F, const double* q, const double* dt,
                           const double* Fb, GasT<double> g, int viscous, const double* x, double* y,
                           const int* active = nullptr);

}  // namespace afx
