// Implicit pseudo-time step on the device (FP64): the finite-difference flux
// Jacobian of implicitSolver::fillRhoLHS (solver.h:979-1075,
// physics.h:533-578) in 4x4 blocks, its block-Jacobi and multicolour block
// DILU preconditioners, the operator product and the kernels of the
// device-resident restarted GMRES driven from afx_capi.hip (the Arnoldi
// coefficients, Givens rotations and convergence flags live in device
// memory; the host reads the flags between chunks of Arnoldi steps).
//
// Blocks are N x N with N = 4 (the reference's four variables) or N = 5 (the
// Spalart-Allmaras model, whose Jacobian is this build's own: the reference's
// SA branch is empty, physics.h:259-261).
//
// Layout: vectors are SoA [k*nT + i] over real and ghost cells (ghost rows of
// the reference's matrix are identity rows with zero right-hand side, so their
// unknowns stay zero and the ghost columns of boundary faces are dropped).
// Per face Jf[2NN*f + ...]: J00 = dF/dq_owner * len (row-major N x N), then
// J01 = dF/dq_neighbour * len.  Per real cell D[NN*c + ...] = A/dt I + sum of
// the cell's own blocks (+ the SA source row), Dinv its inverse.
#include <algorithm>

#include "afx_device.hpp"
#include "afx_implicit.hpp"

namespace afx {

// physics.h:533-578: forward differences with h = max(1e-6, |q|*1e-6), the
// perturbed component restored by subtraction (as the reference does, so a
// rounding difference persists into the later columns)
__global__ void __launch_bounds__(kBlock) k_face_jacobian(CellsT<double> C, FacesT<double> F, const double* __restrict__ q,
                                                          const double* __restrict__ gx, const double* __restrict__ gy,
                                                          GasT<double> g, int viscous, double* __restrict__ Jf) {
    int f = xcd_index();
    if (f >= F.nF) return;
    const size_t nT = (size_t)C.nT;
    const int o = F.c0[f], n = F.c1[f];
    const int kind = F.kind[f];
    const double nx = F.nx[f], ny = F.ny[f], L = F.len[f];
    double qL[4], qR[4];
    for (int k = 0; k < 4; ++k) { qL[k] = q[k * nT + o]; qR[k] = q[k * nT + n]; }
    const bool laminar = (viscous == 1) && (kind == K_INTERNAL);
    double gxa[4] = {0, 0, 0, 0}, gya[4] = {0, 0, 0, 0};
    if (laminar) {
        // solver.h:359-398, from the member state q and its gradients
        double t0 = C.xc[o] + C.xc[n];
        double t1 = C.yc[o] + C.yc[n];
        const double l = __builtin_sqrt(t0 * t0 + t1 * t1);
        t0 /= l; t1 /= l;
        for (int k = 0; k < 4; ++k) {
            double dir = (q[k * nT + o] - q[k * nT + n]) / l;
            double gxb = (gx[k * nT + o] + gx[k * nT + n]) * 0.5;
            double gyb = (gy[k * nT + o] + gy[k * nT + n]) * 0.5;
            const double dot = gxb * t0 + gyb * t1;
            gxa[k] = gxb - (dot - dir) * t0;
            gya[k] = gyb - (dot - dir) * t1;
        }
    }
    double f0[4], fp[4];
    face_flux<double>(g, kind, nx, ny, qL, qR, laminar, gxa, gya, f0);
    double* J = Jf + (size_t)32 * f;
    for (int i = 0; i < 4; ++i) {
        {
            const double a = 1e-6, b = dabs<double>(qL[i]) * 1e-6;
            const double up = (a < b) ? b : a;   // std::max(1e-6, |q|*1e-6)
            qL[i] += up;
            face_flux<double>(g, kind, nx, ny, qL, qR, laminar, gxa, gya, fp);
            qL[i] -= up;
            for (int r = 0; r < 4; ++r) J[4 * r + i] = (fp[r] - f0[r]) / up * L;
        }
        {
            const double a = 1e-6, b = dabs<double>(qR[i]) * 1e-6;
            const double up = (a < b) ? b : a;
            qR[i] += up;
            face_flux<double>(g, kind, nx, ny, qL, qR, laminar, gxa, gya, fp);
            qR[i] -= up;
            for (int r = 0; r < 4; ++r) J[16 + 4 * r + i] = (fp[r] - f0[r]) / up * L;
        }
    }
}

// Spalart-Allmaras: 5x5 blocks by the same rule (forward differences,
// h = max(1e-6, |v|*1e-6), the perturbed component restored by subtraction,
// first-order cell states, times the face length) of the five-variable face
// flux sa_face_flux.  The cell gradients gx, gy (5 planes) stay frozen; the
// face gradients' directional parts (v_n - v_o)/l, l along the cell
// connection, and the no-slip wall's cell-centre nu~ follow the perturbed
// states, so the viscous and nu~ diffusion couplings enter the blocks.  The
// rho nu~ column's step floor is 1e-6 mu_L instead of 1e-6 (rho nu~ is of the
// order mu_L chi; the absolute floor would perturb it by O(1)).
__global__ void __launch_bounds__(kBlock) k_face_jacobian_sa(CellsT<double> C, FacesT<double> F,
                                                             const double* __restrict__ q,
                                                             const double* __restrict__ gx,
                                                             const double* __restrict__ gy, GasT<double> g,
                                                             double* __restrict__ Jf) {
    const int f = xcd_index();
    if (f >= F.nF) return;
    const size_t nT = (size_t)C.nT;
    const int o = F.c0[f], n = F.c1[f];
    const int kind = F.kind[f];
    const double nx = F.nx[f], ny = F.ny[f], L = F.len[f];
    const bool internal = kind == K_INTERNAL;
    double a[5], b[5], gxb[5], gyb[5];
    for (int k = 0; k < 5; ++k) {
        a[k] = q[k * nT + o];
        b[k] = q[k * nT + n];
        gxb[k] = gyb[k] = 0.0;
    }
    double t0 = 0.0, t1 = 0.0, l = 1.0;
    if (internal) {
        t0 = C.xc[n] - C.xc[o];
        t1 = C.yc[n] - C.yc[o];
        l = __builtin_sqrt(t0 * t0 + t1 * t1);
        t0 /= l; t1 /= l;
        for (int k = 0; k < 5; ++k) {
            gxb[k] = (gx[k * nT + o] + gx[k * nT + n]) * 0.5;
            gyb[k] = (gy[k * nT + o] + gy[k * nT + n]) * 0.5;
        }
    }
    const double dn = (F.xf[f] - C.xc[o]) * nx + (F.yf[f] - C.yc[o]) * ny;
    auto flux = [&](double* out) {
        double gxa[5] = {0, 0, 0, 0, 0}, gya[5] = {0, 0, 0, 0, 0};
        if (internal)
            for (int k = 0; k < 5; ++k) {
                const double dir = (b[k] - a[k]) / l;
                const double dot = gxb[k] * t0 + gyb[k] * t1;
                gxa[k] = gxb[k] - (dot - dir) * t0;
                gya[k] = gyb[k] - (dot - dir) * t1;
            }
        sa_face_flux<double>(g, kind, nx, ny, a, b, gxa, gya, a[4] / a[0], dn, out);
    };
    double f0[5], fp[5];
    flux(f0);
    double* J = Jf + (size_t)50 * f;
    for (int i = 0; i < 5; ++i) {
        const double lo = i == 4 ? 1e-6 * g.mu : 1e-6;
        {
            const double hi = dabs<double>(a[i]) * 1e-6;
            const double up = (lo < hi) ? hi : lo;
            a[i] += up;
            flux(fp);
            a[i] -= up;
            for (int r = 0; r < 5; ++r) J[5 * r + i] = (fp[r] - f0[r]) / up * L;
        }
        {
            const double hi = dabs<double>(b[i]) * 1e-6;
            const double up = (lo < hi) ? hi : lo;
            b[i] += up;
            flux(fp);
            b[i] -= up;
            for (int r = 0; r < 5; ++r) J[25 + 5 * r + i] = (fp[r] - f0[r]) / up * L;
        }
    }
}

// N x N inverse by Gauss-Jordan with partial pivoting; returns false if
// singular.  Every loop is unrolled and the row exchange is a select over the
// candidate rows, so M is indexed at compile time only and stays in
// registers (a runtime row index would put it in scratch memory).
template <int N>
__device__ __forceinline__ bool invN(const double* A, double* X) {
    double M[N][2 * N];
#pragma unroll
    for (int r = 0; r < N; ++r)
#pragma unroll
        for (int c = 0; c < N; ++c) { M[r][c] = A[N * r + c]; M[r][c + N] = (r == c) ? 1.0 : 0.0; }
#pragma unroll
    for (int c = 0; c < N; ++c) {
        int p = c;
        double best = dabs<double>(M[c][c]);
#pragma unroll
        for (int r = c + 1; r < N; ++r) {
            const double a = dabs<double>(M[r][c]);
            if (a > best) { best = a; p = r; }
        }
        if (!(best > 0.0) || !isfinite(best)) return false;
#pragma unroll
        for (int r = c + 1; r < N; ++r) {   // exchange rows c and p
            const bool sw = r == p;
#pragma unroll
            for (int k = 0; k < 2 * N; ++k) {
                const double a = M[c][k], b = M[r][k];
                M[c][k] = sw ? b : a;
                M[r][k] = sw ? a : b;
            }
        }
        const double ip = 1.0 / M[c][c];
#pragma unroll
        for (int k = 0; k < 2 * N; ++k) M[c][k] *= ip;
#pragma unroll
        for (int r = 0; r < N; ++r) {
            if (r == c) continue;
            const double fct = M[r][c];
#pragma unroll
            for (int k = 0; k < 2 * N; ++k) M[r][k] -= fct * M[c][k];
        }
    }
#pragma unroll
    for (int r = 0; r < N; ++r)
#pragma unroll
        for (int c = 0; c < N; ++c) X[N * r + c] = M[r][c + N];
    return true;
}

// diagonal blocks (solver.h:1013-1056): A/dt on the diagonal, then the
// cell's own-state blocks of each of its faces in reference face order
// (owner: J00, neighbour: the lower block -J01); then their inverses.
// N = 5 adds the source row: -A dS/dv at the frozen gradients (same step
// rule and rho nu~ floor), its diagonal entry only where >= 0 (destruction),
// so production stays explicit and never lowers the diagonal of the nu~ row.
// With E non-null the same pass over the cell's faces writes the ELL copy of
// its row for the product in cell order (k_lhs_apply; with DILU the product
// reads the sweeps' colour-ordered copy instead): per slot s the off-diagonal
// block (-J00 where the cell is the face's neighbour, J01 where it is its
// owner; zero on empty slots and boundary faces) at E[(s NN + k) nC + c], the
// other cell at nbr[s nC + c] (-1: none), the diagonal block at Ds[k nC + c].
// Every ELL array is read with consecutive lanes on consecutive addresses.
template <int N>
__global__ void __launch_bounds__(kBlock) k_assemble_diag(CellsT<double> C, FacesT<double> F, const double* __restrict__ dt,
                                                          const double* __restrict__ Jf, SaSource src,
                                                          double* __restrict__ D, double* __restrict__ Dinv,
                                                          double* __restrict__ E, double* __restrict__ Ds,
                                                          int32_t* __restrict__ nbr, int* __restrict__ bad) {
    constexpr int NN = N * N;
    int c = xcd_index();
    if (c >= C.nC) return;
    const size_t nC = (size_t)C.nC;
    double B[NN];
    const double ad = C.area[c] / dt[c];
    for (int k = 0; k < NN; ++k) B[k] = 0.0;
    for (int k = 0; k < N; ++k) B[(N + 1) * k] = ad;
    for (int s = 0; s < 4; ++s) {
        const uint32_t e = C.cface[(size_t)s * nC + c];
        int other = -1;
        if (e != 0xFFFFFFFFu) {
            const int f = (int)(e & 0x7FFFFFFFu);
            const double* J = Jf + (size_t)2 * NN * f;
            const bool nb = (e >> 31) != 0;
            if (nb) for (int k = 0; k < NN; ++k) B[k] += -J[NN + k];
            else for (int k = 0; k < NN; ++k) B[k] += J[k];
            if (E && F.kind[f] == K_INTERNAL) {
                other = nb ? F.c0[f] : F.c1[f];
                for (int k = 0; k < NN; ++k) E[((size_t)s * NN + k) * nC + c] = nb ? -J[k] : J[NN + k];
            }
        }
        if (!E) continue;
        nbr[s * nC + c] = other;
        if (other < 0)
            for (int k = 0; k < NN; ++k) E[((size_t)s * NN + k) * nC + c] = 0.0;
    }
    if constexpr (N == 5) {
        if (src.q) {
            const size_t nT = (size_t)C.nT;
            double v[5], sx[5], sy[5];
            for (int k = 0; k < 5; ++k) {
                v[k] = src.q[k * nT + c];
                sx[k] = src.gx[k * nT + c];
                sy[k] = src.gy[k * nT + c];
            }
            const double d = src.wd[c], A = C.area[c];
            const double s0 = sa_cell_source<double>(src.g, v, sx, sy, d);
            for (int k = 0; k < 5; ++k) {
                const double lo = k == 4 ? 1e-6 * src.g.mu : 1e-6, hi = dabs<double>(v[k]) * 1e-6;
                const double up = (lo < hi) ? hi : lo;
                v[k] += up;
                const double sp = sa_cell_source<double>(src.g, v, sx, sy, d);
                v[k] -= up;
                double val = -A * (sp - s0) / up;
                if (k == 4 && val < 0) val = 0;
                B[20 + k] += val;
            }
        }
    }
    for (int k = 0; k < NN; ++k) {
        D[(size_t)NN * c + k] = B[k];
        if (E) Ds[k * nC + c] = B[k];
    }
    double X[NN];
    if (!invN<N>(B, X)) {
        atomicAdd(bad, 1);
        for (int k = 0; k < NN; ++k) X[k] = 0.0;
    }
    for (int k = 0; k < NN; ++k) Dinv[(size_t)NN * c + k] = X[k];
}

// y = LHS x (ghost rows identity; ghost columns dropped since x_ghost = 0)
// from the ELL copy written by k_assemble_diag.  Per row: the diagonal block
// times x_c, then each slot's block times the neighbour's x in slot order
// (the sign sits in the block instead of in x, exactly).
template <int N>
__global__ void __launch_bounds__(kBlock) k_lhs_apply(int32_t nC, int32_t nT, const double* __restrict__ Ds,
                                                      const double* __restrict__ E, const int32_t* __restrict__ nbr,
                                                      const double* __restrict__ x, double* __restrict__ y,
                                                      const int* __restrict__ active) {
    constexpr int NN = N * N;
    if (active && *active == 0) return;
    const int c = xcd_index();
    if (c >= nT) return;
    const size_t n = (size_t)nT, m = (size_t)nC;
    if (c >= nC) {
        for (int k = 0; k < N; ++k) y[k * n + c] = x[k * n + c];
        return;
    }
    int other[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) other[s] = nbr[s * m + c];
    double xc[N], acc[N];
    for (int k = 0; k < N; ++k) xc[k] = x[k * n + c];
    for (int r = 0; r < N; ++r) {
        double t = 0.0;
        for (int k = 0; k < N; ++k) t += Ds[(r * N + k) * m + c] * xc[k];
        acc[r] = t;
    }
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        if (other[s] < 0) continue;
        double xo[N];
        for (int k = 0; k < N; ++k) xo[k] = x[k * n + other[s]];
        const double* B = E + (size_t)s * NN * m + c;
        for (int r = 0; r < N; ++r) {
            double t = 0.0;
            for (int k = 0; k < N; ++k) t += B[(r * N + k) * m] * xo[k];
            acc[r] += t;
        }
    }
    for (int k = 0; k < N; ++k) y[k * n + c] = acc[k];
}

// z = Dinv x (ghost rows identity)
template <int N>
__global__ void __launch_bounds__(kBlock) k_block_jacobi(int32_t nC, int32_t nT, const double* __restrict__ Dinv,
                                                         const double* __restrict__ x, double* __restrict__ z,
                                                         const int* __restrict__ active) {
    if (active && *active == 0) return;
    int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= nT) return;
    const size_t n = (size_t)nT;
    if (c >= nC) {
        for (int k = 0; k < N; ++k) z[k * n + c] = x[k * n + c];
        return;
    }
    double xc[N];
    for (int k = 0; k < N; ++k) xc[k] = x[k * n + c];
    const double* B = Dinv + (size_t)N * N * c;
    for (int r = 0; r < N; ++r) {
        double t = 0.0;
        for (int k = 0; k < N; ++k) t += B[N * r + k] * xc[k];
        z[r * n + c] = t;
    }
}

// y += a * x
__global__ void __launch_bounds__(kBlock) k_axpy(double a, const double* __restrict__ x, double* __restrict__ y, int64_t n) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) y[i] += a * x[i];
}

// ------------------------------------------------ sums over a whole vector --
constexpr int kGsMax = 32;   // most columns of a Gram-Schmidt pass

// the sums over the wavefront of M values per lane (M a power of two, at most
// 32): halving exchanges leave value (lane >> shift) in a[0] of each lane
template <int M>
__device__ __forceinline__ int wave_sums(double* a) {
    const int lane = threadIdx.x & 63;
    int bit = 32;
#pragma unroll
    for (int h = M / 2; h >= 1; h /= 2, bit /= 2) {
        const bool up = (lane & bit) != 0;
#pragma unroll
        for (int q = 0; q < h; ++q) {
            const double give = up ? a[q] : a[q + h], keep = up ? a[q + h] : a[q];
            a[q] = keep + __shfl_xor(give, bit, 64);
        }
    }
    for (; bit >= 1; bit /= 2) a[0] += __shfl_xor(a[0], bit, 64);
    return lane / (64 / M);
}

// the block's sums of a[0 .. cnt): one slot per block in row k of partial
// (rows of gridDim.x); W wavefronts, this one's number wave
template <int M, int W>
__device__ __forceinline__ void block_sums(const double* a, int cnt, int wave, double* __restrict__ partial) {
    constexpr int P = M > 16 ? 32 : M > 8 ? 16 : M > 1 ? 8 : 1;
    __shared__ double red[W][P];
    double v[P];
#pragma unroll
    for (int k = 0; k < P; ++k) v[k] = k < M ? a[k] : 0.0;
    const int lane = threadIdx.x & 63;
    const int mine = wave_sums<P>(v);
    if (lane % (64 / P) == 0) red[wave][mine] = v[0];
    __syncthreads();
    const int k = wave * 64 + lane;
    if (k < cnt) {
        double t = 0.0;
#pragma unroll
        for (int q = 0; q < W; ++q) t += red[q][k];
        partial[(size_t)k * gridDim.x + blockIdx.x] = t;
    }
}
// Adds V_k . w of the wavefront's 64 entries (Ve: its basis entries, column k at
// 64 k) to red[k], k < m, eight columns at a time.  A small mesh runs these
// kernels once per wavefront, so their time is that of fetching their code:
// with all columns unrolled every further one cost 0.4 us, whatever the
// basis' layout; this loop's body is fetched once.
__device__ __forceinline__ void add_dots(const double* __restrict__ Ve, int m, double wi, bool live, double* red) {
    const int lane = threadIdx.x & 63;
#pragma unroll 1
    for (int g = 0; g < m; g += 8) {
        double a[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) a[q] = live ? Ve[64 * (g + q < m ? g + q : m - 1)] * wi : 0.0;
        const int k = g + wave_sums<8>(a);
        if (lane % 8 == 0 && k < m) red[k] += a[0];
    }
}
// the block's sums from its wavefronts' red[wave][k], k < cnt <= 64
template <int W, int C>
__device__ __forceinline__ void store_sums(const double (&red)[W][C], int cnt, double* __restrict__ partial) {
    __syncthreads();
    const int k = (int)threadIdx.y * 64 + (int)threadIdx.x;
    if (k >= cnt) return;
    double t = 0.0;
#pragma unroll
    for (int q = 0; q < W; ++q) t += red[q][k];
    partial[(size_t)k * gridDim.x + blockIdx.x] = t;
}
// sum of the nblk slots of one row by W neighbouring threads, in all of them
template <int W>
__device__ __forceinline__ double row_sum(const double* __restrict__ row, int nblk, int part) {
    double t = 0.0;
#pragma unroll 8
    for (int b = part; b < nblk; b += W) t += row[b];
#pragma unroll
    for (int off = W / 2; off > 0; off >>= 1) t += __shfl_xor(t, off, 64);
    return t;
}

// ------------------------------------------- multicolour block DILU (f1) --
// The reference preconditions GMRES with an incomplete LU (IncompleteLUT,
// solver.h:868-910).  On the device: block DILU in a colour order of the
// real cells (no two face neighbours share a colour), so each colour is one
// parallel sweep.  With A_ij the off-diagonal block of row i, column j:
//   Dt_i = D_i - sum_{j before i} A_ij Dt_j^-1 A_ji          (set-up, by colour)
//   M = (Dt + L) Dt^-1 (Dt + U),  L / U: the blocks A_ij with j before / after i.
// Off-diagonal blocks from the face Jacobians: for face f with owner o and
// neighbour n, A_on = J01(f) and A_no = -J00(f); boundary faces have none.

// the block A_ij (sgn, J) of cell i across its slot entry e, and the other cell
template <int N>
__device__ __forceinline__ const double* offdiag(const FacesT<double>& F, const double* Jf, uint32_t e, int* other,
                                                  double* sgn) {
    const int f = (int)(e & 0x7FFFFFFFu);
    const double* J = Jf + (size_t)2 * N * N * f;
    if (e >> 31) { *other = F.c0[f]; *sgn = -1.0; return J; }        // i is the neighbour: -J00
    *other = F.c1[f]; *sgn = 1.0; return J + N * N;                   // i is the owner: J01
}
// the transposed-position block A_ji of the same face
template <int N>
__device__ __forceinline__ const double* offdiag_t(const double* Jf, uint32_t e, double* sgn) {
    const int f = (int)(e & 0x7FFFFFFFu);
    const double* J = Jf + (size_t)2 * N * N * f;
    if (e >> 31) { *sgn = 1.0; return J + N * N; }
    *sgn = -1.0; return J;
}

// Set-up of colour c over positions p0 .. p0 + ncells of the colour order.
// Besides Dt_i^-1 (AoS, read back by the later colours' set-up) it writes the
// sweeps' colour-ordered ELL copy of row i at its position p: the
// off-diagonal blocks A_ij by slot at Ec[(s NN + k) nC + p], the neighbour
// code nc[s nC + p] = pos_j + 1 for a neighbour of an earlier colour,
// -(pos_j + 1) for a later one, 0 for none (pos_j: the neighbour's position in
// the colour order), Dt_i^-1 at Dc[k nC + p] and D_i at Dp[k nC + p] (for the
// product), so the threads of one colour's sweep read consecutive addresses.
template <int N>
__global__ void __launch_bounds__(kBlock) k_dilu_setup(CellsT<double> C, FacesT<double> F, const uint8_t* __restrict__ colour,
                                                       int c, const int32_t* __restrict__ cells,
                                                       const int32_t* __restrict__ pos, int32_t p0,
                                                       int32_t ncells, const double* __restrict__ D,
                                                       const double* __restrict__ Jf, double* __restrict__ Dti,
                                                       double* __restrict__ Ec, int32_t* __restrict__ nc,
                                                       double* __restrict__ Dc, double* __restrict__ Dp,
                                                       int* __restrict__ bad) {
    constexpr int NN = N * N;
    const int k = xcd_index();
    if (k >= ncells) return;
    const size_t mc = (size_t)C.nC;
    const int p = p0 + k;
    const int i = cells[p];
    double B[NN];
    for (int r = 0; r < NN; ++r) {
        B[r] = D[(size_t)NN * i + r];
        Dp[r * mc + p] = B[r];
    }
    for (int s = 0; s < 4; ++s) {
        const uint32_t e = C.cface[(size_t)s * C.nC + i];
        if (e == 0xFFFFFFFFu) break;
        if (F.kind[e & 0x7FFFFFFFu] != K_INTERNAL) continue;
        int j;
        double sa, sb;
        const double* Aij = offdiag<N>(F, Jf, e, &j, &sa);
        if (colour[j] >= c) continue;
        const double* Aji = offdiag_t<N>(Jf, e, &sb);
        const double* Pj = Dti + (size_t)NN * j;
        double T[NN];   // Dt_j^-1 A_ji
        for (int r = 0; r < N; ++r)
            for (int q = 0; q < N; ++q) {
                double t = 0.0;
                for (int m = 0; m < N; ++m) t += Pj[N * r + m] * Aji[N * m + q];
                T[N * r + q] = sb * t;
            }
        for (int r = 0; r < N; ++r)
            for (int q = 0; q < N; ++q) {
                double t = 0.0;
                for (int m = 0; m < N; ++m) t += Aij[N * r + m] * T[N * m + q];
                B[N * r + q] -= sa * t;
            }
    }
    double X[NN];
    if (!invN<N>(B, X)) {
        atomicAdd(bad, 1);
        for (int r = 0; r < NN; ++r) X[r] = 0.0;
    }
    for (int r = 0; r < NN; ++r) {
        Dti[(size_t)NN * i + r] = X[r];
        Dc[r * mc + p] = X[r];
    }
    for (int s = 0; s < 4; ++s) {
        const uint32_t e = C.cface[(size_t)s * mc + i];
        int code = 0;
        if (e != 0xFFFFFFFFu && F.kind[e & 0x7FFFFFFFu] == K_INTERNAL) {
            int j;
            double sa;
            const double* Aij = offdiag<N>(F, Jf, e, &j, &sa);
            code = colour[j] < c ? pos[j] + 1 : -(pos[j] + 1);
            for (int r = 0; r < NN; ++r) Ec[((size_t)s * NN + r) * mc + p] = sa * Aij[r];
        } else {
            for (int r = 0; r < NN; ++r) Ec[((size_t)s * NN + r) * mc + p] = 0.0;
        }
        nc[s * mc + p] = code;
    }
}

// The sweeps and the product work in the colour order: vectors are nv planes
// of nC by position, and stay so through the whole Arnoldi process.  A
// workgroup takes 64 positions and its wavefronts share the N rows of their
// blocks, R rows each, so that every load reads consecutive addresses; where
// the inverted diagonal block needs all rows they meet in LDS.  One thread per
// cell (R = N) loads a neighbour's vector once for all rows and is bound by
// HBM on large meshes; one thread per row and cell (R = 1) has N times the
// loads in flight, which counts where a colour's few thousand cells leave most
// SIMDs without a wavefront (split_rows below).
// Each XCD takes a contiguous eighth of every colour in all of these kernels,
// sweeps, product and Gram-Schmidt passes alike, so that its share of the
// vectors of a small mesh stays in its L2 from one kernel to the next.
__device__ __forceinline__ int row_position(int32_t n) {
    const int k = xcd_tile((int)blockIdx.x, (int)gridDim.x) * 64 + (int)threadIdx.x;
    return k < n ? k : -1;
}
// position of this lane in the t-th tile (64 positions of one colour) of the
// block's XCD, -1 past the colour's end; t < S.per_xcd
__device__ __forceinline__ int span_position(const Span& S, int t) {
    int c = 0, per = S.per[0];
    while (t >= per) {
        t -= per;
        per = S.per[++c];
    }
    const int p = S.off[c] + ((int)(blockIdx.x & 7) * per + t) * 64 + (int)threadIdx.x;
    return p < S.off[c + 1] ? p : -1;
}
// The Krylov basis of `cap` columns: 64 consecutive positions of one row lie
// together for all columns, column k of position p, row r (of N) at
// basis_at(p, r, N, cap) + 64 k, so a wavefront's reads over the columns stay in
// one or two stretches of 64 cap doubles.
__device__ __forceinline__ size_t basis_at(size_t p, int r, int N, int cap) {
    return ((p >> 6) * N + r) * (size_t)cap * 64 + (p & 63);
}
// acc[rr] += sgn (A x_j)_(r0 + rr) of the N x N block at A (entries stride m apart)
template <int N, int R>
__device__ __forceinline__ void add_rows(const double* __restrict__ A, size_t m, int r0, const double* xj, double sgn,
                                         double* acc) {
#pragma unroll
    for (int rr = 0; rr < R; ++rr) {
        double t = 0.0;
#pragma unroll
        for (int q = 0; q < N; ++q) t += A[((r0 + rr) * N + q) * m] * xj[q];
        acc[rr] += sgn * t;
    }
}
template <int N>
__device__ __forceinline__ void load_cell(const double* __restrict__ x, size_t m, int p, double* v) {
#pragma unroll
    for (int q = 0; q < N; ++q) v[q] = x[q * m + p];
}
// all N rows of acc in every thread of the cell
template <int N, int R>
__device__ __forceinline__ void share_rows(const double* acc, int r0, double* all) {
    if constexpr (R == N) {
#pragma unroll
        for (int q = 0; q < N; ++q) all[q] = acc[q];
    } else {
        __shared__ double sh[N][64];
#pragma unroll
        for (int rr = 0; rr < R; ++rr) sh[r0 + rr][threadIdx.x] = acc[rr];
        __syncthreads();
#pragma unroll
        for (int q = 0; q < N; ++q) all[q] = sh[q][threadIdx.x];
    }
}

// forward sweep of one colour (positions p0 .. p0 + ncells):
//   y_i = Dt_i^-1 (v_i - sum_{j before i} A_ij y_j)
// with v from SRC 0: in; 1: a (in - sum_{k < cols} coef_k V_k), also written to
// column cols of V (the next basis vector); 2: sum_{k < *jend} coef_k V_k (the
// cycle's result)
template <int N, int R, int SRC>
__global__ void __launch_bounds__(64 * N / R) k_dilu_forward(int32_t nC, int32_t p0, int32_t ncells,
                                                             const double* __restrict__ Ec,
                                                             const int32_t* __restrict__ nc,
                                                             const double* __restrict__ Dc,
                                                             const double* __restrict__ in,
                                                             const double* __restrict__ a, double* __restrict__ V,
                                                             int cap, int cols, const int* __restrict__ jend,
                                                             const double* __restrict__ coef, double* __restrict__ yp,
                                                             const int* __restrict__ active) {
    constexpr int NN = N * N;
    const int r0 = threadIdx.y * R;
    const int k = row_position(ncells);
    const size_t m = (size_t)nC;
    const int p = p0 + (k >= 0 ? k : 0);
    // everything whose address is known goes out before the first wait
    const int on = active ? *active : 1;
    int code[4];
#pragma unroll
    for (int sl = 0; sl < 4; ++sl) code[sl] = nc[sl * m + p];
    double acc[R], dc[R == 1 ? N : 1];
#pragma unroll
    for (int rr = 0; rr < R; ++rr) acc[rr] = SRC != 2 ? in[(r0 + rr) * m + p] : 0.0;
    if constexpr (R == 1) {
#pragma unroll
        for (int q = 0; q < N; ++q) dc[q] = Dc[(r0 * N + q) * m + p];
    }
    if (!on) return;
    if (SRC != 0) {
        const double s = SRC == 1 ? *a : 1.0;
        const int nq = SRC == 2 ? *jend : cols;
#pragma unroll
        for (int rr = 0; rr < R; ++rr) {
            double* Ve = V + basis_at(p, r0 + rr, N, cap);
            double t = 0.0;
#pragma unroll 8
            for (int q = 0; q < nq; ++q) t += coef[q] * Ve[64 * q];
            acc[rr] = SRC == 1 ? s * (acc[rr] - t) : t;
            if (SRC == 1 && k >= 0) Ve[64 * cols] = acc[rr];
        }
    }
#pragma unroll
    for (int sl = 0; sl < 4; ++sl) {
        if (code[sl] <= 0) continue;
        double yj[N];
        load_cell<N>(yp, m, code[sl] - 1, yj);
        add_rows<N, R>(Ec + (size_t)sl * NN * m + p, m, r0, yj, -1.0, acc);
    }
    double all[N];
    share_rows<N, R>(acc, r0, all);
    if (k < 0) return;
    double out[R];
#pragma unroll
    for (int rr = 0; rr < R; ++rr) out[rr] = 0.0;
    if constexpr (R == 1) {
#pragma unroll
        for (int q = 0; q < N; ++q) out[0] += dc[q] * all[q];
    } else {
        add_rows<N, R>(Dc + p, m, r0, all, 1.0, out);
    }
#pragma unroll
    for (int rr = 0; rr < R; ++rr) yp[(r0 + rr) * m + p] = out[rr];
}

// backward sweep of one colour, in place:
//   y_i -= Dt_i^-1 sum_{j after i} A_ij y_j
template <int N, int R>
__global__ void __launch_bounds__(64 * N / R) k_dilu_backward(int32_t nC, int32_t p0, int32_t ncells,
                                                              const double* __restrict__ Ec,
                                                              const int32_t* __restrict__ nc,
                                                              const double* __restrict__ Dc, double* __restrict__ yp,
                                                              const int* __restrict__ active) {
    constexpr int NN = N * N;
    const int r0 = threadIdx.y * R;
    const int k = row_position(ncells);
    const size_t m = (size_t)nC;
    const int p = p0 + (k >= 0 ? k : 0);
    const int on = active ? *active : 1;
    int code[4];
#pragma unroll
    for (int sl = 0; sl < 4; ++sl) code[sl] = nc[sl * m + p];
    double acc[R], dc[R == 1 ? N : 1];
#pragma unroll
    for (int rr = 0; rr < R; ++rr) acc[rr] = 0.0;
    if constexpr (R == 1) {
#pragma unroll
        for (int q = 0; q < N; ++q) dc[q] = Dc[(r0 * N + q) * m + p];
    }
    if (!on) return;
    bool any = false;
#pragma unroll
    for (int sl = 0; sl < 4; ++sl) {
        if (code[sl] >= 0) continue;
        any = true;
        double yj[N];
        load_cell<N>(yp, m, -code[sl] - 1, yj);
        add_rows<N, R>(Ec + (size_t)sl * NN * m + p, m, r0, yj, 1.0, acc);
    }
    double all[N];
    share_rows<N, R>(acc, r0, all);
    if (!any || k < 0) return;
    double out[R];
#pragma unroll
    for (int rr = 0; rr < R; ++rr) out[rr] = 0.0;
    if constexpr (R == 1) {
#pragma unroll
        for (int q = 0; q < N; ++q) out[0] += dc[q] * all[q];
    } else {
        add_rows<N, R>(Dc + p, m, r0, all, 1.0, out);
    }
#pragma unroll
    for (int rr = 0; rr < R; ++rr) yp[(r0 + rr) * m + p] -= out[rr];
}

// y = A x by position: the diagonal block times x_i, then each slot's block
// times the neighbour's x in slot order, as k_lhs_apply does in cell order.
// M > 0: also the block's share of V_k . y for the first cols basis vectors (at
// most M with whole cells, any number with split rows) into row k of partial
// (the first Gram-Schmidt pass, without reading y back).
// The grid strides over the tiles of 64 cells.
template <int N, int R, int G, int M>
__global__ void __launch_bounds__(64 * G * N / R) k_colour_apply(int32_t nC, Span S, const double* __restrict__ Dp,
                                                                 const double* __restrict__ Ec,
                                                                 const int32_t* __restrict__ nc,
                                                                 const double* __restrict__ x, double* __restrict__ y,
                                                                 const double* __restrict__ V, int cap, int cols,
                                                                 double* __restrict__ partial,
                                                                 const int* __restrict__ active) {
    constexpr int NN = N * N, Q = N / R;
    const int on = active ? *active : 1;
    if (!on) return;
    const int r0 = ((int)threadIdx.y % Q) * R, group = (int)threadIdx.y / Q;
    const size_t m = (size_t)nC;
    constexpr bool LOOP = R == 1 && M > 0;   // small meshes: see add_dots
    double dots[M > 0 ? M : 1];
#pragma unroll
    for (int k = 0; k < M; ++k) dots[k] = 0.0;
    __shared__ double red[LOOP ? G * Q : 1][LOOP ? kGsMax : 1];
    if (LOOP && threadIdx.x < kGsMax) red[threadIdx.y][threadIdx.x] = 0.0;
    for (int i = (int)(blockIdx.x >> 3) * G + group; i < S.per_xcd; i += (int)(gridDim.x >> 3) * G) {
        const int at = span_position(S, i);
        if (!LOOP && at < 0) continue;
        const int p = at < 0 ? 0 : at;
        double acc[R], xj[N];
#pragma unroll
        for (int rr = 0; rr < R; ++rr) acc[rr] = 0.0;
        load_cell<N>(x, m, p, xj);
        add_rows<N, R>(Dp + p, m, r0, xj, 1.0, acc);
#pragma unroll
        for (int sl = 0; sl < 4; ++sl) {
            const int code = nc[sl * m + p];
            if (code == 0) continue;
            load_cell<N>(x, m, (code > 0 ? code : -code) - 1, xj);
            add_rows<N, R>(Ec + (size_t)sl * NN * m + p, m, r0, xj, 1.0, acc);
        }
        if (at >= 0) {
#pragma unroll
            for (int rr = 0; rr < R; ++rr) y[(r0 + rr) * m + p] = acc[rr];
        }
        if constexpr (LOOP) {
            add_dots(V + basis_at(p, r0, N, cap), cols, acc[0], at >= 0, red[threadIdx.y]);
        } else if constexpr (M > 0) {
#pragma unroll
            for (int rr = 0; rr < R; ++rr) {
                const double* Ve = V + basis_at(p, r0 + rr, N, cap);
#pragma unroll
                for (int k = 0; k < M; ++k)
                    if (k < cols) dots[k] += Ve[64 * k] * acc[rr];
            }
        }
    }
    if constexpr (LOOP) {
        store_sums<G * Q>(red, cols, partial);
    } else if constexpr (M > 0) {
        block_sums<M, G * Q>(dots, cols, threadIdx.y, partial);
    }
}

// between cell order (planes of nT) and the colour order (planes of nC):
// out_p = b_i - w_p (w null: b_i)
__global__ void __launch_bounds__(kBlock) k_to_colour(int32_t nC, int32_t nT, int nv, const int32_t* __restrict__ cells,
                                                      const double* __restrict__ b, const double* __restrict__ w,
                                                      double* __restrict__ out) {
    const int p = xcd_index();
    if (p >= nC) return;
    const int i = cells[p];
    for (int k = 0; k < nv; ++k) {
        const double v = b[(size_t)k * nT + i];
        out[(size_t)k * nC + p] = w ? v - w[(size_t)k * nC + p] : v;
    }
}
// z_i = yp at the position of real cell i; ghost rows are identity rows, z = x
__global__ void __launch_bounds__(kBlock) k_from_colour(int32_t nC, int32_t nT, int nv, const int32_t* __restrict__ pos,
                                                        const double* __restrict__ yp, const double* __restrict__ x,
                                                        double* __restrict__ z) {
    const int i = xcd_index();
    if (i >= nT) return;
    if (i >= nC) {
        for (int k = 0; k < nv; ++k) z[(size_t)k * nT + i] = x[(size_t)k * nT + i];
        return;
    }
    const int p = pos[i];
    for (int r = 0; r < nv; ++r) z[(size_t)r * nT + i] = yp[(size_t)r * nC + p];
}
// end of a restart cycle: x_p = z_p (first cycle) or x_p + z_p, and dq_i = x_p
// in cell order; once converged also q_i += relax dq_i
__global__ void __launch_bounds__(kBlock) k_colour_update(int32_t nC, int32_t nT, int nv,
                                                          const int32_t* __restrict__ pos, int first, double relax,
                                                          const double* __restrict__ z, double* __restrict__ x,
                                                          double* __restrict__ dq, double* __restrict__ q,
                                                          const int* __restrict__ converged) {
    const int i = xcd_index();
    if (i >= nC) return;
    const int p = pos[i];
    const bool add = *converged != 0;
    for (int r = 0; r < nv; ++r) {
        const size_t e = (size_t)r * nC + p, c = (size_t)r * nT + i;
        double v = z[e];
        if (!first) v = x[e] + v;
        x[e] = v;
        dq[c] = v;
        if (add) q[c] += relax * v;
    }
}

// --------------------------------------------- device-resident GMRES (f1) --
// One Arnoldi step j with classical Gram-Schmidt applied twice:
//   (1) h1 = V^T w, block sums in partial (with DILU inside the product);
//   (2) every block adds h1 up, then w -= V h1, and h2 = V^T w and |w|^2 of the
//       result, block sums in the second half of partial;
//   (3) one block: h2, |w - V h2|^2 = |w|^2 - |h2|^2 (V orthonormal, h2 only the
//       rounding of pass 1; at a breakdown, where w is rounding too, summed from
//       the vector, a branch that costs 0.2 us where it is not taken), the Givens
//       step, flags and scale;
//   (4) the next basis vector a (w - V h2), formed where it is first read (the
//       forward sweeps).
// So the basis is read three times and a step of two colours is six launches.
// Sums are added by the kernel that needs them: separate reduction, rotation
// and scaling kernels cost 2.4 to 7.8 us each, five per step, and a last-block
// reduction with an arrival counter 50 to 85 us a pass at 500k cells.  A step of a 16k-cell
// mesh took 78 us in fifteen launches, now 41 in seven or eight (2.3 us is a
// launch); at 500k cells (5x5 blocks) the passes of a short basis went from
// 42 + 19 us to 23 + 7.

// start of a cycle from |r|^2: the first cycle sets beta0 (zero right-hand
// side: converged at once); a restart tests the true residual against tol
// beta0.  One thread.
__device__ __forceinline__ void gm_begin(const GmDev& G, int first, double rr) {
    const double beta = __builtin_sqrt(rr);
    if (first) { G.hdr[0] = beta; G.flags[1] = 0; G.flags[2] = 0; }
    G.hdr[1] = beta;
    G.flags[3] = 0;
    for (int k = 0; k <= G.m; ++k) G.g[k] = 0.0;
    G.g[0] = beta;
    const bool done = first ? !(beta > 0.0) : (beta <= G.tol * G.hdr[0]);
    if (done) {
        G.flags[1] = 1;
        G.flags[0] = 0;
        if (G.seen) {   // the host's copy, in pinned memory
            G.seen[0] = 0;
            G.seen[1] = 1;
            G.seen[2] = G.flags[2];
            G.seen[3] = 0;
        }
    } else {
        G.flags[0] = 1;
        G.hdr[2] = 1.0 / beta;
    }
}

__device__ __forceinline__ double lane_value(double v, int lane) {
    const long long b = __double_as_longlong(v);
    const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)b, lane);
    const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(b >> 32), lane);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// The Gram-Schmidt passes take the vectors as N rows of len positions (DILU:
// N planes of nC in the colour order; otherwise one row) and G tiles of 64
// positions per block and turn, one wavefront per row and tile.
//
// pass 1 on its own: V_k . w, k < m
template <int N, int G, int MM>
__global__ void __launch_bounds__(64 * N * G) k_gs_dots(const double* __restrict__ V, int cap, size_t len, Span S,
                                                        int m, const double* __restrict__ w, double* __restrict__ partial,
                                                        const int* __restrict__ active) {
    if (active && *active == 0) return;
    double acc[MM];
#pragma unroll
    for (int k = 0; k < MM; ++k) acc[k] = 0.0;
    const int r = (int)threadIdx.y % N, group = (int)threadIdx.y / N;
    for (int t = (int)(blockIdx.x >> 3) * G + group; t < S.per_xcd; t += (int)(gridDim.x >> 3) * G) {
        const int p = span_position(S, t);
        if (p < 0) continue;
        const double wi = w[r * len + p];
        const double* Ve = V + basis_at(p, r, N, cap);
#pragma unroll
        for (int k = 0; k < MM; ++k)
            if (k < m) acc[k] += Ve[64 * k] * wi;
    }
    block_sums<MM, N * G>(acc, m, threadIdx.y, partial);
}

// pass 2: h1 from the nblk1 block sums of pass 1 (block 0 keeps it for the
// step), w -= V h1, then V_k . w into rows 0 .. m - 1 and |w|^2 into row kGsMax
// of sums2
template <int N, int G, int MM>
__global__ void __launch_bounds__(64 * N * G) k_gs_update(const double* __restrict__ V, int cap, size_t len, Span S,
                                                          int m, const double* __restrict__ sums1, int nblk1,
                                                          double* __restrict__ w, double* __restrict__ sums2,
                                                          double* __restrict__ h1, const int* __restrict__ active) {
    const int on = active ? *active : 1;
    constexpr int P = MM > 16 ? 32 : MM;
    constexpr int W = kBlock / P;   // the first kBlock threads add the sums up
    __shared__ double hs[P];
    const int tid = (int)threadIdx.y * 64 + (int)threadIdx.x;
    {
        const int k = tid / W, part = tid % W;
        const double t = tid < kBlock ? row_sum<W>(sums1 + (size_t)(k < m ? k : 0) * nblk1, nblk1, part) : 0.0;
        if (!on) return;
        if (tid < kBlock && part == 0) {
            hs[k] = k < m ? t : 0.0;
            if (blockIdx.x == 0 && k < m) h1[k] = t;
        }
    }
    __syncthreads();
    double hk[MM], acc[MM], ww = 0.0;
#pragma unroll
    for (int k = 0; k < MM; ++k) {
        hk[k] = hs[k];
        acc[k] = 0.0;
    }
    const int r = (int)threadIdx.y % N, group = (int)threadIdx.y / N;
    for (int t = (int)(blockIdx.x >> 3) * G + group; t < S.per_xcd; t += (int)(gridDim.x >> 3) * G) {
        const int p = span_position(S, t);
        if (p < 0) continue;
        const size_t i = r * len + p;
        const double* Ve = V + basis_at(p, r, N, cap);
        double v[MM];
        double wi = w[i];
#pragma unroll
        for (int k = 0; k < MM; ++k)
            if (k < m) v[k] = Ve[64 * k];
#pragma unroll
        for (int k = 0; k < MM; ++k)
            if (k < m) wi -= hk[k] * v[k];
        w[i] = wi;
#pragma unroll
        for (int k = 0; k < MM; ++k)
            if (k < m) acc[k] += v[k] * wi;
        ww += wi * wi;
    }
    block_sums<MM, N * G>(acc, m, threadIdx.y, sums2);
    block_sums<1, N * G>(&ww, 1, threadIdx.y, sums2 + (size_t)kGsMax * gridDim.x);
}

// the same for a small mesh (see add_dots), eight columns at a time; the basis
// is read again for the second set of sums, from the caches
template <int N>
__global__ void __launch_bounds__(64 * N) k_gs_update_small(const double* __restrict__ V, int cap, size_t len, Span S,
                                                            int m, const double* __restrict__ sums1, int nblk1,
                                                            double* __restrict__ w, double* __restrict__ sums2,
                                                            double* __restrict__ h1, const int* __restrict__ active) {
    constexpr int W = kBlock / kGsMax;
    __shared__ double hs[kGsMax], red[N][kGsMax], rw[N][1];
    const int tid = (int)threadIdx.y * 64 + (int)threadIdx.x, r = threadIdx.y;
    const int on = active ? *active : 1;
    if (tid < kBlock) {
        const int k = tid / W, part = tid % W;
        const double t = row_sum<W>(sums1 + (size_t)(k < m ? k : 0) * nblk1, nblk1, part);
        if (part == 0) {
            hs[k] = k < m ? t : 0.0;
            if (on && blockIdx.x == 0 && k < m) h1[k] = t;
        }
    }
    if (threadIdx.x < kGsMax) red[r][threadIdx.x] = 0.0;
    if (!on) return;
    __syncthreads();
    double ww = 0.0;
    for (int t = (int)(blockIdx.x >> 3); t < S.per_xcd; t += (int)(gridDim.x >> 3)) {
        const int p = span_position(S, t);
        const size_t i = r * len + (p >= 0 ? p : 0);
        const double* Ve = V + basis_at(p >= 0 ? p : 0, r, N, cap);
        double wi = p >= 0 ? w[i] : 0.0;
#pragma unroll 1
        for (int g = 0; g < m; g += 8) {
            double v[8];
#pragma unroll
            for (int q = 0; q < 8; ++q) v[q] = Ve[64 * (g + q < m ? g + q : m - 1)];
#pragma unroll
            for (int q = 0; q < 8; ++q) wi -= hs[g + q] * v[q];   // zero past the last column
        }
        if (p >= 0) w[i] = wi;
        else wi = 0.0;
        add_dots(Ve, m, wi, p >= 0, red[r]);
        ww += wi * wi;
    }
    (void)wave_sums<1>(&ww);
    if (threadIdx.x == 0) rw[r][0] = ww;
    store_sums<N>(red, m, sums2);
    store_sums<N>(rw, 1, sums2 + (size_t)kGsMax * gridDim.x);
}

// The step: 16 threads add up each of the j + 1 coefficients of pass 2 and
// |w|^2; then one wavefront forms the Hessenberg column j, applies the previous
// Givens rotations and a new one, and sets the residual estimate |g_{j+1}|, the
// flags and the scale of the next basis vector.  Lane i holds entry i of the
// column and rotation i, and the chain of rotations runs on lane reads (from
// memory, one thread's chain took 7.8 us for 30 columns).  show: the host
// reads the flags next (the write to its memory costs about a microsecond).
// The vectors are N rows of len positions.
constexpr int kStepWaves = 9;
__global__ void __launch_bounds__(64 * kStepWaves) k_gm_step(GmDev G, int j, int show, const double* __restrict__ sums2,
                                                             int nblk, const double* __restrict__ V, int N, int64_t len,
                                                             const double* __restrict__ w) {
    __shared__ double h2[kGsMax + 4], left[kStepWaves];
    const int k = threadIdx.x / 16, part = threadIdx.x % 16, lane = threadIdx.x;
    const int m = G.m;
    const int on = G.flags[0], total = G.flags[2] + 1;
    const bool first = lane < 64;
    const double cs = first && lane < j ? G.cs[lane] : 1.0, sn = first && lane < j ? G.sn[lane] : 0.0;
    const double h1 = first && lane <= j ? G.h1[lane] : 0.0;
    const double gj = G.g[j], target = G.tol * G.hdr[0];
    const int row = k <= j ? k : kGsMax;   // j + 1: |w|^2
    const double t = row_sum<16>(sums2 + (size_t)row * nblk, nblk, part);
    if (!on) return;
    if (part == 0 && k <= j + 1) h2[k] = t;
    __syncthreads();
    const int at = lane & 63;
    const double c2 = at <= j ? h2[at] : 0.0;
    if (lane <= j) G.h2[lane] = c2;
    double hh = c2 * c2;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) hh += __shfl_xor(hh, off, 64);
    double ww = h2[j + 1] - hh;
    // A breakdown: most of what pass 1 left lies in the basis' span, so it is
    // rounding and the difference has few digits or none.  Every wave sees the
    // same sums and goes the same way.
    if (ww < 0.25 * h2[j + 1]) {
        double sum = 0.0;
        const int64_t tiles = (len + 63) / 64 * N;
        for (int64_t q = lane >> 6; q < tiles; q += kStepWaves) {
            const int r = (int)(q % N);
            const int64_t p = q / N * 64 + at;
            if (p >= len) continue;
            const double* Ve = V + basis_at((size_t)p, r, N, m + 1);
            double v = 0.0;
            for (int i = 0; i <= j; ++i) v += h2[i] * Ve[64 * i];
            v = w[r * len + p] - v;
            sum += v * v;
        }
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) sum += __shfl_xor(sum, off, 64);
        if (at == 0) left[lane >> 6] = sum;
        __syncthreads();
        ww = 0.0;
        for (int q = 0; q < kStepWaves; ++q) ww += left[q];
    }
    if (!first) return;
    const double nrm = __builtin_sqrt(ww > 0.0 ? ww : 0.0);
    const double h = h1 + c2;
    double mine = 0.0, a = lane_value(h, 0);
    for (int i = 0; i < j; ++i) {
        const double bb = lane_value(h, i + 1), c = lane_value(cs, i), s = lane_value(sn, i);
        const double top = c * a + s * bb;
        a = -s * a + c * bb;
        mine = lane == i ? top : mine;
    }
    double* H = G.H;
    if (lane < j) H[(size_t)lane * m + j] = mine;
    if (lane != 0) return;
    const double r = hypot(a, nrm);
    const double c = r > 0 ? a / r : 1.0, s = r > 0 ? nrm / r : 0.0;
    const double next = -s * gj;
    G.cs[j] = c;
    G.sn[j] = s;
    H[(size_t)j * m + j] = r;
    H[(size_t)(j + 1) * m + j] = 0.0;
    G.g[j + 1] = next;
    G.g[j] = c * gj;
    const bool converged = fabs(next) <= target;
    const bool active = !converged && nrm > 0 && total < G.maxit;
    if (active) G.hdr[2] = 1.0 / nrm;
    G.flags[0] = active;
    G.flags[1] = converged;
    G.flags[2] = total;
    G.flags[3] = j + 1;
    if (G.seen && (show || !active)) {
        G.seen[0] = active;
        G.seen[1] = converged;
        G.seen[2] = total;
        G.seen[3] = j + 1;
    }
}

// |r|^2, block sums in partial, and a cycle's set-up from them
__global__ void __launch_bounds__(kBlock) k_gm_norm(const double* __restrict__ r, int64_t n,
                                                    double* __restrict__ partial) {
    double t = 0.0;
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += (int64_t)gridDim.x * kBlock)
        t += r[i] * r[i];
    block_sums<1, kBlock / 64>(&t, 1, threadIdx.x >> 6, partial);
}
__global__ void __launch_bounds__(64) k_gm_begin(GmDev G, int first, const double* __restrict__ partial, int nblk) {
    const double rr = row_sum<64>(partial, nblk, threadIdx.x);
    if (threadIdx.x == 0) gm_begin(G, first, rr);
}

// y = H^-1 g over the cycle's jend columns (upper triangular), lane i holding
// g_i and subtracting column after column
__global__ void __launch_bounds__(64) k_gm_solve(GmDev G) {
    const int m = G.m, jend = G.flags[3], lane = threadIdx.x;
    double g = lane < jend ? G.g[lane] : 0.0;
    for (int k = jend - 1; k >= 0; --k) {
        const double col = lane <= k ? G.H[(size_t)lane * m + k] : 0.0;
        const double y = lane_value(g, k) / lane_value(col, k);
        if (lane < k) g -= col * y;
        if (lane == k) G.y[k] = y;
    }
}

// the next basis vector a (w - sum_{k < m} h2_k V_k) into column m of V and
// into v (which may be w)
__global__ void __launch_bounds__(kBlock) k_next_vector(const double* __restrict__ a, const double* __restrict__ h2,
                                                        int m, const double* w, double* __restrict__ V, int cap,
                                                        double* v, int64_t n, const int* __restrict__ active) {
    if (active && *active == 0) return;
    const double s = *a;
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double* Ve = V + basis_at(i, 0, 1, cap);
    double t = 0.0;
#pragma unroll 8
    for (int k = 0; k < m; ++k) t += h2[k] * Ve[64 * k];
    const double next = s * (w[i] - t);
    Ve[64 * m] = next;
    v[i] = next;
}

// x = sum_{k < jend} y_k V_k, jend on the device
__global__ void __launch_bounds__(kBlock) k_lincomb_dev(const double* __restrict__ V, int cap,
                                                        const int* __restrict__ jend, const double* __restrict__ y,
                                                        double* __restrict__ x, int64_t n) {
    const int m = *jend;
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double* Ve = V + basis_at(i, 0, 1, cap);
    double acc = 0.0;
    for (int k = 0; k < m; ++k) acc += y[k] * Ve[64 * k];
    x[i] = acc;
}

// r = b - w
__global__ void __launch_bounds__(kBlock) k_sub(const double* __restrict__ b, const double* __restrict__ w,
                                                double* __restrict__ r, int64_t n) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) r[i] = b[i] - w[i];
}

// ---------------------------------------------- matrix-free operator (a18) --
// RansMatrix * x (ransMatrix.h:138-178, the RANS_MATRIX_FREE build): the
// operator calls each face's flux with two arguments, i.e. at cell values and
// zero gradients, with one step h = 1e-6 along the whole 4-vector of the
// perturbed side and no face length.  Per face it adds
// (F(q_L + h x_L, q_R) - F)/h to the owner row and, for two-sided faces,
// subtracts (F(q_L, q_R + h x_R) - F)/h from the neighbour row: every row sees
// only its own block of x.  Real rows start from x A / dt, ghost rows are x.

// F(q_L, q_R) per face at the current state (SoA Fb[k * nF + f])
__global__ void __launch_bounds__(kBlock) k_mf_base(CellsT<double> C, FacesT<double> F, const double* __restrict__ q,
                                                    GasT<double> g, int viscous, double* __restrict__ Fb) {
    int f = blockIdx.x * blockDim.x + threadIdx.x;
    if (f >= F.nF) return;
    const size_t nT = (size_t)C.nT, nF = (size_t)F.nF;
    const int o = F.c0[f], n = F.c1[f], kind = F.kind[f];
    double qL[4], qR[4], f0[4];
    const double z[4] = {0, 0, 0, 0};
    for (int k = 0; k < 4; ++k) { qL[k] = q[k * nT + o]; qR[k] = q[k * nT + n]; }
    face_flux<double>(g, kind, F.nx[f], F.ny[f], qL, qR, (viscous == 1) && (kind == K_INTERNAL), z, z, f0);
    for (int k = 0; k < 4; ++k) Fb[k * nF + f] = f0[k];
}

// one thread per cell; the cell's faces in reference face order, as the
// reference's edge loop reaches them
__global__ void __launch_bounds__(kBlock) k_mf_apply(CellsT<double> C, FacesT<double> F, const double* __restrict__ q,
                                                     const double* __restrict__ dt, const double* __restrict__ Fb,
                                                     GasT<double> g, int viscous, const double* __restrict__ x,
                                                     double* __restrict__ y, const int* __restrict__ active) {
    if (active && *active == 0) return;
    int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= C.nT) return;
    const size_t nT = (size_t)C.nT, nF = (size_t)F.nF;
    double xc[4];
    for (int k = 0; k < 4; ++k) xc[k] = x[k * nT + c];
    if (c >= C.nC) {
        for (int k = 0; k < 4; ++k) y[k * nT + c] = xc[k];
        return;
    }
    constexpr double h = 1e-6;
    const double z[4] = {0, 0, 0, 0};
    double acc[4], qc[4], qp[4], qo[4], fp[4];
    for (int k = 0; k < 4; ++k) {
        acc[k] = xc[k] * C.area[c] / dt[c];
        qc[k] = q[k * nT + c];
        qp[k] = qc[k] + h * xc[k];
    }
    for (int s = 0; s < 4; ++s) {
        uint32_t e = C.cface[(size_t)s * C.nC + c];
        if (e == 0xFFFFFFFFu) break;
        const int f = (int)(e & 0x7FFFFFFFu);
        const int kind = F.kind[f];
        const bool lam = (viscous == 1) && (kind == K_INTERNAL);
        if (e >> 31) {   // neighbour row of a two-sided face
            if (kind != K_INTERNAL) continue;
            const int o = F.c0[f];
            for (int k = 0; k < 4; ++k) qo[k] = q[k * nT + o];
            face_flux<double>(g, kind, F.nx[f], F.ny[f], qo, qp, lam, z, z, fp);
            for (int k = 0; k < 4; ++k) acc[k] -= (fp[k] - Fb[k * nF + f]) / h;
        } else {         // owner row
            const int n = F.c1[f];
            for (int k = 0; k < 4; ++k) qo[k] = q[k * nT + n];
            face_flux<double>(g, kind, F.nx[f], F.ny[f], qp, qo, lam, z, z, fp);
            for (int k = 0; k < 4; ++k) acc[k] += (fp[k] - Fb[k * nF + f]) / h;
        }
    }
    for (int k = 0; k < 4; ++k) y[k * nT + c] = acc[k];
}

// ---------------------------------------------------------------- launchers --
hipError_t launch_face_jacobian(hipStream_t s, CellsT<double> C, FacesT<double> F, const double* q, const double* gx,
                                const double* gy, GasT<double> g, int viscous, double* Jf) {
    hipLaunchKernelGGL(k_face_jacobian, dim3(xcd_grid(F.nF)), dim3(kBlock), 0, s, C, F, q, gx, gy, g, viscous, Jf);
    return hipGetLastError();
}
hipError_t launch_face_jacobian_sa(hipStream_t s, CellsT<double> C, FacesT<double> F, const double* q, const double* gx,
                                   const double* gy, GasT<double> g, double* Jf) {
    hipLaunchKernelGGL(k_face_jacobian_sa, dim3(xcd_grid(F.nF)), dim3(kBlock), 0, s, C, F, q, gx, gy, g, Jf);
    return hipGetLastError();
}
hipError_t launch_assemble_diag(hipStream_t s, int nv, CellsT<double> C, FacesT<double> F, const double* dt,
                                const double* Jf, SaSource src, double* D, double* Dinv, double* E, double* Ds,
                                int32_t* nbr, int* bad) {
    if (nv == 5)
        hipLaunchKernelGGL(k_assemble_diag<5>, dim3(xcd_grid(C.nC)), dim3(kBlock), 0, s, C, F, dt, Jf, src, D, Dinv, E,
                           Ds, nbr, bad);
    else if (nv == 4)
        hipLaunchKernelGGL(k_assemble_diag<4>, dim3(xcd_grid(C.nC)), dim3(kBlock), 0, s, C, F, dt, Jf, src, D, Dinv, E,
                           Ds, nbr, bad);
    else
        return hipErrorInvalidValue;
    return hipGetLastError();
}
hipError_t launch_lhs_apply(hipStream_t s, int nv, int32_t nC, int32_t nT, const double* Ds, const double* E,
                            const int32_t* nbr, const double* x, double* y, const int* active) {
    if (nv == 5)
        hipLaunchKernelGGL(k_lhs_apply<5>, dim3(xcd_grid(nT)), dim3(kBlock), 0, s, nC, nT, Ds, E, nbr, x, y, active);
    else if (nv == 4)
        hipLaunchKernelGGL(k_lhs_apply<4>, dim3(xcd_grid(nT)), dim3(kBlock), 0, s, nC, nT, Ds, E, nbr, x, y, active);
    else
        return hipErrorInvalidValue;
    return hipGetLastError();
}
hipError_t launch_block_jacobi(hipStream_t s, int nv, int32_t nC, int32_t nT, const double* Dinv, const double* x,
                               double* z, const int* active) {
    if (nv == 5)
        hipLaunchKernelGGL(k_block_jacobi<5>, dim3(nblocks(nT)), dim3(kBlock), 0, s, nC, nT, Dinv, x, z, active);
    else if (nv == 4)
        hipLaunchKernelGGL(k_block_jacobi<4>, dim3(nblocks(nT)), dim3(kBlock), 0, s, nC, nT, Dinv, x, z, active);
    else
        return hipErrorInvalidValue;
    return hipGetLastError();
}
template <int N>
static hipError_t dilu_setup_n(hipStream_t s, CellsT<double> C, FacesT<double> F, const ColourOrder& O, const double* D,
                               const double* Jf, double* Dti, const ColourMatrix& M, int* bad) {
    for (int c = 0; c < O.ncolours; ++c) {
        const int32_t n = O.off[c + 1] - O.off[c];
        if (n == 0) continue;
        hipLaunchKernelGGL(k_dilu_setup<N>, dim3(xcd_grid(n)), dim3(kBlock), 0, s, C, F, O.colour, c, O.cells, O.pos,
                           O.off[c], n, D, Jf, Dti, M.E, M.nbr, M.Dti, M.D, bad);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}
hipError_t launch_dilu_setup(hipStream_t s, int nv, CellsT<double> C, FacesT<double> F, const ColourOrder& O,
                             const double* D, const double* Jf, double* Dti, const ColourMatrix& M, int* bad) {
    if (nv == 5) return dilu_setup_n<5>(s, C, F, O, D, Jf, Dti, M, bad);
    if (nv == 4) return dilu_setup_n<4>(s, C, F, O, D, Jf, Dti, M, bad);
    return hipErrorInvalidValue;
}
namespace {
inline int row_grid(int32_t n) { return (((n + 63) / 64) + 7) & ~7; }
// one thread per row and cell below this many cells in the launch, one per
// cell from there on: at 8k cells (4x4) a backward sweep takes 4.0 us split and
// 4.9 whole, at 125k cells (5x5) 34 and 28; the product 142 and 92 at 500k
constexpr int32_t kSplitBelow = 32768;
inline bool split_rows(int32_t n) { return n < kSplitBelow; }
}
template <int N, int R, int SRC>
static void dilu_forward(hipStream_t s, int32_t nC, int32_t p0, int32_t n, const ColourMatrix& M, const double* in,
                         const double* a, double* V, int cap, int cols, const int* jend, const double* coef,
                         double* y, const int* active) {
    hipLaunchKernelGGL((k_dilu_forward<N, R, SRC>), dim3(row_grid(n)), dim3(64, N / R), 0, s, nC, p0, n, M.E, M.nbr,
                       M.Dti, in, a, V, cap, cols, jend, coef, y, active);
}
template <int N, int SRC>
static hipError_t dilu_sweeps(hipStream_t s, const ColourOrder& O, const ColourMatrix& M, const double* in,
                              const double* a, double* V, int cap, int cols, const int* jend, const double* coef,
                              double* y, const int* active) {
    const int32_t nC = O.off[O.ncolours];
    hipError_t e;
    for (int c = 0; c < O.ncolours; ++c) {
        const int32_t n = O.off[c + 1] - O.off[c];
        if (n == 0) continue;
        if (split_rows(n)) dilu_forward<N, 1, SRC>(s, nC, O.off[c], n, M, in, a, V, cap, cols, jend, coef, y, active);
        else dilu_forward<N, N, SRC>(s, nC, O.off[c], n, M, in, a, V, cap, cols, jend, coef, y, active);
        if ((e = hipGetLastError()) != hipSuccess) return e;
    }
    for (int c = O.ncolours - 2; c >= 0; --c) {
        const int32_t n = O.off[c + 1] - O.off[c];
        if (n == 0) continue;
        if (split_rows(n))
            hipLaunchKernelGGL((k_dilu_backward<N, 1>), dim3(row_grid(n)), dim3(64, N), 0, s, nC, O.off[c], n, M.E,
                               M.nbr, M.Dti, y, active);
        else
            hipLaunchKernelGGL((k_dilu_backward<N, N>), dim3(row_grid(n)), dim3(64), 0, s, nC, O.off[c], n, M.E, M.nbr,
                               M.Dti, y, active);
        if ((e = hipGetLastError()) != hipSuccess) return e;
    }
    return hipSuccess;
}
hipError_t launch_dilu_apply(hipStream_t s, int nv, const ColourOrder& O, const ColourMatrix& M, const double* in,
                             double* y) {
    if (nv == 5) return dilu_sweeps<5, 0>(s, O, M, in, nullptr, nullptr, 0, 0, nullptr, nullptr, y, nullptr);
    if (nv == 4) return dilu_sweeps<4, 0>(s, O, M, in, nullptr, nullptr, 0, 0, nullptr, nullptr, y, nullptr);
    return hipErrorInvalidValue;
}
hipError_t launch_dilu_apply_next(hipStream_t s, int nv, const ColourOrder& O, const ColourMatrix& M, const GmDev& G,
                                  const double* w, double* V, int cols, double* y) {
    if (nv == 5) return dilu_sweeps<5, 1>(s, O, M, w, G.hdr + 2, V, G.m + 1, cols, nullptr, G.h2, y, G.flags);
    if (nv == 4) return dilu_sweeps<4, 1>(s, O, M, w, G.hdr + 2, V, G.m + 1, cols, nullptr, G.h2, y, G.flags);
    return hipErrorInvalidValue;
}
hipError_t launch_dilu_apply_sum(hipStream_t s, int nv, const ColourOrder& O, const ColourMatrix& M, const GmDev& G,
                                 double* V, double* y) {
    if (nv == 5) return dilu_sweeps<5, 2>(s, O, M, nullptr, nullptr, V, G.m + 1, 0, G.flags + 3, G.y, y, nullptr);
    if (nv == 4) return dilu_sweeps<4, 2>(s, O, M, nullptr, nullptr, V, G.m + 1, 0, G.flags + 3, G.y, y, nullptr);
    return hipErrorInvalidValue;
}
namespace {
// the tiles of a vector's positions by colour (or as one stretch)
Span span_of(const int32_t* off, int ncolours) {
    Span S{};
    for (int c = 0; c < ncolours; ++c) {
        S.off[c] = off[c];
        S.per[c] = ((off[c + 1] - off[c] + 63) / 64 + 7) / 8;
        S.per_xcd += S.per[c];
    }
    S.off[ncolours] = off[ncolours];
    return S;
}
// blocks that take `group` tiles of the span each, at most kGsBlocks in turns,
// so that the next pass adds their sums up in passing
int span_grid(const Span& S, int group) { return 8 * std::min((S.per_xcd + group - 1) / group, kGsBlocks / 8); }
constexpr int kTiles = 4;   // tiles per block of whole cells (or of single rows)
}
template <int N>
static hipError_t colour_apply(hipStream_t s, const ColourOrder& O, const ColourMatrix& A, const double* x, double* y,
                               const double* V, int cap, int cols, double* partial, int* nblk, const int* active) {
    const int32_t nC = O.off[O.ncolours];
    if (nC <= 0) return hipSuccess;
    if (cols > kGsMax) return hipErrorInvalidValue;
    const Span S = span_of(O.off, O.ncolours);
    const bool split = split_rows(nC);
    const int grid = span_grid(S, split ? 1 : kTiles);
    if (nblk) *nblk = grid;
    auto product = split        ? (cols == 0 ? k_colour_apply<N, 1, 1, 0> : k_colour_apply<N, 1, 1, 1>)
                   : cols == 0  ? k_colour_apply<N, N, kTiles, 0>
                   : cols <= 8  ? k_colour_apply<N, N, kTiles, 8>
                   : cols <= 16 ? k_colour_apply<N, N, kTiles, 16>
                   : cols <= 24 ? k_colour_apply<N, N, kTiles, 24>
                                : k_colour_apply<N, N, kTiles, kGsMax>;
    hipLaunchKernelGGL(product, dim3(grid), dim3(64, split ? N : kTiles), 0, s, nC, S, A.D, A.E, A.nbr, x, y, V, cap,
                       cols, partial, active);
    return hipGetLastError();
}
hipError_t launch_colour_apply(hipStream_t s, int nv, const ColourOrder& O, const ColourMatrix& M, const double* x,
                               double* y) {
    if (nv == 5) return colour_apply<5>(s, O, M, x, y, nullptr, 0, 0, nullptr, nullptr, nullptr);
    if (nv == 4) return colour_apply<4>(s, O, M, x, y, nullptr, 0, 0, nullptr, nullptr, nullptr);
    return hipErrorInvalidValue;
}
hipError_t launch_colour_apply_dots(hipStream_t s, int nv, const ColourOrder& O, const ColourMatrix& M,
                                    const GmDev& G, const double* x, double* y, const double* V, int cols,
                                    int* nblk) {
    if (nv == 5) return colour_apply<5>(s, O, M, x, y, V, G.m + 1, cols, G.sums, nblk, G.flags);
    if (nv == 4) return colour_apply<4>(s, O, M, x, y, V, G.m + 1, cols, G.sums, nblk, G.flags);
    return hipErrorInvalidValue;
}
hipError_t launch_to_colour(hipStream_t s, int nv, int32_t nT, const ColourOrder& O, const double* b, const double* w,
                            double* out) {
    const int32_t nC = O.off[O.ncolours];
    if (nC <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_to_colour, dim3(xcd_grid(nC)), dim3(kBlock), 0, s, nC, nT, nv, O.cells, b, w, out);
    return hipGetLastError();
}
hipError_t launch_from_colour(hipStream_t s, int nv, int32_t nT, const ColourOrder& O, const double* y, const double* x,
                              double* z) {
    hipLaunchKernelGGL(k_from_colour, dim3(xcd_grid(nT)), dim3(kBlock), 0, s, O.off[O.ncolours], nT, nv, O.pos, y, x,
                       z);
    return hipGetLastError();
}
hipError_t launch_colour_update(hipStream_t s, int nv, int32_t nT, const ColourOrder& O, int first, double relax,
                                const double* z, double* x, double* dq, double* q, const int* converged) {
    const int32_t nC = O.off[O.ncolours];
    if (nC <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_colour_update, dim3(xcd_grid(nC)), dim3(kBlock), 0, s, nC, nT, nv, O.pos, first, relax, z, x,
                       dq, q, converged);
    return hipGetLastError();
}
// the variant of a pass with the fewest registers that holds m columns: the
// small bases of short restart cycles keep more waves in flight per SIMD
hipError_t launch_gs_dots(hipStream_t s, const GmDev& G, const double* V, int64_t n, int m, const double* w,
                          int* nblk) {
    if (m > kGsMax) return hipErrorInvalidValue;
    const int32_t off[2] = {0, (int32_t)n};
    const Span S = span_of(off, 1);
    *nblk = span_grid(S, kTiles);
    auto pass = m <= 8    ? k_gs_dots<1, kTiles, 8>
                : m <= 16 ? k_gs_dots<1, kTiles, 16>
                : m <= 24 ? k_gs_dots<1, kTiles, 24>
                          : k_gs_dots<1, kTiles, kGsMax>;
    hipLaunchKernelGGL(pass, dim3(*nblk), dim3(64, kTiles), 0, s, V, G.m + 1, (size_t)n, S, m, w, G.sums,
                       G.flags);
    return hipGetLastError();
}
template <int N>
static hipError_t gs_update_small(hipStream_t s, const GmDev& G, const Span& S, const double* V, size_t len, int m,
                                  double* w, int nblk1, double* sums2, int* nblk) {
    *nblk = span_grid(S, 1);
    hipLaunchKernelGGL(k_gs_update_small<N>, dim3(*nblk), dim3(64, N), 0, s, V, G.m + 1, len, S, m, G.sums, nblk1, w,
                       sums2, G.h1, G.flags);
    return hipGetLastError();
}
template <int N, int T>
static hipError_t gs_update(hipStream_t s, const GmDev& G, const Span& S, const double* V, size_t len, int m, double* w,
                            int nblk1, double* sums2, int* nblk) {
    *nblk = span_grid(S, T);
    auto pass = m <= 8    ? k_gs_update<N, T, 8>
                : m <= 16 ? k_gs_update<N, T, 16>
                : m <= 24 ? k_gs_update<N, T, 24>
                          : k_gs_update<N, T, kGsMax>;
    hipLaunchKernelGGL(pass, dim3(*nblk), dim3(64, N * T), 0, s, V, G.m + 1, len, S, m, G.sums, nblk1, w, sums2, G.h1,
                       G.flags);
    return hipGetLastError();
}
hipError_t launch_gm_step(hipStream_t s, const GmDev& G, const ColourOrder* O, int nv, const double* V, int64_t n, int j,
                          bool show, double* w, int nblk1) {
    const int m = j + 1;
    if (m > kGsMax) return hipErrorInvalidValue;
    double* sums2 = G.sums + (size_t)(kGsMax + 1) * kGsBlocks;
    int nblk = 0;
    hipError_t e;
    if (O) {
        const Span S = span_of(O->off, O->ncolours);
        const size_t len = (size_t)O->off[O->ncolours];
        if (nv != 4 && nv != 5) return hipErrorInvalidValue;
        if (split_rows((int32_t)len))
            e = nv == 5 ? gs_update_small<5>(s, G, S, V, len, m, w, nblk1, sums2, &nblk)
                        : gs_update_small<4>(s, G, S, V, len, m, w, nblk1, sums2, &nblk);
        else
            e = nv == 5 ? gs_update<5, 1>(s, G, S, V, len, m, w, nblk1, sums2, &nblk)
                        : gs_update<4, 1>(s, G, S, V, len, m, w, nblk1, sums2, &nblk);
    } else {
        const int32_t off[2] = {0, (int32_t)n};
        e = gs_update<1, kTiles>(s, G, span_of(off, 1), V, (size_t)n, m, w, nblk1, sums2, &nblk);
    }
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_gm_step, dim3(1), dim3(64 * kStepWaves), 0, s, G, j, show ? 1 : 0, sums2, nblk, V, O ? nv : 1,
                       O ? (int64_t)O->off[O->ncolours] : n, w);
    return hipGetLastError();
}
hipError_t launch_next_vector(hipStream_t s, const GmDev& G, const double* w, double* V, int cols, double* v,
                              int64_t n) {
    hipLaunchKernelGGL(k_next_vector, dim3(nblocks(n)), dim3(kBlock), 0, s, G.hdr + 2, G.h2, cols, w, V, G.m + 1, v, n,
                       G.flags);
    return hipGetLastError();
}
hipError_t launch_gm_begin(hipStream_t s, const GmDev& G, const double* r, int64_t n, int first) {
    const int nblk = (int)std::max<int64_t>(1, std::min<int64_t>((n + kBlock - 1) / kBlock, kGsBlocks));
    hipLaunchKernelGGL(k_gm_norm, dim3(nblk), dim3(kBlock), 0, s, r, n, G.sums);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_gm_begin, dim3(1), dim3(64), 0, s, G, first, G.sums, nblk);
    return hipGetLastError();
}
hipError_t launch_gm_solve(hipStream_t s, const GmDev& G) {
    hipLaunchKernelGGL(k_gm_solve, dim3(1), dim3(64), 0, s, G);
    return hipGetLastError();
}
hipError_t launch_lincomb(hipStream_t s, const GmDev& G, const double* V, double* x, int64_t n) {
    hipLaunchKernelGGL(k_lincomb_dev, dim3(nblocks(n)), dim3(kBlock), 0, s, V, G.m + 1, G.flags + 3, G.y, x, n);
    return hipGetLastError();
}
hipError_t launch_sub(hipStream_t s, const double* b, const double* w, double* r, int64_t n) {
    hipLaunchKernelGGL(k_sub, dim3(nblocks(n)), dim3(kBlock), 0, s, b, w, r, n);
    return hipGetLastError();
}
hipError_t launch_axpy(hipStream_t s, double a, const double* x, double* y, int64_t n) {
    hipLaunchKernelGGL(k_axpy, dim3(nblocks(n)), dim3(kBlock), 0, s, a, x, y, n);
    return hipGetLastError();
}

hipError_t launch_mf_base(hipStream_t s, CellsT<double> C, FacesT<double> F, const double* q, GasT<double> g,
                          int viscous, double* Fb) {
    hipLaunchKernelGGL(k_mf_base, dim3(nblocks(F.nF)), dim3(kBlock), 0, s, C, F, q, g, viscous, Fb);
    return hipGetLastError();
}
hipError_t launch_mf_apply(hipStream_t s, CellsT<double> C, FacesT<double> F, const double* q, const double* dt,
                           const double* Fb, GasT<double> g, int viscous, const double* x, double* y, const int* active) {
    hipLaunchKernelGGL(k_mf_apply, dim3(nblocks(C.nT)), dim3(kBlock), 0, s, C, F, q, dt, Fb, g, viscous, x, y, active);
    return hipGetLastError();
}

}  // namespace afx
