// Adjoint of the FP64 residual with respect to the state: lambda = (dR/dq)^T w
// for the inviscid and laminar residual of fillRhoRHS (solver.h:1079-1152)
// with Green-Gauss gradients (solver.h:428-469), the limiter of
// solver.h:517-593 and MUSCL reconstruction, first or second order.  The
// laminar terms (physics.h:230-258 at the face gradient of
// average_gradients, solver.h:359-398) add their adjoints in passes 2 and 3.
//
// Five atomics-free passes over the device layout (cells SoA q[k*nT+i]):
//   1 cells  gradients, limiters and the limiter's active branch (the face
//            that gives the minimum, the neighbour that gives q_max / q_min)
//   2 faces  reconstruction, adjoint of the Roe flux (hand-written reverse
//            sweep) and of the boundary states (forward-mode 4x4 Jacobian of
//            face_vars): adjoints of the reconstructed left/right states
//   3 cells  gather: direct state adjoint, gradient adjoint, limiter adjoint
//            (active branch; the part owed to the q_max/q_min neighbour is
//            kept for pass 5)
//   4 faces  transpose of the Green-Gauss face values
//   5 cells  gather of pass 4 and of the neighbours' limiter parts
// The wall/slip ghost states are copies of their owners that no flux reads;
// the farfield ghost states are boundary data and get no adjoint.
//
// With geometry on, passes 2-4 also accumulate the adjoints of the face and
// cell metrics the residual reads (normal, length, Green-Gauss weight,
// reconstruction offsets x_f - x_c, cell area), and three more passes carry
// them back to the node coordinates through the metric definitions of
// mesh.h:378-453, 744-787 and solver.h:436-444:
//   6 faces  face ends and the two centroids (normal, length, midpoint,
//            weight |x_f - x_0| / |x_0 - x_1|, ghost centroid x_f + |x_f - x_0| n)
//   7 cells  centroid (mean of the nodes) and area (two triangles) to vertices
//   8 nodes  gather over each node's face ends and cell vertices (CSR)
#include "afx_device.hpp"
#include "afx_adjoint.hpp"
#include "afx_adjoint_kernels.hpp"

namespace afx {

template <> __device__ __forceinline__ Dual1 ddiv<Dual1>(Dual1 a, Dual1 b) { return a / b; }
template <> __device__ __forceinline__ Dual1 dsqrt<Dual1>(Dual1 x) { return dual_sqrt(x); }
template <> __device__ __forceinline__ Dual1 dcbrt<Dual1>(Dual1 x) { return dual_cbrt(x); }

namespace {

__device__ __forceinline__ GasT<Dual1> dual_gas(const GasT<double>& g) {
    return GasT<Dual1>{Dual1(g.gamma), Dual1(g.R), Dual1(g.mu), Dual1(g.k), Dual1(g.cp), Dual1(g.PrL), Dual1(g.PrT)};
}

// component j of (d face_vars(kind, qL, qbc) / d qL)^T a  (qbc is boundary data)
__device__ __forceinline__ double face_vars_vjp(const GasT<double>& g, int kind, double nx, double ny, const double* qL,
                                                const double* qbc, const double* a, int j) {
    const GasT<Dual1> gd = dual_gas(g);
    Dual1 in[4], bc[4], out[4];
    for (int k = 0; k < 4; ++k) {
        in[k] = Dual1(qL[k], k == j ? 1.0 : 0.0);
        bc[k] = Dual1(qbc[k]);
    }
    face_vars<Dual1>(gd, kind, Dual1(nx), Dual1(ny), in, bc, out);
    double s = 0.0;
    for (int k = 0; k < 4; ++k) s += out[k].d * a[k];
    return s;
}

// component j of (d face_vars(kind, qL, qbc) / d qbc)^T a  (farfield boundary data)
__device__ __forceinline__ double face_vars_vjp_bc(const GasT<double>& g, int kind, double nx, double ny,
                                                   const double* qL, const double* qbc, const double* a, int j) {
    const GasT<Dual1> gd = dual_gas(g);
    Dual1 in[4], bc[4], out[4];
    for (int k = 0; k < 4; ++k) {
        in[k] = Dual1(qL[k]);
        bc[k] = Dual1(qbc[k], k == j ? 1.0 : 0.0);
    }
    face_vars<Dual1>(gd, kind, Dual1(nx), Dual1(ny), in, bc, out);
    double s = 0.0;
    for (int k = 0; k < 4; ++k) s += out[k].d * a[k];
    return s;
}

__device__ __forceinline__ double pick4(const double* v, int k) {
    return k == 0 ? v[0] : k == 1 ? v[1] : k == 2 ? v[2] : v[3];
}

// sum over the four lanes of a boundary face
__device__ __forceinline__ double quad_sum(double v) {
    v += __shfl_xor(v, 1);
    return v + __shfl_xor(v, 2);
}

// d face_vars(kind, qL, qbc; n) / d n_dir, dir 0 = x, 1 = y
__device__ __forceinline__ void face_vars_dn(const GasT<double>& g, int kind, double nx, double ny, const double* qL,
                                             const double* qbc, int dir, double* out_d) {
    const GasT<Dual1> gd = dual_gas(g);
    Dual1 a[4], bc[4], o[4];
    for (int k = 0; k < 4; ++k) { a[k] = Dual1(qL[k]); bc[k] = Dual1(qbc[k]); }
    face_vars<Dual1>(gd, kind, Dual1(nx, dir == 0 ? 1.0 : 0.0), Dual1(ny, dir == 1 ? 1.0 : 0.0), a, bc, o);
    for (int k = 0; k < 4; ++k) out_d[k] = o[k].d;
}

// bF . d roe(qL, qR(n), n) / d n_dir with qR = face_vars(qL, qbc; n) on boundary faces
__device__ __forceinline__ double roe_dn(const GasT<double>& g, int kind, double nx, double ny, const double* qL,
                                         const double* qR, const double* bF, int dir) {
    const GasT<Dual1> gd = dual_gas(g);
    const Dual1 nxd(nx, dir == 0 ? 1.0 : 0.0), nyd(ny, dir == 1 ? 1.0 : 0.0);
    Dual1 a[4], b[4], f[4];
    for (int k = 0; k < 4; ++k) a[k] = Dual1(qL[k]);
    if (kind == K_INTERNAL) {
        for (int k = 0; k < 4; ++k) b[k] = Dual1(qR[k]);
    } else {
        Dual1 bc[4];
        for (int k = 0; k < 4; ++k) bc[k] = Dual1(qR[k]);
        face_vars<Dual1>(gd, kind, nxd, nyd, a, bc, b);
    }
    roe_flux<Dual1>(gd, nxd, nyd, a, b, false, nullptr, nullptr, f);
    double s = 0.0;
    for (int k = 0; k < 4; ++k) s += bF[k] * f[k].d;
    return s;
}

// VJP of the laminar terms (viscous_terms, physics.h:230-258) of a face with
// respect to its reconstructed states and its face gradients: bL, bR +=
// (d F_v / d q)^T bF and bgx, bgy = (d F_v / d grad)^T bF, by sixteen
// forward-mode sweeps of the same device code
__device__ void viscous_vjp(const GasT<double>& g, double nx, double ny, const double* qL, const double* qR,
                            const double* gxa, const double* gya, const double* bF, double* bL, double* bR,
                            double* bgx, double* bgy) {
    const GasT<Dual1> gd = dual_gas(g);
    for (int j = 0; j < 16; ++j) {
        Dual1 a[4], b[4], gx[4], gy[4];
        for (int k = 0; k < 4; ++k) {
            a[k] = Dual1(qL[k], j == k ? 1.0 : 0.0);
            b[k] = Dual1(qR[k], j == 4 + k ? 1.0 : 0.0);
            gx[k] = Dual1(gxa[k], j == 8 + k ? 1.0 : 0.0);
            gy[k] = Dual1(gya[k], j == 12 + k ? 1.0 : 0.0);
        }
        Dual1 f1(0.0), f2(0.0), f3(0.0);
        viscous_terms<Dual1>(gd, Dual1(nx), Dual1(ny), a, b, gx, gy, gd.mu, gd.k, f1, f2, f3);
        const double v = bF[1] * f1.d + bF[2] * f2.d + bF[3] * f3.d;
        if (j < 4) bL[j] += v;
        else if (j < 8) bR[j - 4] += v;
        else if (j < 12) bgx[j - 8] = v;
        else bgy[j - 12] = v;
    }
}

// pass 1: gradients, limiters and the active branch of every (cell, variable),
// and in a reversed step the reverse of the stage's update.  Bound by the chain of
// dependent loads (slot word, face, cells), so the words and cells of all four
// slots are read first; the gradients of the step's start are formed with the
// first stage reversed and read by the others: 15 to 13 us a stage at 56k cells,
// with the update, which was a launch of 5 us.
__global__ void __launch_bounds__(kBlock)
k_adj_forward(CellsT<double> C, FacesT<double> F, const double* qg, const double* q, GasT<double> g, int second_order,
              double limiter_k, AdjBufs A, RevStage R) {
    const int c = xcd_index();
    if (c >= C.nC) return;
    const size_t nT = (size_t)C.nT, nC = (size_t)C.nC;
    if (R.g) {   // reverse of q_s+1 = q + W_s dt coef
        double sdt = 0.0;
        for (int k = 0; k < 4; ++k) {
            const size_t i = k * nT + c;
            const double gk = R.g[i];
            R.qbar[i] = R.first ? gk : R.qbar[i] + gk;
            R.wseed[i] = gk * R.dt[c] * R.coef / C.area[c];
            sdt += gk * R.W[i] * R.coef;
        }
        R.dtbar[c] = R.first ? sdt : R.dtbar[c] + sdt;
    }
    // gradients and limiters of one state (qg == q): the neighbour extrema
    // come from the values the gradient loop already holds
    const bool same = qg == q;
    double qc[4], sx[4] = {0, 0, 0, 0}, sy[4] = {0, 0, 0, 0};
    double mn[4], mx[4];
    int jmn[4] = {-1, -1, -1, -1}, jmx[4] = {-1, -1, -1, -1};
    for (int k = 0; k < 4; ++k) { qc[k] = q[k * nT + c]; mn[k] = qc[k]; mx[k] = qc[k]; }
    const bool have = R.g && !R.first;   // the gradients of the step's start, from its first reversed stage
    uint32_t es[4];
    int os[4], ns[4], ks[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) es[s] = C.cface[(size_t)s * nC + c];
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        const int f = es[s] == 0xFFFFFFFFu ? 0 : (int)(es[s] & 0x7FFFFFFFu);
        os[s] = F.c0[f];
        ns[s] = F.c1[f];
        ks[s] = F.kind[f];
    }
#pragma unroll 1
    for (int s = 0; s < 4 && !have; ++s) {
        const uint32_t e = es[s];
        if (e == 0xFFFFFFFFu) break;
        const int f = (int)(e & 0x7FFFFFFFu);
        const int o = os[s], n = ns[s], kind = ks[s];
        double qo[4], qn[4], qv[4];
        for (int k = 0; k < 4; ++k) { qo[k] = qg[k * nT + o]; qn[k] = qg[k * nT + n]; }
        face_vars<double>(g, kind, F.nx[f], F.ny[f], qo, qn, qv);
        const double gw = F.gw[f], L = F.len[f];
        for (int k = 0; k < 4; ++k) {
            const double fk = (qo[k] * (1.0 - gw) + qv[k] * gw) * L;
            if (e >> 31) { sx[k] -= fk * F.nx[f]; sy[k] -= fk * F.ny[f]; }
            else { sx[k] += fk * F.nx[f]; sy[k] += fk * F.ny[f]; }
        }
        if (same && second_order && kind != K_WALL && kind != K_SLIP) {   // wall ghost = owner copy
            const int other = (e >> 31) ? o : n;
            for (int k = 0; k < 4; ++k) {
                const double v = (e >> 31) ? qo[k] : qn[k];
                if (v < mn[k]) { mn[k] = v; jmn[k] = other; }
                if (mx[k] < v) { mx[k] = v; jmx[k] = other; }
            }
        }
    }
    const double Ar = C.area[c];
    double gx[4], gy[4];
    for (int k = 0; k < 4; ++k) {
        if (have) {
            gx[k] = A.gx[k * nT + c];
            gy[k] = A.gy[k * nT + c];
        } else {
            A.gx[k * nT + c] = gx[k] = sx[k] / Ar;
            A.gy[k * nT + c] = gy[k] = sy[k] / Ar;
        }
    }
    if (!second_order) return;
    if (!same || have)
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const uint32_t e = es[s];
            const int kind = ks[s];
            const int other = (e >> 31) ? os[s] : ns[s];
            double qv[4];
            for (int k = 0; k < 4; ++k) qv[k] = q[k * nT + other];
            if (e == 0xFFFFFFFFu || kind == K_WALL || kind == K_SLIP) continue;   // ghost = owner copy
            for (int k = 0; k < 4; ++k) {
                const double v = qv[k];
                if (v < mn[k]) { mn[k] = v; jmn[k] = other; }
                if (mx[k] < v) { mx[k] = v; jmx[k] = other; }
            }
        }
    const double Ka = limiter_k * sqrt(Ar), K3a = Ka * Ka * Ka;
    double lm[4] = {1, 1, 1, 1};
    int act[4] = {-1, -1, -1, -1};
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        const uint32_t e = es[s];
        if (e == 0xFFFFFFFFu) break;
        const int f = (int)(e & 0x7FFFFFFFu);
        const double dx = F.xf[f] - C.xc[c], dy = F.yf[f] - C.yc[c];
        for (int k = 0; k < 4; ++k) {
            const double dqg = gx[k] * dx + gy[k] * dy;
            const double l = limiter_phi<double>(dqg, mx[k] - qc[k], mn[k] - qc[k], K3a);
            if (l < lm[k]) { lm[k] = l; act[k] = s; }
        }
    }
    for (int k = 0; k < 4; ++k) {
        A.lim[k * nT + c] = lm[k];
        A.act[k * nC + c] = (int8_t)act[k];
        A.jmax[k * nC + c] = jmx[k];
        A.jmin[k * nC + c] = jmn[k];
    }
}

// The face passes take the interior faces (PART 1) a thread each and the boundary
// faces (PART 2), from the list A.bface, four lanes each, in one launch: blocks
// below `nbb` the boundary faces, the rest the interior ones in XCD-aware order.
// The lanes share a boundary face's forward-mode sweeps, a direction per lane.  A
// thread per boundary face in a launch of its own took 30 us for the 500 faces of
// a 56k-cell mesh (15 in pass 4) behind the 19 (10) of its 84k interior faces,
// where the joint launch takes 24 (11).  The joint kernel holds two waves per SIMD
// where the interior one holds three, yet is no slower at any size: the inviscid
// adjoint of 115k and 500k cells takes 69 and 217 us with it, 75 and 220 with
// launches apart.
constexpr int kBndLanes = 4;
inline int bnd_blocks(const AdjBufs& A) {   // a multiple of 8, so that the interior blocks keep their XCDs
    return (((kBndLanes * A.nbf + kBlock - 1) / kBlock) + 7) & ~7;
}

// pass 2: per face, adjoints of the reconstructed states.  LAM compiles the
// laminar terms in (interior faces of the laminar residual, A.vgx set); without
// them the inviscid instances need far fewer registers.
template <bool GEO, bool GHOST, int PART, bool LAM>
__device__ __forceinline__ void adj_face_body(const CellsT<double>& C, const FacesT<double>& F,
                                              const double* __restrict__ q, const double* __restrict__ w,
                                              const GasT<double>& g, int second_order, const AdjBufs& A,
                                              const GeoBufs& G, double* __restrict__ ghost, int i) {
    int f;
    const int lane = PART == 1 ? 0 : (int)(threadIdx.x & (kBndLanes - 1));
    if constexpr (PART == 1) {
        f = i;
        if (f >= F.nF || F.kind[f] != K_INTERNAL) return;
    } else {
        if (i / kBndLanes >= A.nbf) return;
        f = A.bface[i / kBndLanes];
    }
    const size_t nT = (size_t)C.nT, nF = (size_t)F.nF;
    const int o = F.c0[f], n = F.c1[f];
    const int kind = PART == 1 ? (int)K_INTERNAL : (int)F.kind[f];
    const double nx = F.nx[f], ny = F.ny[f], L = F.len[f];
    double qL[4], qR[4];
    for (int k = 0; k < 4; ++k) { qL[k] = q[k * nT + o]; qR[k] = q[k * nT + n]; }
    if (second_order) {
        const double d0x = F.xf[f] - C.xc[o], d0y = F.yf[f] - C.yc[o];
        for (int k = 0; k < 4; ++k)
            qL[k] += (A.gx[k * nT + o] * d0x + A.gy[k * nT + o] * d0y) * A.lim[k * nT + o];
        if (kind == K_INTERNAL) {
            const double d1x = F.xf[f] - C.xc[n], d1y = F.yf[f] - C.yc[n];
            for (int k = 0; k < 4; ++k)
                qR[k] += (A.gx[k * nT + n] * d1x + A.gy[k * nT + n] * d1y) * A.lim[k * nT + n];
        }
    }
    double bF[4], bL[4], bR[4];
    for (int k = 0; k < 4; ++k)
        bF[k] = kind == K_INTERNAL ? L * (w[k * nT + n] - w[k * nT + o]) : -L * w[k * nT + o];
    if (kind == K_INTERNAL) {
        roe_flux_vjp<double>(g.gamma, nx, ny, qL, qR, bF, bL, bR);
        if (LAM && A.vgx) {
            // laminar terms at the face gradient of average_gradients
            // (solver.h:359-398, A1): g = gbar - (gbar . t - dir) t with t the
            // normalised sum of the centroids and dir = (q_0 - q_1) / |x_0 + x_1|
            double t0 = C.xc[o] + C.xc[n], t1 = C.yc[o] + C.yc[n];
            const double l = sqrt(t0 * t0 + t1 * t1);
            t0 /= l;
            t1 /= l;
            double gxa[4], gya[4], bgx[4], bgy[4];
            for (int k = 0; k < 4; ++k) {
                const double dir = (q[k * nT + o] - q[k * nT + n]) / l;
                const double gxb = (A.gx[k * nT + o] + A.gx[k * nT + n]) * 0.5;
                const double gyb = (A.gy[k * nT + o] + A.gy[k * nT + n]) * 0.5;
                const double dot = gxb * t0 + gyb * t1;
                gxa[k] = gxb - (dot - dir) * t0;
                gya[k] = gyb - (dot - dir) * t1;
            }
            viscous_vjp(g, nx, ny, qL, qR, gxa, gya, bF, bL, bR, bgx, bgy);
            for (int k = 0; k < 4; ++k) {
                const double bt = bgx[k] * t0 + bgy[k] * t1;   // the adjoint of dir
                A.vgx[k * nF + f] = 0.5 * (bgx[k] - t0 * bt);
                A.vgy[k * nF + f] = 0.5 * (bgy[k] - t1 * bt);
                A.vdq[k * nF + f] = bt / l;
            }
        }
    } else {
        double qb[4], bB[4];
        face_vars<double>(g, kind, nx, ny, qL, qR, qb);
        roe_flux_vjp<double>(g.gamma, nx, ny, qL, qb, bF, bL, bB);
        bL[0] = pick4(bL, lane) + face_vars_vjp(g, kind, nx, ny, qL, qR, bB, lane);   // this lane's component
        if (GHOST && kind == K_FARFIELD) {   // the ghost's first adjoint write of this evaluation
            const double gb = face_vars_vjp_bc(g, kind, nx, ny, qL, qR, bB, lane);
            ghost[lane * nT + n] = A.add ? ghost[lane * nT + n] + gb : gb;
        }
    }
    if constexpr (PART == 1) {
        for (int k = 0; k < 4; ++k) {
            A.bL[k * nF + f] = bL[k];
            A.bR[k * nF + f] = bR[k];
        }
    } else {
        A.bL[lane * nF + f] = bL[0];
        A.bR[lane * nF + f] = 0.0;
    }
    if (!GEO) return;
    // metric adjoints of F(qL, qR; n) len: length, normal, reconstruction offsets
    auto put = [&](int plane, double v) {
        double* to = G.fbar + plane * nF + f;
        *to = G.add ? *to + v : v;
    };
    double fl[4], qRuse[4];
    if (kind == K_INTERNAL) {
        for (int k = 0; k < 4; ++k) qRuse[k] = qR[k];
    } else {
        face_vars<double>(g, kind, nx, ny, qL, qR, qRuse);
    }
    roe_flux<double>(g, nx, ny, qL, qRuse, false, nullptr, nullptr, fl);
    double lb = 0.0;
    for (int k = 0; k < 4; ++k) lb += (kind == K_INTERNAL ? w[k * nT + n] - w[k * nT + o] : -w[k * nT + o]) * fl[k];
    double d0b[2] = {0.0, 0.0}, d1b[2] = {0.0, 0.0};
    if constexpr (PART == 1) {
        const double nbx = roe_dn(g, kind, nx, ny, qL, qR, bF, 0), nby = roe_dn(g, kind, nx, ny, qL, qR, bF, 1);
        if (second_order)
            for (int k = 0; k < 4; ++k) {
                const double p0 = A.lim[k * nT + o] * bL[k], p1 = A.lim[k * nT + n] * bR[k];
                d0b[0] += p0 * A.gx[k * nT + o];
                d0b[1] += p0 * A.gy[k * nT + o];
                d1b[0] += p1 * A.gx[k * nT + n];
                d1b[1] += p1 * A.gy[k * nT + n];
            }
        put(0, nbx);
        put(1, nby);
        put(2, lb);
        put(3, 0.0);
        put(4, d0b[0]);
        put(5, d0b[1]);
        put(6, d1b[0]);
        put(7, d1b[1]);
    } else {
        const double nb = roe_dn(g, kind, nx, ny, qL, qR, bF, lane & 1);
        if (second_order) {
            const double p0 = A.lim[lane * nT + o] * bL[0];
            d0b[0] = quad_sum(p0 * A.gx[lane * nT + o]);
            d0b[1] = quad_sum(p0 * A.gy[lane * nT + o]);
        }
        if (lane < 2) {
            put(lane, nb);
            put(4 + lane, lane == 0 ? d0b[0] : d0b[1]);
        } else {
            put(lane, lane == 2 ? lb : 0.0);
            put(4 + lane, 0.0);
        }
    }
}

template <bool GEO, bool GHOST, bool LAM>
__global__ void __launch_bounds__(kBlock) k_adj_face(CellsT<double> C, FacesT<double> F, const double* __restrict__ q,
                                                     const double* __restrict__ w, GasT<double> g, int second_order,
                                                     AdjBufs A, GeoBufs G, double* __restrict__ ghost, int nbb) {
    const int b = (int)blockIdx.x;
    if (b < nbb)
        adj_face_body<GEO, GHOST, 2, false>(C, F, q, w, g, second_order, A, G, ghost, b * kBlock + (int)threadIdx.x);
    else
        adj_face_body<GEO, GHOST, 1, LAM>(C, F, q, w, g, second_order, A, G, ghost,
                                          xcd_tile(b - nbb, (int)gridDim.x - nbb) * kBlock + (int)threadIdx.x);
}

// pass 3: per cell, state / gradient / limiter adjoints
template <bool GEO, bool GHOST>
__global__ void __launch_bounds__(kBlock) k_adj_cell1(CellsT<double> C, FacesT<double> F, const double* __restrict__ q,
                                                      int second_order, double limiter_k, AdjBufs A,
                                                      double* __restrict__ lam, GeoBufs G,
                                                      double* __restrict__ ghost) {
    const int c = xcd_index();
    if (c >= C.nC) return;
    const size_t nT = (size_t)C.nT, nC = (size_t)C.nC, nF = (size_t)F.nF;
    double lq[4] = {0, 0, 0, 0}, lgx[4] = {0, 0, 0, 0}, lgy[4] = {0, 0, 0, 0}, lphi[4] = {0, 0, 0, 0};
    double gx[4], gy[4], ph[4];
    for (int k = 0; k < 4; ++k) { gx[k] = A.gx[k * nT + c]; gy[k] = A.gy[k * nT + c]; ph[k] = A.lim[k * nT + c]; }
    uint32_t es[4] = {0xFFFFFFFFu, 0xFFFFFFFFu, 0xFFFFFFFFu, 0xFFFFFFFFu};   // the slots' words and offsets, kept
    double dxs[4] = {0, 0, 0, 0}, dys[4] = {0, 0, 0, 0};                   // for the limiter's active slot
#pragma unroll
    for (int s = 0; s < 4; ++s) es[s] = C.cface[(size_t)s * nC + c];
#pragma unroll
    for (int s = 0; s < 4; ++s) {   // the offsets of all slots in one round trip
        const int f = es[s] == 0xFFFFFFFFu ? 0 : (int)(es[s] & 0x7FFFFFFFu);
        dxs[s] = F.xf[f] - C.xc[c];
        dys[s] = F.yf[f] - C.yc[c];
    }
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        const uint32_t e = es[s];
        if (e == 0xFFFFFFFFu) break;
        const int f = (int)(e & 0x7FFFFFFFu);
        const bool nb = (e >> 31) != 0;
        const double dx = dxs[s], dy = dys[s];
        for (int k = 0; k < 4; ++k) {
            const double b = nb ? A.bR[k * nF + f] : A.bL[k * nF + f];
            lq[k] += b;
            if (second_order) {
                lphi[k] += b * (gx[k] * dx + gy[k] * dy);
                lgx[k] += b * ph[k] * dx;
                lgy[k] += b * ph[k] * dy;
            }
        }
        if (A.vgx && F.kind[f] == K_INTERNAL)   // laminar terms: face gradient and difference quotient
            for (int k = 0; k < 4; ++k) {
                lgx[k] += A.vgx[k * nF + f];
                lgy[k] += A.vgy[k * nF + f];
                lq[k] += nb ? -A.vdq[k * nF + f] : A.vdq[k * nF + f];
            }
    }
    double abar = 0.0;
    for (int k = 0; k < 4; ++k) {
        double nbv = 0.0;
        int nbj = -1;
        const int s = second_order ? (int)A.act[k * nC + c] : -1;
        if (s >= 0) {
            const uint32_t e = s == 0 ? es[0] : s == 1 ? es[1] : s == 2 ? es[2] : es[3];
            const int f = (int)(e & 0x7FFFFFFFu);
            const double dx = s == 0 ? dxs[0] : s == 1 ? dxs[1] : s == 2 ? dxs[2] : dxs[3];
            const double dy = s == 0 ? dys[0] : s == 1 ? dys[1] : s == 2 ? dys[2] : dys[3];
            const double qc = q[k * nT + c];
            const double dqg = gx[k] * dx + gy[k] * dy;
            const int j = dqg > 1e-16 ? A.jmax[k * nC + c] : A.jmin[k * nC + c];
            const double D = (j >= 0 ? q[k * nT + j] : qc) - qc;
            const double Ka = limiter_k * sqrt(C.area[c]), K3a = Ka * Ka * Ka;
            double d_dqg, d_D, d_K = 0.0;
            (void)limiter_phi_d<double>(dqg, D, K3a, &d_dqg, &d_D, GEO ? &d_K : nullptr);
            lgx[k] += lphi[k] * d_dqg * dx;
            lgy[k] += lphi[k] * d_dqg * dy;
            if (GEO) {
                // K3a = (K sqrt(A))^3, and the offset of the limiting face
                abar += lphi[k] * d_K * 1.5 * K3a / C.area[c];
                const size_t side = (e >> 31) ? 6 : 4;
                G.fbar[side * nF + f] += lphi[k] * d_dqg * gx[k];
                G.fbar[(side + 1) * nF + f] += lphi[k] * d_dqg * gy[k];
            }
            if (j >= 0) {   // D = q_j - q_c (a limiter on q_c itself has D = 0 and no net dependence)
                lq[k] -= lphi[k] * d_D;
                if (j < C.nC) { nbv = lphi[k] * d_D; nbj = j; }
                else if (GHOST) ghost[k * nT + j] += lphi[k] * d_D;   // farfield ghost (its owner is this cell)
            }
        }
        lam[k * nT + c] = lq[k];
        A.lgx[k * nT + c] = A.add_lg ? A.lgx[k * nT + c] + lgx[k] : lgx[k];
        A.lgy[k * nT + c] = A.add_lg ? A.lgy[k * nT + c] + lgy[k] : lgy[k];
        A.nbv[k * nC + c] = nbv;
        A.nbj[k * nC + c] = nbj;
    }
    if (GEO) {
        // gradient = S / A
        if (second_order)
            for (int k = 0; k < 4; ++k) abar -= (lgx[k] * gx[k] + lgy[k] * gy[k]) / C.area[c];
        G.abar[c] = G.add ? G.abar[c] + abar : abar;
    }
}

// pass 4: transpose of the Green-Gauss face values
template <bool GEO, bool GHOST, int PART>
__device__ __forceinline__ void adj_face2_body(const CellsT<double>& C, const FacesT<double>& F,
                                               const double* __restrict__ q, const GasT<double>& g, const AdjBufs& A,
                                               const GeoBufs& G, double* __restrict__ ghost, int i) {
    int f;
    const int lane = PART == 1 ? 0 : (int)(threadIdx.x & (kBndLanes - 1));
    if constexpr (PART == 1) {
        f = i;
        if (f >= F.nF || F.kind[f] != K_INTERNAL) return;
    } else {
        if (i / kBndLanes >= A.nbf) return;
        f = A.bface[i / kBndLanes];
    }
    const size_t nT = (size_t)C.nT, nF = (size_t)F.nF;
    const int o = F.c0[f], n = F.c1[f];
    const int kind = PART == 1 ? (int)K_INTERNAL : (int)F.kind[f];
    const double nx = F.nx[f], ny = F.ny[f], L = F.len[f], gw = F.gw[f];
    constexpr bool two = PART == 1;
    double lfv[4];
    for (int k = 0; k < 4; ++k) {
        double v = (A.lgx[k * nT + o] * nx + A.lgy[k * nT + o] * ny) * L / C.area[o];
        if (two) v -= (A.lgx[k * nT + n] * nx + A.lgy[k * nT + n] * ny) * L / C.area[n];
        lfv[k] = v;
    }
    if constexpr (two) {   // face value q_o (1 - gw) + (q_o + q_n) gw / 2
        for (int k = 0; k < 4; ++k) {
            A.co[k * nF + f] = lfv[k] * (1.0 - 0.5 * gw);
            A.cn[k * nF + f] = lfv[k] * (0.5 * gw);
        }
    } else {     // q_o (1 - gw) + face_vars(q_o, q_ghost) gw
        double a[4], qo[4], qn[4];
        for (int k = 0; k < 4; ++k) {
            a[k] = lfv[k] * gw;
            qo[k] = q[k * nT + o];
            qn[k] = q[k * nT + n];
        }
        A.co[lane * nF + f] = pick4(lfv, lane) * (1.0 - gw) + face_vars_vjp(g, kind, nx, ny, qo, qn, a, lane);
        A.cn[lane * nF + f] = 0.0;
        if (GHOST && kind == K_FARFIELD) ghost[lane * nT + n] += face_vars_vjp_bc(g, kind, nx, ny, qo, qn, a, lane);
    }
    if (!GEO) return;
    // face value fv (as in pass 1) and the metric adjoints of fv n len / A
    double qo[4], qn[4], qv[4], fv[4];
    for (int k = 0; k < 4; ++k) { qo[k] = q[k * nT + o]; qn[k] = q[k * nT + n]; }
    face_vars<double>(g, kind, nx, ny, qo, qn, qv);
    for (int k = 0; k < 4; ++k) fv[k] = qo[k] * (1.0 - gw) + qv[k] * gw;
    const double Ao = C.area[o], An = two ? C.area[n] : 1.0;
    double nbx = 0.0, nby = 0.0, lb = 0.0, gb = 0.0;
    for (int k = 0; k < 4; ++k) {
        double ax = A.lgx[k * nT + o] / Ao, ay = A.lgy[k * nT + o] / Ao;
        if (two) { ax -= A.lgx[k * nT + n] / An; ay -= A.lgy[k * nT + n] / An; }
        nbx += fv[k] * L * ax;
        nby += fv[k] * L * ay;
        lb += fv[k] * (ax * nx + ay * ny);
        gb += lfv[k] * (qv[k] - qo[k]);
    }
    if constexpr (two) {
        G.fbar[0 * nF + f] += nbx;
        G.fbar[1 * nF + f] += nby;
        G.fbar[2 * nF + f] += lb;
        G.fbar[3 * nF + f] += gb;
    } else {
        double dv[4], nb = lane == 0 ? nbx : nby;
        face_vars_dn(g, kind, nx, ny, qo, qn, lane & 1, dv);
        for (int k = 0; k < 4; ++k) nb += lfv[k] * gw * dv[k];
        G.fbar[lane * nF + f] += lane < 2 ? nb : lane == 2 ? lb : gb;
    }
}

template <bool GEO, bool GHOST>
__global__ void __launch_bounds__(kBlock) k_adj_face2(CellsT<double> C, FacesT<double> F, const double* __restrict__ q,
                                                      GasT<double> g, AdjBufs A, GeoBufs G,
                                                      double* __restrict__ ghost, int nbb) {
    const int b = (int)blockIdx.x;
    if (b < nbb)
        adj_face2_body<GEO, GHOST, 2>(C, F, q, g, A, G, ghost, b * kBlock + (int)threadIdx.x);
    else
        adj_face2_body<GEO, GHOST, 1>(C, F, q, g, A, G, ghost,
                                      xcd_tile(b - nbb, (int)gridDim.x - nbb) * kBlock + (int)threadIdx.x);
}

// pass 6: face metrics -> face ends and centroids (mesh.h:378-453, 744-787;
// solver.h:436-444).  n = s (-dy, dx) / L with the sign s fixed by the mesh,
// L = |b - a|, x_f = (a + b) / 2, gw = |x_f - x_o| / |x_o - x_n| with x_n the
// ghost centroid x_f + |x_f - x_o| n on boundary faces.
__global__ void __launch_bounds__(kBlock) k_geo_face(CellsT<double> C, FacesT<double> F, GeoBufs G) {
    const int f = blockIdx.x * blockDim.x + threadIdx.x;
    if (f >= F.nF) return;
    const size_t nF = (size_t)F.nF;
    const int a = G.fnode[f], b = G.fnode[nF + f];
    const int o = F.c0[f], n = F.c1[f];
    const bool two = F.kind[f] == K_INTERNAL;
    const double xa = G.nodex[a], ya = G.nodey[a], xb = G.nodex[b], yb = G.nodey[b];
    const double dx = xb - xa, dy = yb - ya, L = sqrt(dx * dx + dy * dy);
    const double nx = F.nx[f], ny = F.ny[f];
    const double xf = 0.5 * (xa + xb), yf = 0.5 * (ya + yb);
    double nbx = G.fbar[0 * nF + f], nby = G.fbar[1 * nF + f], lb = G.fbar[2 * nF + f], gb = G.fbar[3 * nF + f];
    const double d0x = G.fbar[4 * nF + f], d0y = G.fbar[5 * nF + f], d1x = G.fbar[6 * nF + f], d1y = G.fbar[7 * nF + f];
    double xfb = d0x + d1x, yfb = d0y + d1y;
    double xob = -d0x, yob = -d0y, xnb = -d1x, ynb = -d1y;
    // Green-Gauss weight
    const double e1x = xf - C.xc[o], e1y = yf - C.yc[o], r1 = sqrt(e1x * e1x + e1y * e1y);
    const double e2x = C.xc[o] - C.xc[n], e2y = C.yc[o] - C.yc[n], r2 = sqrt(e2x * e2x + e2y * e2y);
    if (r1 > 0.0 && r2 > 0.0) {
        const double u1x = e1x / r1, u1y = e1y / r1, u2x = e2x / r2, u2y = e2y / r2;
        xfb += gb * u1x / r2;
        yfb += gb * u1y / r2;
        xob += gb * (-u1x / r2 - r1 / (r2 * r2) * u2x);
        yob += gb * (-u1y / r2 - r1 / (r2 * r2) * u2y);
        xnb += gb * (r1 / (r2 * r2) * u2x);
        ynb += gb * (r1 / (r2 * r2) * u2y);
        if (!two) {   // ghost centroid x_f + r1 n
            const double sg = nx * xnb + ny * ynb;
            xfb += xnb + sg * u1x;
            yfb += ynb + sg * u1y;
            xob -= sg * u1x;
            yob -= sg * u1y;
            nbx += r1 * xnb;
            nby += r1 * ynb;
            xnb = 0.0;
            ynb = 0.0;
        }
    }
    // normal and length -> edge vector (dx, dy)
    const double sgn = (nx * (-dy) + ny * dx) >= 0.0 ? 1.0 : -1.0;
    const double nn = nx * nbx + ny * nby;
    const double ubx = sgn * (nbx - nx * nn) / L, uby = sgn * (nby - ny * nn) / L;
    const double dxb = uby + lb * dx / L, dyb = -ubx + lb * dy / L;
    G.fend[0 * nF + f] = 0.5 * xfb - dxb;
    G.fend[1 * nF + f] = 0.5 * yfb - dyb;
    G.fend[2 * nF + f] = 0.5 * xfb + dxb;
    G.fend[3 * nF + f] = 0.5 * yfb + dyb;
    G.fcen[0 * nF + f] = xob;
    G.fcen[1 * nF + f] = yob;
    G.fcen[2 * nF + f] = xnb;
    G.fcen[3 * nF + f] = ynb;
}

// pass 7: centroid (node mean) and area (|triangle| sums) to cell vertices
__global__ void __launch_bounds__(kBlock) k_geo_cell(CellsT<double> C, FacesT<double> F, GeoBufs G) {
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= C.nC) return;
    const size_t nC = (size_t)C.nC, nF = (size_t)F.nF;
    double xcb = 0.0, ycb = 0.0;
    for (int s = 0; s < 4; ++s) {
        const uint32_t e = C.cface[(size_t)s * nC + c];
        if (e == 0xFFFFFFFFu) break;
        const size_t f = e & 0x7FFFFFFFu;
        const size_t side = (e >> 31) ? 2 : 0;
        xcb += G.fcen[side * nF + f];
        ycb += G.fcen[(side + 1) * nF + f];
    }
    int v[4];
    for (int s = 0; s < 4; ++s) v[s] = G.cnode[(size_t)s * nC + c];
    const int nv = v[3] < 0 ? 3 : 4;
    double bx[4] = {0, 0, 0, 0}, by[4] = {0, 0, 0, 0};
    for (int s = 0; s < nv; ++s) { bx[s] = xcb / nv; by[s] = ycb / nv; }
    const double Ab = G.abar[c];
    auto tri = [&](int i1, int i2, int i3) {
        const double x1 = G.nodex[v[i1]], y1 = G.nodey[v[i1]], x2 = G.nodex[v[i2]], y2 = G.nodey[v[i2]];
        const double x3 = G.nodex[v[i3]], y3 = G.nodey[v[i3]];
        const double S = x1 * (y2 - y3) + x2 * (y3 - y1) + x3 * (y1 - y2);
        const double h = 0.5 * Ab * (S >= 0.0 ? 1.0 : -1.0);
        bx[i1] += h * (y2 - y3); by[i1] += h * (x3 - x2);
        bx[i2] += h * (y3 - y1); by[i2] += h * (x1 - x3);
        bx[i3] += h * (y1 - y2); by[i3] += h * (x2 - x1);
    };
    tri(0, 1, 2);
    if (nv == 4) tri(0, 2, 3);
    for (int s = 0; s < 4; ++s) {
        G.cvert[(size_t)(2 * s) * nC + c] = bx[s];
        G.cvert[(size_t)(2 * s + 1) * nC + c] = by[s];
    }
}

// pass 8: per node, the sum over its face ends and cell vertices
__global__ void __launch_bounds__(kBlock) k_geo_node(CellsT<double> C, FacesT<double> F, GeoBufs G) {
    const int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= G.nN) return;
    const size_t nF = (size_t)F.nF, nC = (size_t)C.nC;
    double x = 0.0, y = 0.0;
    for (int i = G.n_off[v]; i < G.n_off[v + 1]; ++i) {
        const int e = G.n_ent[i];
        if (e >= 0) {
            const size_t f = (size_t)(e >> 1), end = (size_t)(e & 1);
            x += G.fend[(2 * end) * nF + f];
            y += G.fend[(2 * end + 1) * nF + f];
        } else {
            const int idx = -(e + 1);
            const size_t c = (size_t)(idx >> 2), slot = (size_t)(idx & 3);
            x += G.cvert[(2 * slot) * nC + c];
            y += G.cvert[(2 * slot + 1) * nC + c];
        }
    }
    G.xbar[2 * (size_t)v] = x;
    G.xbar[2 * (size_t)v + 1] = y;
}

// pass 5: gather of the Green-Gauss transpose (gg) and the neighbours' limiter
// parts.  lam gets the state part (pass 3 + neighbours' limiter parts), lam_g the
// Green-Gauss part (the gradient's source state); with lam_g == lam both add.  In
// a reversed step the state part is the next stage's seed (R.g), or with the
// step's last stage joins the Green-Gauss part in R.qbar.
__global__ void __launch_bounds__(kBlock) k_adj_cell2(CellsT<double> C, FacesT<double> F, AdjBufs A,
                                                      double* __restrict__ lam, double* lam_g, int gg, RevStage R) {
    const int c = xcd_index();
    if (c >= C.nC) return;
    const size_t nT = (size_t)C.nT, nC = (size_t)C.nC, nF = (size_t)F.nF;
    double acc[4], accg[4] = {0.0, 0.0, 0.0, 0.0};
    for (int k = 0; k < 4; ++k) acc[k] = lam[k * nT + c];
    // the four slots' words, then their neighbours, then those cells' limiting
    // neighbours: each in one round trip (slot by slot, 13 us at 56k cells)
    uint32_t e[4];
    int other[4], j[4][4];
#pragma unroll
    for (int s = 0; s < 4; ++s) e[s] = C.cface[(size_t)s * nC + c];
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        const int f = e[s] == 0xFFFFFFFFu ? 0 : (int)(e[s] & 0x7FFFFFFFu);
        other[s] = (e[s] >> 31) ? F.c0[f] : F.c1[f];
        if (e[s] == 0xFFFFFFFFu || other[s] >= C.nC) other[s] = -1;
    }
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int k = 0; k < 4; ++k) j[s][k] = A.nbj[k * nC + max(other[s], 0)];
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        if (gg && e[s] != 0xFFFFFFFFu) {
            const int f = (int)(e[s] & 0x7FFFFFFFu);
            const double* from = (e[s] >> 31) ? A.cn : A.co;
            for (int k = 0; k < 4; ++k) accg[k] += from[k * nF + f];
        }
#pragma unroll
        for (int k = 0; k < 4; ++k)
            if (other[s] >= 0 && j[s][k] == c) acc[k] += A.nbv[k * nC + other[s]];
    }
    for (int k = 0; k < 4; ++k) {
        const size_t i = k * nT + c;
        if (R.g) {
            if (R.last) R.qbar[i] += accg[k] + acc[k];
            else R.g[i] = acc[k];
        } else if (lam_g == lam) {
            lam[i] = acc[k] + accg[k];
        } else {
            lam[i] = acc[k];
            lam_g[i] = accg[k];
        }
    }
}

}  // namespace

namespace {

// spectral radius sqrt(gamma p / rho) + |V| of one state on a face and its
// gradient with respect to the state (k_dt, solver.h:308-356)
__device__ inline double eig_and_grad(const GasT<double>& g, double nx, double ny, const double* qc, double* d) {
    const double gm1 = g.gamma - 1.0;
    const double r = qc[0], ru = qc[1], rv = qc[2], re = qc[3];
    const double V = (ru * nx + rv * ny) / r;
    const double p = gm1 * (re - 0.5 / r * (ru * ru + rv * rv));
    const double a = sqrt(p * g.gamma / r);
    const double dp[4] = {gm1 * 0.5 * (ru * ru + rv * rv) / (r * r), -gm1 * ru / r, -gm1 * rv / r, gm1};
    const double sv = V < 0.0 ? -1.0 : 1.0;
    const double dV[4] = {-V / r, nx / r, ny / r, 0.0};
    for (int k = 0; k < 4; ++k) {
        const double da = g.gamma / (2.0 * a) * (dp[k] / r - (k == 0 ? p / (r * r) : 0.0));
        d[k] = da + sv * dV[k];
    }
    return a + (V < 0.0 ? -V : V);
}

// ebar_f = len_f (sbar_o + sbar_n), sbar_c = d dt_c / d s_c dtbar_c = -dtbar_c dt_c^2 / (cfl A_c)
__global__ void __launch_bounds__(kBlock) k_dt_bar_face(CellsT<double> C, FacesT<double> F,
                                                        const double* __restrict__ dt, const double* __restrict__ dtbar,
                                                        double cfl, double* __restrict__ ebar) {
    const int f = blockIdx.x * blockDim.x + threadIdx.x;
    if (f >= F.nF) return;
    const int o = F.c0[f], n = F.c1[f];
    double e = -dtbar[o] * dt[o] * dt[o] / (cfl * C.area[o]);
    if (F.kind[f] == K_INTERNAL) e += -dtbar[n] * dt[n] * dt[n] / (cfl * C.area[n]);
    ebar[f] = e * F.len[f];
}

// per cell: the faces on which this cell's state gives max(eig_o, eig_n)
__global__ void __launch_bounds__(kBlock) k_dt_bar_cell(CellsT<double> C, FacesT<double> F, const double* __restrict__ q,
                                                        GasT<double> g, const double* __restrict__ ebar,
                                                        const double* __restrict__ qbar, double* __restrict__ out) {
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= C.nC) return;
    const size_t nT = (size_t)C.nT, nC = (size_t)C.nC;
    double acc[4] = {0.0, 0.0, 0.0, 0.0};
    uint32_t es[4];
    int os[4], ns[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) es[s] = C.cface[(size_t)s * nC + c];
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        const int f = es[s] == 0xFFFFFFFFu ? 0 : (int)(es[s] & 0x7FFFFFFFu);
        os[s] = F.c0[f];
        ns[s] = F.c1[f];
    }
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        if (es[s] == 0xFFFFFFFFu) break;
        const int f = (int)(es[s] & 0x7FFFFFFFu);
        const int o = os[s], n = ns[s];
        const double nx = F.nx[f], ny = F.ny[f];
        double qo[4], d[4];
        for (int k = 0; k < 4; ++k) qo[k] = q[k * nT + o];
        const double eo = eig_and_grad(g, nx, ny, qo, d);
        int active = o;
        if (F.kind[f] == K_INTERNAL) {
            double qn[4], dn[4];
            for (int k = 0; k < 4; ++k) qn[k] = q[k * nT + n];
            const double en = eig_and_grad(g, nx, ny, qn, dn);
            if (eo < en) { active = n; for (int k = 0; k < 4; ++k) d[k] = dn[k]; }
        }
        if (active != c) continue;
        for (int k = 0; k < 4; ++k) acc[k] += ebar[f] * d[k];
    }
    for (int k = 0; k < 4; ++k) out[k * nT + c] = qbar[k * nT + c] + acc[k];
}

// metric part of the local time step's VJP: dt_c = cfl A_c / S_c with
// S_c = sum_f lambda_f len_f and lambda_f = max over the face's sides of
// c + |u n_x + v n_y| (the owner only on boundary faces).  With
// sbar_c = -dtbar_c dt_c^2 / (cfl A_c): lenbar_f += lambda_f (sbar_o + sbar_n),
// (nbar_x, nbar_y)_f += len_f (sbar_o + sbar_n) sign(V) (u, v) of the active
// side.  (The area term dtbar dt / A cancels the residual's division by the
// area in the stage update, so neither is added.)
__global__ void __launch_bounds__(kBlock) k_dt_bar_geo(CellsT<double> C, FacesT<double> F, const double* __restrict__ q,
                                                       GasT<double> g, const double* __restrict__ dt,
                                                       const double* __restrict__ dtbar, double cfl,
                                                       double* __restrict__ facc) {
    const int f = blockIdx.x * blockDim.x + threadIdx.x;
    if (f >= F.nF) return;
    const size_t nT = (size_t)C.nT, nF = (size_t)F.nF;
    const int o = F.c0[f], n = F.c1[f];
    const double nx = F.nx[f], ny = F.ny[f];
    double sb = -dtbar[o] * dt[o] * dt[o] / (cfl * C.area[o]);
    double qa[4], d[4];
    for (int k = 0; k < 4; ++k) qa[k] = q[k * nT + o];
    double lam = eig_and_grad(g, nx, ny, qa, d);
    if (F.kind[f] == K_INTERNAL) {
        sb += -dtbar[n] * dt[n] * dt[n] / (cfl * C.area[n]);
        double qn[4];
        for (int k = 0; k < 4; ++k) qn[k] = q[k * nT + n];
        const double en = eig_and_grad(g, nx, ny, qn, d);
        if (lam < en) { lam = en; for (int k = 0; k < 4; ++k) qa[k] = qn[k]; }
    }
    const double u = qa[1] / qa[0], v = qa[2] / qa[0];
    const double sv = (u * nx + v * ny) < 0.0 ? -1.0 : 1.0;
    const double e = F.len[f] * sb;
    facc[0 * nF + f] += e * sv * u;
    facc[1 * nF + f] += e * sv * v;
    facc[2 * nF + f] += lam * sb;
}

// acc[k][j] += ghost[k*nT + cell_j] over the farfield ghost cells
__global__ void __launch_bounds__(kBlock) k_ghost_acc(const double* __restrict__ ghost, const int32_t* __restrict__ cells,
                                                      int32_t n, int32_t nT, double* __restrict__ acc) {
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= n) return;
    for (int k = 0; k < 4; ++k) acc[(size_t)k * n + j] += ghost[(size_t)k * nT + cells[j]];
}

}  // namespace

hipError_t launch_dt_vjp_geo(hipStream_t s, CellsT<double> C, FacesT<double> F, const double* q, GasT<double> g,
                             const double* dt, const double* dtbar, double cfl, double* facc) {
    hipLaunchKernelGGL(k_dt_bar_geo, dim3((F.nF + kBlock - 1) / kBlock), dim3(kBlock), 0, s, C, F, q, g, dt, dtbar,
                       cfl, facc);
    return hipGetLastError();
}

hipError_t launch_geo_to_nodes(hipStream_t s, CellsT<double> C, FacesT<double> F, const GeoBufs& G) {
    hipLaunchKernelGGL(k_geo_face, dim3((F.nF + kBlock - 1) / kBlock), dim3(kBlock), 0, s, C, F, G);
    hipLaunchKernelGGL(k_geo_cell, dim3((C.nC + kBlock - 1) / kBlock), dim3(kBlock), 0, s, C, F, G);
    hipLaunchKernelGGL(k_geo_node, dim3((G.nN + kBlock - 1) / kBlock), dim3(kBlock), 0, s, C, F, G);
    return hipGetLastError();
}

hipError_t launch_ghost_acc(hipStream_t s, const double* ghost, const int32_t* cells, int32_t n, int32_t nT,
                            double* acc) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_ghost_acc, dim3((n + kBlock - 1) / kBlock), dim3(kBlock), 0, s, ghost, cells, n, nT, acc);
    return hipGetLastError();
}

hipError_t launch_dt_vjp(hipStream_t s, CellsT<double> C, FacesT<double> F, const double* q, GasT<double> g,
                         const double* dt, const double* dtbar, double cfl, double* ebar, const double* qbar,
                         double* out) {
    hipLaunchKernelGGL(k_dt_bar_face, dim3((F.nF + kBlock - 1) / kBlock), dim3(kBlock), 0, s, C, F, dt, dtbar, cfl,
                       ebar);
    hipLaunchKernelGGL(k_dt_bar_cell, dim3((C.nC + kBlock - 1) / kBlock), dim3(kBlock), 0, s, C, F, q, g, ebar, qbar, out);
    return hipGetLastError();
}

namespace {
// R.g null: the adjoint of one residual; otherwise one stage of a reversed step,
// whose Green-Gauss transpose (linear in the gradient adjoints, and of the
// step's start in every stage) is applied once, to the sum over the stages
template <bool GEO, bool GHOST>
void adjoint_passes(hipStream_t s, CellsT<double> C, FacesT<double> F, const double* qg, const double* q,
                    const double* w, GasT<double> g, int second_order, double limiter_k, AdjBufs A, double* lam,
                    double* lam_g, double* ghost, const GeoBufs& G, const RevStage& R = RevStage{}) {
    // the pass kernels index cells and interior faces in XCD-aware block order
    const int nbc = xcd_grid(C.nC), nbf = xcd_grid(F.nF), nbb = bnd_blocks(A);
    const bool gradients = second_order || A.vgx;   // they enter the residual (reconstruction or laminar terms)
    const bool gg = gradients && (!R.g || R.last);
    hipLaunchKernelGGL(k_adj_forward, dim3(nbc), dim3(kBlock), 0, s, C, F, qg, q, g, second_order, limiter_k, A, R);
    if (A.vgx)
        hipLaunchKernelGGL((k_adj_face<GEO, GHOST, true>), dim3(nbb + nbf), dim3(kBlock), 0, s, C, F, q, w, g,
                           second_order, A, G, ghost, nbb);
    else
        hipLaunchKernelGGL((k_adj_face<GEO, GHOST, false>), dim3(nbb + nbf), dim3(kBlock), 0, s, C, F, q, w, g,
                           second_order, A, G, ghost, nbb);
    hipLaunchKernelGGL((k_adj_cell1<GEO, GHOST>), dim3(nbc), dim3(kBlock), 0, s, C, F, q, second_order, limiter_k, A,
                       lam, G, ghost);
    if (gg)
        hipLaunchKernelGGL((k_adj_face2<GEO, GHOST>), dim3(nbb + nbf), dim3(kBlock), 0, s, C, F, qg, g, A, G, ghost, nbb);
    if (gradients || R.g)
        hipLaunchKernelGGL(k_adj_cell2, dim3(nbc), dim3(kBlock), 0, s, C, F, A, lam, lam_g, gg ? 1 : 0, R);
    if (GEO && !R.g) {
        hipLaunchKernelGGL(k_geo_face, dim3(nbf), dim3(kBlock), 0, s, C, F, G);
        hipLaunchKernelGGL(k_geo_cell, dim3(nbc), dim3(kBlock), 0, s, C, F, G);
        hipLaunchKernelGGL(k_geo_node, dim3((G.nN + kBlock - 1) / kBlock), dim3(kBlock), 0, s, C, F, G);
    }
}
}  // namespace

hipError_t launch_reverse_stage(hipStream_t s, CellsT<double> C, FacesT<double> F, const double* qg, const double* q,
                                GasT<double> g, int second_order, double limiter_k, AdjBufs A, double* lam,
                                const RevStage& R, double* ghost, const GeoBufs* Gp) {
    if (!ghost == !Gp) return hipErrorInvalidValue;   // the boundary data's adjoints or the metrics'
    A.add = 1;
    A.add_lg = R.first ? 0 : 1;
    GeoBufs G = Gp ? *Gp : GeoBufs{};
    G.add = 1;
    if (Gp) adjoint_passes<true, false>(s, C, F, qg, q, R.wseed, g, second_order, limiter_k, A, lam, lam, nullptr, G, R);
    else adjoint_passes<false, true>(s, C, F, qg, q, R.wseed, g, second_order, limiter_k, A, lam, lam, ghost, G, R);
    return hipGetLastError();
}

hipError_t launch_adjoint_state(hipStream_t s, CellsT<double> C, FacesT<double> F, const double* q, const double* w,
                                GasT<double> g, int second_order, double limiter_k, AdjBufs A, double* lam,
                                const GeoBufs* Gp) {
    if (Gp) adjoint_passes<true, false>(s, C, F, q, q, w, g, second_order, limiter_k, A, lam, lam, nullptr, *Gp);
    else adjoint_passes<false, false>(s, C, F, q, q, w, g, second_order, limiter_k, A, lam, lam, nullptr, GeoBufs{});
    return hipGetLastError();
}

// ------------------------------------------------------------------ tangent --
// Tangent of the FP64 residual: the fused tile kernel k_residual_tile
// instantiated with Dual1, so R and (dR/dq) v come out of the same operations
// as the plain residual (gradients, limiter on its active branch, Roe, laminar
// and Spalart-Allmaras terms, cell sums).  The value parts reproduce the FP64
// residual bit for bit; the derivative parts are the exact directional
// derivative of the piecewise-smooth residual.
namespace {
__global__ void __launch_bounds__(kBlock) k_to_dual(const double* __restrict__ x, int64_t n, Dual1* __restrict__ out) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = Dual1(x[i]);
}
// q + eps v over nv planes of nT cells; ghost cells (i >= nC) keep a zero
// derivative: their states are boundary data
__global__ void __launch_bounds__(kBlock) k_dual_state(const double* __restrict__ q, const double* __restrict__ v,
                                                       int32_t nT, int32_t nC, int nv, Dual1* __restrict__ out) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (int64_t)nv * nT) return;
    const int32_t c = (int32_t)(i % nT);
    out[i] = Dual1(q[i], c < nC ? v[i] : 0.0);
}
__global__ void __launch_bounds__(kBlock) k_dual_parts(const Dual1* __restrict__ x, int64_t n, double* __restrict__ val,
                                                       double* __restrict__ der) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    if (val) val[i] = x[i].v;
    der[i] = x[i].d;
}
inline unsigned nblk(int64_t n) { return (unsigned)((n + kBlock - 1) / kBlock); }
}  // namespace

hipError_t launch_to_dual(hipStream_t s, const double* x, int64_t n, Dual1* out) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_to_dual, dim3(nblk(n)), dim3(kBlock), 0, s, x, n, out);
    return hipGetLastError();
}
hipError_t launch_dual_state(hipStream_t s, const double* q, const double* v, int32_t nT, int32_t nC, int nv,
                             Dual1* out) {
    hipLaunchKernelGGL(k_dual_state, dim3(nblk((int64_t)nv * nT)), dim3(kBlock), 0, s, q, v, nT, nC, nv, out);
    return hipGetLastError();
}
hipError_t launch_dual_parts(hipStream_t s, const Dual1* x, int64_t n, double* val, double* der) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_dual_parts, dim3(nblk(n)), dim3(kBlock), 0, s, x, n, val, der);
    return hipGetLastError();
}
size_t tile_lds_bytes_tangent(int32_t lmax, int32_t gmax, int32_t ftmax, int nv) {
    return tile_lds_bytes<Dual1>(lmax, gmax, ftmax, nv);
}
hipError_t launch_residual_tile_tangent(hipStream_t s, TilesT<Dual1> S, const Dual1* q, int32_t nT, int32_t nC,
                                        const Dual1* area, const Dual1* lsq, const Dual1* xc, const Dual1* yc,
                                        const Dual1* wd, GasT<double> g64, int gg, int so, double limiter_k,
                                        int viscous, Dual1* R) {
    const int nb = ((S.ntiles + 7) / 8) * 8;
    const GasT<Dual1> g{Dual1(g64.gamma), Dual1(g64.R), Dual1(g64.mu), Dual1(g64.k), Dual1(g64.cp), Dual1(g64.PrL),
                        Dual1(g64.PrT)};
    const int nv = viscous == 2 ? 5 : 4;
    const size_t lds = tile_lds_bytes<Dual1>(S.lmax, S.gmax, S.ftmax, nv);
    hipError_t e;
    // the state array is also the ghost array: the kernel refreshes the
    // wall/slip ghosts of its tiles from their owners (set_walls_from_internal)
    Dual1* qg = const_cast<Dual1*>(q);
    if (nv == 5) {
        if ((e = hipFuncSetAttribute(reinterpret_cast<const void*>(&k_residual_tile<Dual1, 5>),
                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds)) != hipSuccess)
            return e;
        hipLaunchKernelGGL((k_residual_tile<Dual1, 5>), dim3(nb), dim3(kBlock), lds, s, S, q, nT, nC, area, lsq, xc,
                           yc, wd, g, gg, so, Dual1(limiter_k), viscous, R, qg);
    } else {
        if ((e = hipFuncSetAttribute(reinterpret_cast<const void*>(&k_residual_tile<Dual1, 4>),
                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds)) != hipSuccess)
            return e;
        hipLaunchKernelGGL((k_residual_tile<Dual1, 4>), dim3(nb), dim3(kBlock), lds, s, S, q, nT, nC, area, lsq, xc,
                           yc, wd, g, gg, so, Dual1(limiter_k), viscous, R, qg);
    }
    return hipGetLastError();
}

}  // namespace afx
