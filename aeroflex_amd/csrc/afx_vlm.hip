// Vortex-lattice aerodynamic influence matrix and its dense solve on MI355X
// (include/afx_vlm.h).
//
// Device side of the coupling path of AeroFLEX's src/vlm:
//   - panel geometry, collocation points, right-hand side and wake rings
//     (panel.cpp:46-128, surface.cpp:35-58, solver.cpp:256-290);
//   - the FP64 influence matrix, one thread per matrix entry, four Biot-Savart
//     segments per ring (potential.cpp:36-58, solver.cpp:139-254);
//   - FP32 LU with partial pivoting: a cooperative panel kernel (rows of the
//     panel in LDS, pivot keys exchanged between workgroups), row
//     interchanges with a wavefront triangular solve for the block row, and the
//     trailing update as a hand-written FP32 GEMM on the matrix cores
//     (k_gemm_sub_f32, v_mfma_f32_32x32x2f32);
//   - FP64 iterative refinement on the FP64 matrix with the FP32 factor as
//     the preconditioner (replaces Eigen's BiCGSTAB, solver.cpp:41-50);
//   - Kutta-Joukowski ring forces (surface.cpp:164-201).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <cmath>
#include <cstring>
#include <exception>
#include <string>
#include <vector>

#include "../../include/afx_vlm.h"
#include "afx_exchange.hpp"
#include "afx_vlm.hpp"

using afx::api_fail;

namespace {

// (the error is read, or the next call's launch check would report it again)
int hip_fail(const char* what, hipError_t e) {
    (void)hipGetLastError();
    return api_fail(AFX_EHIP, std::string(what) + ": " + hipGetErrorString(e));
}
#define VCHK(x)                                              \
    do {                                                     \
        hipError_t e_ = (x);                                 \
        if (e_ != hipSuccess) return hip_fail(#x, e_);       \
    } while (0)

constexpr int LU_NB = 128;          // panel width = trailing-update depth = solve block
constexpr int PANEL_R = 256;        // panel rows per workgroup held in LDS (256 x 128 FP32 = 128 of 160 KiB)
constexpr int MAX_PANEL_WG = 240;   // one to a compute unit, -> n <= 61440
constexpr int SUB = 16;             // columns of a sub-panel
constexpr int KEY_STRIDE = 256;     // words of a key buffer: MAX_PANEL_WG in whole wavefronts
constexpr unsigned SPIN_LIMIT = 1u << 21;
constexpr double FOUR_PI = 12.566370614359172;

// ------------------------------------------------- panel pivot exchange --
// Candidate of one workgroup for one column as one ordered key: |a| bits (31) |
// 0x1ffff - row (17) | sequence (16), so the largest key is the largest |a| and,
// among equals, the lowest row.  The sequence is the 1-based column of the whole
// matrix: a key left from an earlier column (or an earlier factorisation: the
// words are cleared before each one) never matches.  Row 0x1ffff: no candidate.
constexpr unsigned NO_ROW = 0x1ffffu;
__device__ inline unsigned long long make_key(float absval, unsigned row, unsigned seq) {
    const unsigned long long ab = (unsigned long long)(__float_as_uint(absval) & 0x7fffffffu);
    return (ab << 33) | ((unsigned long long)(NO_ROW - row) << 16) | (unsigned long long)(seq & 0xffffu);
}
__device__ inline int key_row(unsigned long long k) { return (int)(NO_ROW - ((unsigned)(k >> 16) & NO_ROW)); }

// maximum of a 32-bit unsigned over the wavefront's 64 lanes, through DPP lane
// moves: pairs and quads (quad_perm), half rows and rows (mirrors), then rows 1
// and 3 from lane 15 of the row below (row_bcast15) and rows 2 and 3 from lane 31
// (row_bcast31); lane 63 then holds it
template <int CTRL, int ROW_MASK>
__device__ inline unsigned dpp_max_step(unsigned k) {
    return max(k, (unsigned)__builtin_amdgcn_update_dpp((int)k, (int)k, CTRL, ROW_MASK, 0xF, false));
}
__device__ inline unsigned wave_max(unsigned k) {
    k = dpp_max_step<0xB1, 0xF>(k);    // quad_perm [1,0,3,2]
    k = dpp_max_step<0x4E, 0xF>(k);    // quad_perm [2,3,0,1]
    k = dpp_max_step<0x141, 0xF>(k);   // row_half_mirror
    k = dpp_max_step<0x140, 0xF>(k);   // row_mirror
    k = dpp_max_step<0x142, 0xA>(k);   // row_bcast15
    k = dpp_max_step<0x143, 0xC>(k);   // row_bcast31
    return (unsigned)__builtin_amdgcn_readlane((int)k, 63);
}
// the lane holding the largest (hi, lo), 0 <= lo; -1 where every hi is zero.
// The low words are compared only among lanes that share the largest high word.
__device__ inline int wave_winner(unsigned hi, unsigned lo) {
    const unsigned top = wave_max(hi);
    unsigned long long who = __ballot(hi == top);
    if (__builtin_expect((who & (who - 1ull)) != 0ull, 0)) {
        if (top == 0u) return -1;
        const unsigned low = hi == top ? lo : 0u;
        const unsigned most = wave_max(low);
        who = __ballot(hi == top && low == most);
    }
    return __ffsll(who) - 1;
}

// --------------------------------------------------- panel factorisation --
// LU with partial pivoting of the m x nbc panel whose top-left entry is
// A(j0, j0) (column-major, leading dimension lda).  Workgroup w holds the panel
// rows [w R, w R + R) of all nbc columns in LDS, one row per thread, and no row
// moves before the end: a thread knows its row's position, which the
// interchanges change, and writes it there.
//
// The panel advances in sub-panels of SUB columns, whose entries a thread keeps
// in registers (the current column in a[0]).  Per column every wave leaves its
// candidate (key and SUB values) in LDS; wave 0 posts the workgroup's best as
// value | sequence words and its key, polls the keys of all workgroups and then
// reads the winner's values: no counter and no fence, since each word carries its
// sequence.  Only one wave polls: with all four, and every candidate's values in
// the same round trip, the requests to those few lines took longer than the
// second trip (690 us a panel of 16 384 rows).  Meanwhile the owner of the last
// pivot row publishes the rest of it (L to the left inside the sub-panel, the
// columns to the right as they stand).  After SUB columns every workgroup reads
// those rows, solves for their U (the substitution is repeated in every
// workgroup: a column per thread) and updates its own rows of the remaining
// columns, four rows per lane and a quarter of the columns per wave.  Every
// element takes the operations of the plain right-looking order.
//
// Words alternate between two buffers, so posting for column j + 1 cannot
// overwrite what a slower workgroup still reads for column j: it cannot post
// j + 2 before every workgroup has posted j + 1, which each does only after
// reading column j's words; the published rows alternate by sub-panel alike.
// With one workgroup (m <= R) nothing is exchanged.  Every wait is bounded: a
// wave that polls longer than spin_limit raises `abort` and every workgroup
// returns.  What is queued behind the panel then runs on an unfinished one:
// src and dst of rows that were not placed keep an earlier panel's values, all
// of them rows of the panel, so every access stays inside the matrix, and the
// host refuses the factor.
//
// Bound by the latency of that exchange (a word takes about 0.55 us from one
// compute unit to another) and, with one workgroup, by the column's chain of
// maximum, LDS exchange, division and update.  Keys go to a mailbox of each
// reader: one row of keys polled by all cost 1.1 us more a column at 64
// workgroups.  A panel of 256, 2 048 and 16 384 rows takes 133, 320 and 352 us
// alone; with a row's 128 columns exchanged and updated per column, 120 rows to a
// workgroup, it took 520, 554 and 554.
__device__ inline unsigned long long tagged(unsigned seq, float v) {
    return ((unsigned long long)seq << 32) | (unsigned long long)__float_as_uint(v);
}
// wait (bounded) for a value | sequence word of this sequence; false on timeout
__device__ inline bool wait_tagged(const unsigned long long* p, unsigned seq, unsigned limit, float& v) {
    unsigned spins = 0;
    unsigned long long w;
    while (((w = __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) >> 32) != seq) {
        if (++spins > limit) { v = 0.f; return false; }
        __builtin_amdgcn_s_sleep(1);
    }
    v = __uint_as_float((unsigned)(w & 0xFFFFFFFFull));
    return true;
}

__global__ __launch_bounds__(256, 1) void k_panel_lu(float* __restrict__ A, int lda, int m, int nbc, int j0,
                                                     int* __restrict__ ipiv, int* __restrict__ src,
                                                     int* __restrict__ dst, unsigned long long* keys,
                                                     unsigned long long* vals, unsigned long long* prow,
                                                     unsigned* abort_flag, unsigned spin_limit,
                                                     int* __restrict__ info) {
    __shared__ float4 slab4[LU_NB * PANEL_R / 4];     // panel column c at slab[c * PANEL_R]
    __shared__ float4 U4[(LU_NB - SUB) * SUB / 4];    // U of the sub-panel's rows, column by column
    __shared__ float4 Ls4[SUB * SUB / 4];             // L of the sub-panel's rows
    __shared__ float4 cand4[2][4][SUB / 4];           // the waves' candidates
    __shared__ float4 urow4[2][SUB / 4];              // the pivot row
    __shared__ unsigned long long wk[2][4], s_win[2];
    __shared__ int lrow[SUB];                         // the sub-panel's pivot rows in this workgroup
    __shared__ int s_fail;
    float* slab = reinterpret_cast<float*>(slab4);
    float* Ls = reinterpret_cast<float*>(Ls4);
    const int t = threadIdx.x, lane = t & 63, w = blockIdx.x, nwg = gridDim.x;
    const int wv = __builtin_amdgcn_readfirstlane(t >> 6);
    const int rbase = w * PANEL_R;
    const int rows = min(PANEL_R, m - rbase);
    float* P = A + (size_t)j0 * lda + j0;

    {
        const float* mine = P + rbase + min(t, rows - 1);
#pragma unroll 1
        for (int c = 0; c < LU_NB; c += 32) {
            float v[32];
#pragma unroll
            for (int i = 0; i < 32; ++i) v[i] = mine[(size_t)min(c + i, nbc - 1) * lda];
#pragma unroll
            for (int i = 0; i < 32; ++i) slab[(c + i) * PANEL_R + t] = (t < rows && c + i < nbc) ? v[i] : 0.f;
        }
    }
    if (t == 0) s_fail = 0;
    __syncthreads();
    int pos = t < rows ? rbase + t : -1;   // the row's position in the panel, -1: none

    for (int c0 = 0;; c0 += SUB) {
        const int sw = min(SUB, nbc - c0), sub = (c0 / SUB) & 1;
        unsigned long long* rest = prow + (size_t)sub * SUB * LU_NB;
        auto publish = [&](int jj, int i) {   // row jj of the sub-panel, from its first column on
            if (i >= 0 && i < nbc - c0)
                __hip_atomic_store(&rest[jj * LU_NB + i],
                                   tagged((unsigned)(j0 + c0 + jj + 1), slab[(c0 + i) * PANEL_R + lrow[jj]]),
                                   __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        };
        float a[SUB];   // (columns past the last are zero in the slab)
#pragma unroll
        for (int i = 0; i < SUB; ++i) a[i] = slab[(c0 + i) * PANEL_R + t];
        bool won = false;
        for (int jj = 0; jj < sw; ++jj) {
            const int j = c0 + jj, par = j & 1;
            const unsigned seq = (unsigned)(j0 + j + 1);
            // the wave's candidate: largest |a|, a NaN taken as the largest
            // number; rows already chosen offer none
            const float fa = fabsf(a[0]);
            const unsigned mag = __float_as_uint(fa == fa ? fa : INFINITY);
            const int best = wave_winner(pos >= j ? mag + 1u : 0u, NO_ROW - (unsigned)pos);
            if (lane == max(best, 0)) {
                wk[par][wv] = best < 0 ? 0ull : make_key(__uint_as_float(mag), (unsigned)pos, seq);
#pragma unroll
                for (int i = 0; i < SUB / 4; ++i)
                    cand4[par][wv][i] = make_float4(a[4 * i], a[4 * i + 1], a[4 * i + 2], a[4 * i + 3]);
            }
            __syncthreads();
            const unsigned long long k0 = wk[par][0], k1 = wk[par][1], k2 = wk[par][2], k3 = wk[par][3];
            const unsigned long long k01 = k0 > k1 ? k0 : k1, k23 = k2 > k3 ? k2 : k3;
            const int m01 = k0 > k1 ? 0 : 1, m23 = k2 > k3 ? 2 : 3;
            const unsigned long long mine = k01 > k23 ? k01 : k23;
            const int mw = k01 > k23 ? m01 : m23;
            unsigned long long win = mine;
            const float4* ur = cand4[par][mw];
            int fail = 0;
            if (nwg > 1) {
                if (wv == 0) {
                    unsigned long long* kbox = keys + par * KEY_STRIDE;   // reader q's at 2 q KEY_STRIDE
                    unsigned long long* vbox = vals + par * SUB;          // workgroup q's at 2 q SUB
                    const unsigned long long post = mine != 0ull ? mine : make_key(0.f, NO_ROW, seq);
                    for (int q = lane; q < nwg; q += 64)
                        __hip_atomic_store(&kbox[2 * q * KEY_STRIDE + w], post, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    kbox += 2 * w * KEY_STRIDE;
                    if (lane < SUB)
                        __hip_atomic_store(&vbox[2 * w * SUB + lane], tagged(seq, reinterpret_cast<const float*>(ur)[lane]),
                                           __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    constexpr int SLOTS = KEY_STRIDE / 64;
                    unsigned long long kk = 0ull;
                    int kq = 0;
                    unsigned spins = 0;
                    bool late = false;
                    for (;;) {
                        bool ok = true;
                        kk = 0ull;
#pragma unroll
                        for (int sl = 0; sl < SLOTS; ++sl) {
                            if (sl * 64 >= nwg) break;
                            const int q = sl * 64 + lane;   // (past nwg: words of earlier, taller panels)
                            unsigned long long k =
                                __hip_atomic_load(&kbox[q], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                            ok = ok && (q >= nwg || (unsigned)(k & 0xffffu) == (seq & 0xffffu));
                            k = q < nwg ? k : 0ull;
                            kq = k > kk ? q : kq;
                            kk = k > kk ? k : kk;
                        }
                        if (__all(ok)) break;
                        if (++spins > spin_limit ||
                            ((spins & 63u) == 0u &&
                             __hip_atomic_load(abort_flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0u)) {
                            late = true;
                            break;
                        }
                    }
                    if (!late) {
                        // (every key ends in the sequence: the high words
                        // hold |a| and the top of the row, never all zero
                        // while a live row is left)
                        const int wl = max(0, wave_winner((unsigned)(kk >> 32), (unsigned)kk));
                        const int wq = __builtin_amdgcn_readlane(kq, wl);
                        const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)kk, wl);
                        const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(kk >> 32), wl);
                        float f = 0.f;
                        if (lane < SUB) late = !wait_tagged(&vbox[2 * wq * SUB + lane], seq, spin_limit, f);
                        if (lane < SUB) reinterpret_cast<float*>(urow4[par])[lane] = f;
                        if (lane == 0) s_win[par] = ((unsigned long long)hi << 32) | lo;
                    }
                    if (__any(late)) {
                        if (lane == 0) {
                            s_fail = 1;
                            __hip_atomic_store(abort_flag, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                        }
                    }
                } else if (won) {
                    publish(jj - 1, t - 64);
                }
                __syncthreads();
                win = s_win[par];
                ur = urow4[par];
                fail = s_fail;
            }
            float u[SUB];
#pragma unroll
            for (int i = 0; i < SUB / 4; ++i) {
                const float4 v = ur[i];
                u[4 * i] = v.x; u[4 * i + 1] = v.y; u[4 * i + 2] = v.z; u[4 * i + 3] = v.w;
            }
            if (fail) return;
            won = win == mine;
            const int p = key_row(win);   // panel-relative pivot position, >= j
            if (won && pos == p) {
                lrow[jj] = t;
                ipiv[j0 + j] = j0 + p;
            }
            pos = pos == j ? p : pos == p ? j : pos;
            const bool upd = __builtin_amdgcn_readfirstlane((int)(__float_as_uint(u[0]) << 1)) != 0;
            if (__builtin_expect(upd, 1)) {
                if (pos > j) {
                    const float l = a[0] / u[0];
                    slab[j * PANEL_R + t] = l;
#pragma unroll
                    for (int i = 0; i + 1 < SUB; ++i) a[i] = a[i + 1] - l * u[i + 1];
                    a[SUB - 1] = 0.f;
                }
            } else {   // a zero pivot leaves the column, whose entries are all zero, alone
                if (w == 0 && t == 0 && *info == 0) *info = j0 + j + 1;
                if (pos > j) {
                    slab[j * PANEL_R + t] = a[0];
#pragma unroll
                    for (int i = 0; i + 1 < SUB; ++i) a[i] = a[i + 1];
                    a[SUB - 1] = 0.f;
                }
            }
        }
        const int rem = nbc - c0 - SUB;
        __syncthreads();   // lrow and L of the last columns
        if (nwg > 1 && rem > 0 && won) publish(SUB - 1, t);
        if (pos >= c0 && pos < c0 + sw) {   // the sub-panel's part of U, as the row stood when it was chosen
            const int k = pos - c0;
#pragma unroll
            for (int i = 0; i < SUB; ++i)
                if (k + i < sw) slab[(pos + i) * PANEL_R + t] = a[i];
        }
        if (rem <= 0) break;
        // the pivot rows: L of the sub-panel, and the columns right of it
        float v[SUB];
        bool ok = true;
        {
            const int k = t / SUB, i = t % SUB;
            float l = 0.f;
            if (i < k) {
                if (nwg == 1) l = slab[(c0 + i) * PANEL_R + lrow[k]];
                else ok = wait_tagged(&rest[k * LU_NB + i], (unsigned)(j0 + c0 + k + 1), spin_limit, l);
            }
            Ls[t] = l;
        }
        if (t < rem) {
            if (nwg == 1) {
#pragma unroll
                for (int k = 0; k < SUB; ++k) v[k] = slab[(c0 + SUB + t) * PANEL_R + lrow[k]];
            } else {
                unsigned long long x[SUB];   // all at once; the last few may not be there yet
#pragma unroll
                for (int k = 0; k < SUB; ++k)
                    x[k] = __hip_atomic_load(&rest[k * LU_NB + SUB + t], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
                for (int k = 0; k < SUB; ++k) {
                    const unsigned seq = (unsigned)(j0 + c0 + k + 1);
                    v[k] = __uint_as_float((unsigned)x[k]);
                    if ((unsigned)(x[k] >> 32) != seq)
                        ok = wait_tagged(&rest[k * LU_NB + SUB + t], seq, spin_limit, v[k]) && ok;
                }
            }
        }
        if (!ok) {
            s_fail = 1;
            __hip_atomic_store(abort_flag, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        __syncthreads();
        if (s_fail) return;
        if (t < rem) {
#pragma unroll
            for (int k = 1; k < SUB; ++k)
#pragma unroll
                for (int i = 0; i < k; ++i) v[k] -= Ls[k * SUB + i] * v[i];
#pragma unroll
            for (int k = 0; k < SUB / 4; ++k) {
                const float4 x = make_float4(v[4 * k], v[4 * k + 1], v[4 * k + 2], v[4 * k + 3]);
                U4[t * (SUB / 4) + k] = x;
                // every workgroup has read its rows of A by now
                if (w == 0) *reinterpret_cast<float4*>(P + (size_t)(c0 + SUB + t) * lda + c0 + 4 * k) = x;
            }
        }
        __syncthreads();
        // rows that are pivots by now take part: what becomes of their remaining
        // entries is not read again
        {
            float4 l[SUB];
#pragma unroll
            for (int k = 0; k < SUB; ++k) l[k] = slab4[(c0 + k) * (PANEL_R / 4) + lane];
#pragma unroll 4
            for (int c = wv; c < rem; c += 4) {
                float4 x = slab4[(c0 + SUB + c) * (PANEL_R / 4) + lane];
                float uc[SUB];
#pragma unroll
                for (int k = 0; k < SUB / 4; ++k) {
                    const float4 y = U4[c * (SUB / 4) + k];
                    uc[4 * k] = y.x; uc[4 * k + 1] = y.y; uc[4 * k + 2] = y.z; uc[4 * k + 3] = y.w;
                }
#pragma unroll
                for (int k = 0; k < SUB; ++k) {
                    x.x -= l[k].x * uc[k];
                    x.y -= l[k].y * uc[k];
                    x.z -= l[k].z * uc[k];
                    x.w -= l[k].w * uc[k];
                }
                slab4[(c0 + SUB + c) * (PANEL_R / 4) + lane] = x;
            }
        }
        __syncthreads();
    }
    // a pivot row's columns right of its sub-panel were written as U above
    if (pos >= 0) {
        const int end = pos < nbc ? min(nbc, (pos / SUB + 1) * SUB) : nbc;
#pragma unroll 1
        for (int c = 0; c < LU_NB; c += SUB) {
            float v[SUB];
#pragma unroll
            for (int i = 0; i < SUB; ++i) v[i] = slab[(c + i) * PANEL_R + t];
#pragma unroll
            for (int i = 0; i < SUB; ++i)
                if (c + i < end) P[(size_t)(c + i) * lda + pos] = v[i];
        }
        // the interchanges as a whole: which row each of the panel's first nbc
        // positions takes, and where the rows that were there go
        if (pos < nbc) src[j0 + pos] = rbase + t;
        if (rbase + t < nbc) dst[j0 + rbase + t] = pos;
    }
}

__device__ inline float readlane_f(float v, int lane) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}

// The row interchanges of the panel [j0, j0 + nbc) applied to the columns
// [cbeg, cend), and with SOLVE (nbc = 128) the block row solved at once:
// A(j0:j0+128, cbeg:cend) <- L11^-1 of it, L11 unit lower.  A wavefront takes CPW
// columns, two of the panel's rows per lane: it gathers the rows that come to the
// top, solves, and stores them and the rows that they displace (all reads of a
// column precede its writes, and the column belongs to this wave).  The columns'
// substitution chains are independent, so CPW of them hide the latency of each
// step (readlane of x_k after its last update); two are enough where the
// columns are few and every wave runs at once.  Without SOLVE `extra` is one more
// column (the permutation, as bits).  Interchanges column by column in their own
// kernel, a chain of 128 dependent loads, took 9 to 110 us a panel, and the
// solve with its L11 staged by single words 45.
template <int CPW, bool SOLVE>
__global__ __launch_bounds__(256) void k_swap_solve(float* __restrict__ A, int lda, int cbeg, int cend, int j0,
                                                    int nbc, const int* __restrict__ src,
                                                    const int* __restrict__ dst, float* __restrict__ extra) {
    __shared__ float4 Ls4[SOLVE ? LU_NB * LU_NB / 4 : 1];   // column k at Ls[k * LU_NB], zero on and above the diagonal
    const float* Ls = reinterpret_cast<const float*>(Ls4);
    const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
    if (SOLVE) {
#pragma unroll
        for (int q = 0; q < LU_NB * LU_NB / 4 / 256; ++q) {
            const int idx = q * 256 + t, k = idx / (LU_NB / 4), r = (idx % (LU_NB / 4)) * 4;
            float4 v = *reinterpret_cast<const float4*>(A + (size_t)(j0 + k) * lda + j0 + r);
            v.x = r > k ? v.x : 0.f;
            v.y = r + 1 > k ? v.y : 0.f;
            v.z = r + 2 > k ? v.z : 0.f;
            v.w = r + 3 > k ? v.w : 0.f;
            Ls4[idx] = v;
        }
        __syncthreads();
    }
    const int c0 = cbeg + (blockIdx.x * 4 + wv) * CPW, ncol = cend + (extra ? 1 : 0) - c0;
    if (ncol <= 0) return;
    const bool in0 = lane < nbc, in1 = lane + 64 < nbc;
    const int s0 = in0 ? src[j0 + lane] : 0, s1 = in1 ? src[j0 + lane + 64] : 0;
    const int d0 = in0 ? dst[j0 + lane] : 0, d1 = in1 ? dst[j0 + lane + 64] : 0;
    float b0[CPW], b1[CPW], o0[CPW], o1[CPW];
#pragma unroll
    for (int q = 0; q < CPW; ++q) {
        const float* cp = c0 + q < cend ? A + (size_t)(c0 + q) * lda + j0 : extra + j0;
        const bool live = q < ncol;
        b0[q] = live && in0 ? cp[s0] : 0.f;
        b1[q] = live && in1 ? cp[s1] : 0.f;
        o0[q] = live && d0 >= nbc ? cp[lane] : 0.f;
        o1[q] = live && d1 >= nbc ? cp[lane + 64] : 0.f;
    }
    if (SOLVE) {
#pragma unroll 2
        for (int k = 0; k < 64; ++k) {
            const float l0 = Ls[k * LU_NB + lane], l1 = Ls[k * LU_NB + lane + 64];
#pragma unroll
            for (int q = 0; q < CPW; ++q) {
                const float xk = readlane_f(b0[q], k);
                b0[q] -= l0 * xk;
                b1[q] -= l1 * xk;
            }
        }
#pragma unroll 2
        for (int k = 64; k < LU_NB; ++k) {
            const float l1 = Ls[k * LU_NB + lane + 64];
#pragma unroll
            for (int q = 0; q < CPW; ++q) b1[q] -= l1 * readlane_f(b1[q], k - 64);
        }
    }
#pragma unroll
    for (int q = 0; q < CPW; ++q) {
        if (q >= ncol) break;
        float* cp = c0 + q < cend ? A + (size_t)(c0 + q) * lda + j0 : extra + j0;
        if (in0 && (SOLVE || s0 != lane)) cp[lane] = b0[q];
        if (in1 && (SOLVE || s1 != lane + 64)) cp[lane + 64] = b1[q];
        if (d0 >= nbc) cp[d0] = o0[q];
        if (d1 >= nbc) cp[d1] = o1[q];
    }
}

// FP64 row-major -> FP32 column-major (the factor's working copy)
__global__ __launch_bounds__(256) void k_to_cm32(const double* __restrict__ A64, int n, float* __restrict__ A32,
                                                 int lda) {
    __shared__ float tile[64][65];
    const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
    const int i0 = blockIdx.y * 64, j0 = blockIdx.x * 64;
    for (int k = ty; k < 64; k += 4) {
        const int i = i0 + k, j = j0 + tx;
        tile[k][tx] = (i < n && j < n) ? (float)A64[(size_t)i * n + j] : 0.f;
    }
    __syncthreads();
    for (int k = ty; k < 64; k += 4) {
        const int j = j0 + k, i = i0 + tx;
        if (i < n && j < n) A32[(size_t)j * lda + i] = tile[tx][k];
    }
}

// ------------------------------------------------- triangular solves ----
// State of a refined solve, kept on the device so that its steps can be queued
// without waiting for each: the kernels of a step return at once when done.
struct SolveState {
    double anorm, prev, contraction, backward;
    int it, converged, done;
    unsigned aborted;
};

// Inverses of the 128 x 128 diagonal blocks of the factor, unit lower L
// (blockIdx.y = 0) and upper U (1, as the lower U^T), blocks past n padded with
// the identity; the triangular solves apply these with a matrix-vector product
// instead of a 128-step substitution.  One workgroup per block, in LDS: the eight
// 16 x 16 diagonal blocks by substitution, a column per thread, then doubled:
// the inverse of [A 0; C B] has -B^-1 (C A^-1) below the diagonal, two products
// in which each of the 256 threads forms S / 16 rows of four columns.  Column by
// column with two barriers each it took 190 us for L and 350 us for U.
constexpr int INV_LD = LU_NB + 4;
template <int S>
__device__ inline void inv_double(float (*X)[INV_LD], float* W, int t) {
    constexpr int TR = S / 16;
    const int p = t / (4 * S), q = t % (4 * S), cg = (q % (S / 4)) * 4, rg = (q / (S / 4)) * TR;
    const int o = 2 * S * p;
    float* Wp = W + p * S * S;
    float s[TR][4];
    auto product = [&](auto left, auto right) {
#pragma unroll
        for (int i = 0; i < TR; ++i)
#pragma unroll
            for (int c = 0; c < 4; ++c) s[i][c] = 0.f;
#pragma unroll 4
        for (int k = 0; k < S; ++k) {
            const float4 m = *reinterpret_cast<const float4*>(right(k));
#pragma unroll
            for (int i = 0; i < TR; ++i) {
                const float l = left(rg + i, k);
                s[i][0] += l * m.x;
                s[i][1] += l * m.y;
                s[i][2] += l * m.z;
                s[i][3] += l * m.w;
            }
        }
    };
    product([&](int r, int k) { return X[o + S + r][o + k]; }, [&](int k) { return &X[o + k][o + cg]; });
#pragma unroll
    for (int i = 0; i < TR; ++i)
        *reinterpret_cast<float4*>(&Wp[(rg + i) * S + cg]) = make_float4(s[i][0], s[i][1], s[i][2], s[i][3]);
    __syncthreads();
    product([&](int r, int k) { return X[o + S + r][o + S + k]; }, [&](int k) { return &Wp[k * S + cg]; });
#pragma unroll
    for (int i = 0; i < TR; ++i)
        *reinterpret_cast<float4*>(&X[o + S + rg + i][o + cg]) = make_float4(-s[i][0], -s[i][1], -s[i][2], -s[i][3]);
    __syncthreads();
}

__global__ __launch_bounds__(256) void k_tri_inv(const float* __restrict__ A, int lda, int n, float* __restrict__ Linv,
                                                 float* __restrict__ Uinv) {
    __shared__ alignas(16) float X[LU_NB][INV_LD];   // row r of the lower triangle
    __shared__ alignas(16) float W[64 * 64];
    const int t = threadIdx.x, b0 = blockIdx.x * LU_NB, nb = min(LU_NB, n - b0);
    const bool upper = blockIdx.y == 1;
#pragma unroll 16
    for (int q = 0; q < LU_NB * LU_NB / 256; ++q) {
        const int idx = q * 256 + t, k = idx / LU_NB, i = idx % LU_NB;   // row i, column k of the factor
        float v = k == i ? 1.f : 0.f;
        if (k < nb && i < nb && (upper ? i <= k : i > k)) v = A[(size_t)(b0 + k) * lda + b0 + i];
        if (upper) X[k][i] = v;
        else X[i][k] = v;
    }
    __syncthreads();
    float x[16];
    const int o = (t / 16) * 16, c = t % 16;
    if (t < LU_NB) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            float v = r == c ? 1.f : 0.f;
#pragma unroll
            for (int k = 0; k < r; ++k) v -= X[o + r][o + k] * x[k];
            x[r] = upper ? v * (1.f / X[o + r][o + r]) : v;
        }
    }
    __syncthreads();
    if (t < LU_NB)
#pragma unroll
        for (int r = 0; r < 16; ++r) X[o + r][o + c] = x[r];
    __syncthreads();
    inv_double<16>(X, W, t);
    inv_double<32>(X, W, t);
    inv_double<64>(X, W, t);
    float* out = (upper ? Uinv : Linv) + (size_t)blockIdx.x * LU_NB * LU_NB;
#pragma unroll 8
    for (int q = 0; q < LU_NB * LU_NB / 256; ++q) {
        const int idx = q * 256 + t, k = idx / LU_NB, i = idx % LU_NB;
        out[idx] = upper ? X[k][i] : X[i][k];
    }
}

// Blocked triangular solve in one launch: forward y <- L^-1 P r (r in FP64,
// rounded to FP32), backward x += U^-1 y (x in FP64).  Each workgroup takes a
// ticket; ticket t owns block row t (forward) or nblk - 1 - t (backward), so a
// workgroup only waits on blocks owned by workgroups that started before it.  It
// accumulates T(b, c) x_c over the blocks c it depends on, applies the inverse of
// its diagonal block and publishes x_b.  Publication is one 64-bit word per
// element, the value in the low half and the call's epoch in the high half: a
// consumer thread polls the element it needs, so the value arrives with its own
// flag in a single round trip (no separate flag, fence or reload).  Every wait is
// bounded (abort flag, the grid still drains).
//
// Bound by the chain of blocks: a message between compute units and two
// products of a 128 x 128 block per link.  A row of the block is shared by four
// threads, 32 columns each in two sums, and the next block's columns are
// loaded before the wait for this one's x: at order 1 280 and 16 384 the forward
// solve takes 11 and 198 us; two threads per row, one sum and each block's loads
// exposed took 32 and 420.
constexpr int TRSV_G = 4, TRSV_K = LU_NB / TRSV_G;   // threads of a row, columns of a thread
template <bool LOWER>
__global__ __launch_bounds__(LU_NB * TRSV_G) void k_trsv(const float* __restrict__ A, int lda,
                                                         const float* __restrict__ Tinv, const double* __restrict__ r64,
                                                         const int* __restrict__ perm, float* __restrict__ y,
                                                         double* __restrict__ x64, int n, int nblk, unsigned* ticket,
                                                         unsigned base, unsigned long long* yx, unsigned epoch,
                                                         unsigned* abort_flag, const SolveState* __restrict__ st) {
    __shared__ float4 xs4[2][LU_NB / 4];
    __shared__ float part[TRSV_G][LU_NB];
    __shared__ int s_b;
    const int t = threadIdx.x, r = t & (LU_NB - 1), g = t >> 7;
    if (t == 0) s_b = (int)(atomicAdd(ticket, 1u) - base);
    if (st->done) return;
    __syncthreads();
    const int b = LOWER ? s_b : nblk - 1 - s_b;
    const int b0 = b * LU_NB, nb = min(LU_NB, n - b0), k0 = g * TRSV_K;
    const float* Ar = A + b0 + min(r, nb - 1);
    const int ndep = LOWER ? b : nblk - 1 - b;
    // columns past n (in the last block alone) are read as the last, times zero
    auto load = [&](int d, float* a) {
        const int c0 = (LOWER ? d : nblk - 1 - d) * LU_NB, last = n - 1 - c0;
#pragma unroll
        for (int q = 0; q < TRSV_K; ++q) a[q] = Ar[(size_t)(c0 + min(k0 + q, last)) * lda];
    };
    float a[TRSV_K], next[TRSV_K], tinv[TRSV_K];
    if (ndep > 0) load(0, next);
    const float* Tb = Tinv + (size_t)b * LU_NB * LU_NB + k0 * LU_NB + r;
#pragma unroll
    for (int q = 0; q < TRSV_K; ++q) tinv[q] = Tb[q * LU_NB];
    float rhs = 0.f;
    if (t < nb) rhs = LOWER ? (float)r64[perm[b0 + t]] : y[b0 + t];
    auto dot = [&](const float* m, const float4* x) {
        float s0 = 0.f, s1 = 0.f;
#pragma unroll
        for (int q = 0; q < TRSV_K / 4; ++q) {
            const float4 v = x[k0 / 4 + q];
            s0 += m[4 * q] * v.x;
            s1 += m[4 * q + 1] * v.y;
            s0 += m[4 * q + 2] * v.z;
            s1 += m[4 * q + 3] * v.w;
        }
        return s0 + s1;
    };
    float acc = 0.f;
    for (int d = 0; d < ndep; ++d) {
        const int c0 = (LOWER ? d : nblk - 1 - d) * LU_NB, nc = min(LU_NB, n - c0);
#pragma unroll
        for (int q = 0; q < TRSV_K; ++q) a[q] = next[q];
        if (d + 1 < ndep) load(d + 1, next);
        float* xs = reinterpret_cast<float*>(xs4[d & 1]);   // (its last readers passed the barrier of d - 1)
        if (t < LU_NB) {
            float v = 0.f;
            if (t < nc) {
                unsigned spins = 0;
                unsigned long long w = 0ull;
                while (true) {
                    w = __hip_atomic_load(&yx[c0 + t], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    if ((unsigned)(w >> 32) == epoch) break;
                    if ((spins & 31u) == 31u &&
                        __hip_atomic_load(abort_flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0u)
                        break;
                    if (++spins > SPIN_LIMIT) {
                        __hip_atomic_store(abort_flag, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                        break;
                    }
                    __builtin_amdgcn_s_sleep(1);
                }
                v = __uint_as_float((unsigned)(w & 0xFFFFFFFFull));
            }
            xs[t] = v;
        }
        __syncthreads();
        acc += dot(a, xs4[d & 1]);
    }
    part[g][r] = acc;
    __syncthreads();
    if (t < LU_NB)
        reinterpret_cast<float*>(xs4[0])[t] = t < nb ? rhs - ((part[0][t] + part[1][t]) + (part[2][t] + part[3][t])) : 0.f;
    __syncthreads();
    part[g][r] = dot(tinv, xs4[0]);
    __syncthreads();
    if (t < nb) {
        const float xv = (part[0][t] + part[1][t]) + (part[2][t] + part[3][t]);
        __hip_atomic_store(&yx[b0 + t], ((unsigned long long)epoch << 32) | (unsigned long long)__float_as_uint(xv),
                           __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (LOWER) y[b0 + t] = xv;
        else x64[b0 + t] += (double)xv;
    }
}

// ------------------------------------------------------ FP64 residual ----
constexpr int RES_ROWS = 4;   // matrix rows per wavefront (x is read once per 4 rows)
__global__ __launch_bounds__(256) void k_resid64(const double* __restrict__ A, int n, const double* __restrict__ x,
                                                 const double* __restrict__ b, double* __restrict__ r,
                                                 double* __restrict__ rowabs, const SolveState* __restrict__ st) {
    if (st && st->done) return;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int row0 = (blockIdx.x * 4 + wv) * RES_ROWS;
    if (row0 >= n) return;
    const int nrow = min(RES_ROWS, n - row0);
    const double* Ar[RES_ROWS];
#pragma unroll
    for (int q = 0; q < RES_ROWS; ++q) Ar[q] = A + (size_t)(row0 + min(q, nrow - 1)) * n;
    double acc[RES_ROWS], aab[RES_ROWS];
#pragma unroll
    for (int q = 0; q < RES_ROWS; ++q) { acc[q] = 0.0; aab[q] = 0.0; }
    int j = lane;
    for (; j + 192 < n; j += 256) {
        double xv[4], av[RES_ROWS][4];
#pragma unroll
        for (int u = 0; u < 4; ++u) xv[u] = x[j + 64 * u];
#pragma unroll
        for (int q = 0; q < RES_ROWS; ++q)
#pragma unroll
            for (int u = 0; u < 4; ++u) av[q][u] = __builtin_nontemporal_load(Ar[q] + j + 64 * u);
#pragma unroll
        for (int q = 0; q < RES_ROWS; ++q)
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                acc[q] += av[q][u] * xv[u];
                aab[q] += fabs(av[q][u]);
            }
    }
    for (; j < n; j += 64) {
        const double xj = x[j];
#pragma unroll
        for (int q = 0; q < RES_ROWS; ++q) {
            const double a = Ar[q][j];
            acc[q] += a * xj;
            aab[q] += fabs(a);
        }
    }
#pragma unroll
    for (int q = 0; q < RES_ROWS; ++q) {
        for (int off = 32; off > 0; off >>= 1) {
            acc[q] += __shfl_xor(acc[q], off);
            aab[q] += __shfl_xor(aab[q], off);
        }
    }
    if (lane < nrow) {
        double a = 0.0, s = 0.0;
#pragma unroll
        for (int q = 0; q < RES_ROWS; ++q) if (q == lane) { a = acc[q]; s = aab[q]; }
        r[row0 + lane] = b[row0 + lane] - a;
        if (rowabs) rowabs[row0 + lane] = s;
    }
}

// The end of a refinement step, one workgroup: the normwise backward error
// |r| / (|A| |x| + |b|) (|A| from rowabs when given) and whether to go on.
__global__ __launch_bounds__(1024) void k_refine_check(const double* __restrict__ r, const double* __restrict__ x,
                                                       const double* __restrict__ b,
                                                       const double* __restrict__ rowabs, int n, int it, double tol,
                                                       int max_iter, const unsigned* __restrict__ abort_flag,
                                                       SolveState* __restrict__ st) {
    __shared__ double red[4][16];
    if (it > 0 && st->done) return;
    double m[4] = {0.0, 0.0, 0.0, 0.0};
    for (int i = threadIdx.x; i < n; i += 1024) {
        m[0] = fmax(m[0], fabs(r[i]));
        m[1] = fmax(m[1], fabs(x[i]));
        m[2] = fmax(m[2], fabs(b[i]));
        if (rowabs) m[3] = fmax(m[3], rowabs[i]);
    }
    for (int q = 0; q < 4; ++q)
        for (int off = 32; off > 0; off >>= 1) m[q] = fmax(m[q], __shfl_xor(m[q], off));
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    if (lane == 0) for (int q = 0; q < 4; ++q) red[q][wv] = m[q];
    __syncthreads();
    if (threadIdx.x != 0) return;
    for (int q = 0; q < 4; ++q) {
        double v = 0.0;
        for (int k = 0; k < 16; ++k) v = fmax(v, red[q][k]);
        m[q] = v;
    }
    const double anorm = rowabs ? m[3] : st->anorm, denom = anorm * m[1] + m[2];
    const double be = denom > 0.0 ? m[0] / denom : 0.0;
    st->anorm = anorm;
    st->backward = be;
    st->contraction = it > 0 && st->prev > 0.0 ? m[0] / st->prev : it > 0 ? st->contraction : 0.0;
    st->prev = m[0];
    st->it = it;
    st->aborted = *abort_flag;
    st->converged = be <= tol;
    st->done = st->aborted != 0u || !isfinite(be) || be <= tol || it >= max_iter;
}

// ---------------------------------------------------------- VLM kernels --
// Ring geometry (panel.cpp:46-72, 103-120): corners copied per ring, centre,
// unit normal -sum dl_i x dl_i+1, collocation point k centre + (1 - k) leading-
// edge midpoint, and rhs_i = -Vinf . n_i (solver.cpp:256-268).
__global__ void k_ring_geom(const double* __restrict__ nodes, const int* __restrict__ rn, int nr, double kfac,
                            double vx, double vy, double vz, double* __restrict__ corner,
                            double* __restrict__ colloc, double* __restrict__ normal, double* __restrict__ rhs) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= nr) return;
    double p[4][3];
    for (int a = 0; a < 4; ++a) {
        const int id = rn[4 * k + a];
        for (int d = 0; d < 3; ++d) {
            p[a][d] = nodes[3 * id + d];
            corner[12 * k + 3 * a + d] = p[a][d];
        }
    }
    double c[3], nrm[3] = {0.0, 0.0, 0.0}, dl[4][3];
    for (int d = 0; d < 3; ++d) c[d] = (((p[0][d] + p[1][d]) + p[2][d]) + p[3][d]) / 4.0;
    for (int a = 0; a < 4; ++a)
        for (int d = 0; d < 3; ++d) dl[a][d] = p[(a + 1) & 3][d] - p[a][d];
    for (int a = 0; a < 4; ++a) {
        const double* u = dl[a];
        const double* v = dl[(a + 1) & 3];
        nrm[0] -= u[1] * v[2] - u[2] * v[1];
        nrm[1] -= u[2] * v[0] - u[0] * v[2];
        nrm[2] -= u[0] * v[1] - u[1] * v[0];
    }
    const double len = sqrt(nrm[0] * nrm[0] + nrm[1] * nrm[1] + nrm[2] * nrm[2]);
    for (int d = 0; d < 3; ++d) {
        nrm[d] /= len;
        normal[3 * k + d] = nrm[d];
        colloc[3 * k + d] = kfac * c[d] + (1.0 - kfac) * (0.5 * (p[0][d] + p[1][d]));
    }
    rhs[k] = -(vx * nrm[0] + vy * nrm[1] + vz * nrm[2]);
}

// wake ring of every station (surface.cpp:35-58): trailing-edge nodes 3 and
// 2 of the station's last ring, then the same points moved wake_length along
// the unit freestream
__global__ void k_wake(const double* __restrict__ corner, const int* __restrict__ soff, int ns, double L,
                       double wx, double wy, double wz, double* __restrict__ wcorner) {
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= ns) return;
    const int k = soff[s + 1] - 1;
    const double* p = corner + 12 * k;
    const double w[3] = {wx, wy, wz};
    for (int d = 0; d < 3; ++d) {
        const double p1 = p[9 + d], p2 = p[6 + d];
        wcorner[12 * s + 0 + d] = p1;
        wcorner[12 * s + 3 + d] = p2;
        wcorner[12 * s + 6 + d] = p2 + L * w[d];
        wcorner[12 * s + 9 + d] = p1 + L * w[d];
    }
}

// velocity induced at P by a unit-strength ring with corners q[0..3]
// (4 pi times vortexRing::influence, panel.cpp:122-128).  Per segment a->b
// with r1 = P - a, r2 = P - b the reference's h and direction
// (potential.cpp:36-58) give v = (dl.r1/|r1| - dl.r2/|r2|) (r1 x r2) / |r1 x r2|^2
// since dl x r1 = r1 x r2 and |dl x r1| = |r1 x r2|; the Lamb-Oseen factor
// 1 - exp(-(h/rc)^2) multiplies it when rc > 0.
__device__ inline void ring_velocity(const double P[3], const double q[12], double rc, double v[3]) {
    double r[4][3], ir[4];
    for (int a = 0; a < 4; ++a) {
        for (int d = 0; d < 3; ++d) r[a][d] = P[d] - q[3 * a + d];
        ir[a] = rsqrt(r[a][0] * r[a][0] + r[a][1] * r[a][1] + r[a][2] * r[a][2]);
    }
#pragma unroll
    for (int a = 0; a < 4; ++a) {
        const int b = (a + 1) & 3;
        const double* r1 = r[a];
        const double* r2 = r[b];
        const double c0 = r1[1] * r2[2] - r1[2] * r2[1];
        const double c1 = r1[2] * r2[0] - r1[0] * r2[2];
        const double c2 = r1[0] * r2[1] - r1[1] * r2[0];
        const double cc = c0 * c0 + c1 * c1 + c2 * c2;
        const double d0 = q[3 * b] - q[3 * a], d1 = q[3 * b + 1] - q[3 * a + 1], d2 = q[3 * b + 2] - q[3 * a + 2];
        const double tt = (d0 * r1[0] + d1 * r1[1] + d2 * r1[2]) * ir[a] - (d0 * r2[0] + d1 * r2[1] + d2 * r2[2]) * ir[b];
        double s = tt / cc;
        if (rc > 0.0) {
            const double h = sqrt(cc) / tt;
            s *= 1.0 - exp(-(h / rc) * (h / rc));
        }
        v[0] += s * c0;
        v[1] += s * c1;
        v[2] += s * c2;
    }
}

// AIC ring part: A(i, j) = v_j(P_i) . n_i.  Block = 64 columns x 64 rows;
// a wavefront holds 64 consecutive columns of one row, so its stores are
// contiguous in the row-major matrix and its row data is an LDS broadcast.
constexpr int AIC_ROWS_PER_WAVE = 16;
__global__ __launch_bounds__(256) void k_aic(const double* __restrict__ colloc, const double* __restrict__ normal,
                                             const double* __restrict__ corner, int n, double rc,
                                             double* __restrict__ A) {
    __shared__ double sP[64][6];
    const int t = threadIdx.x;
    const int rbase = blockIdx.y * 64;
    if (t < 64) {
        const int i = rbase + t;
        for (int d = 0; d < 3; ++d) {
            sP[t][d] = i < n ? colloc[3 * i + d] : 0.0;
            sP[t][3 + d] = i < n ? normal[3 * i + d] : 0.0;
        }
    }
    __syncthreads();
    const int j = blockIdx.x * 64 + (t & 63);
    if (j >= n) return;
    double q[12];
    for (int a = 0; a < 12; ++a) q[a] = corner[12 * j + a];
    const int r0 = (t >> 6) * AIC_ROWS_PER_WAVE;
    for (int rr = 0; rr < AIC_ROWS_PER_WAVE; ++rr) {
        const int il = r0 + rr, i = rbase + il;
        if (i >= n) break;
        const double P[3] = {sP[il][0], sP[il][1], sP[il][2]};
        double v[3] = {0.0, 0.0, 0.0};
        ring_velocity(P, q, rc, v);
        A[(size_t)i * n + j] = (v[0] * sP[il][3] + v[1] * sP[il][4] + v[2] * sP[il][5]) / FOUR_PI;
    }
}

// wake rings added to their trailing-edge ring's column (solver.cpp:221-236)
__global__ __launch_bounds__(256) void k_aic_wake(const double* __restrict__ colloc, const double* __restrict__ normal,
                                                  const double* __restrict__ wcorner, const int* __restrict__ soff,
                                                  int ns, int n, double rc, double* __restrict__ A) {
    const long long idx = (long long)blockIdx.x * 256 + threadIdx.x;
    if (idx >= (long long)n * ns) return;
    const int s = (int)(idx % ns), i = (int)(idx / ns);
    double q[12];
    for (int a = 0; a < 12; ++a) q[a] = wcorner[12 * s + a];
    const double P[3] = {colloc[3 * i], colloc[3 * i + 1], colloc[3 * i + 2]};
    double v[3] = {0.0, 0.0, 0.0};
    ring_velocity(P, q, rc, v);
    const int te = soff[s + 1] - 1;
    A[(size_t)i * n + te] += (v[0] * normal[3 * i] + v[1] * normal[3 * i + 1] + v[2] * normal[3 * i + 2]) / FOUR_PI;
}

// Kutta-Joukowski per ring, leading to trailing edge of each station
// (wingStation::computeForces, surface.cpp:164-201, with the local stream
// equal to the freestream of the linear solver)
__global__ void k_forces(const double* __restrict__ corner, const double* __restrict__ gamma,
                         const int* __restrict__ soff, int ns, double rho, double vx, double vy, double vz,
                         double* __restrict__ rforce, double* __restrict__ sforce) {
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= ns) return;
    double prev = 0.0, F[3] = {0.0, 0.0, 0.0};
    for (int k = soff[s]; k < soff[s + 1]; ++k) {
        const double* p = corner + 12 * k;
        const double dl0 = p[3] - p[0], dl1 = p[4] - p[1], dl2 = p[5] - p[2];
        const double g = rho * (gamma[k] - prev);
        const double f0 = (vy * dl2 - vz * dl1) * g;
        const double f1 = (vz * dl0 - vx * dl2) * g;
        const double f2 = (vx * dl1 - vy * dl0) * g;
        rforce[3 * k] = f0;
        rforce[3 * k + 1] = f1;
        rforce[3 * k + 2] = f2;
        F[0] += f0;
        F[1] += f1;
        F[2] += f2;
        prev = gamma[k];
    }
    for (int d = 0; d < 3; ++d) sforce[3 * s + d] = F[d];
}

// nonlinear::steady::buildRHS (solver.cpp:303-316): rhs_i = -V(alpha_s).n_i
// with the local angle of the ring's station
__global__ void k_rhs_stations(const double* __restrict__ normal, const int* __restrict__ rst, int nr, double vinf,
                               const double* __restrict__ alpha_deg, double* __restrict__ rhs) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= nr) return;
    const double a = alpha_deg[rst[k]] * M_PI / 180.0;
    rhs[k] = -(vinf * cos(a) * normal[3 * k] + vinf * sin(a) * normal[3 * k + 2]);
}

// Kutta-Joukowski with each station's local stream (wingStation::computeForces
// with inertial_stream() = V(alpha_s))
__global__ void k_forces_stations(const double* __restrict__ corner, const double* __restrict__ gamma,
                                  const int* __restrict__ soff, int ns, double rho, double vinf,
                                  const double* __restrict__ alpha_deg, double* __restrict__ sforce) {
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= ns) return;
    const double a = alpha_deg[s] * M_PI / 180.0;
    const double vx = vinf * cos(a), vz = vinf * sin(a);
    double prev = 0.0, F[3] = {0.0, 0.0, 0.0};
    for (int k = soff[s]; k < soff[s + 1]; ++k) {
        const double* p = corner + 12 * k;
        const double dl0 = p[3] - p[0], dl1 = p[4] - p[1], dl2 = p[5] - p[2];
        const double g = rho * (gamma[k] - prev);
        F[0] += (0.0 * dl2 - vz * dl1) * g;
        F[1] += (vz * dl0 - vx * dl2) * g;
        F[2] += (vx * dl1 - 0.0 * dl0) * g;
        prev = gamma[k];
    }
    for (int d = 0; d < 3; ++d) sforce[3 * s + d] = F[d];
}

// ------------------------------------------------- trailing update (MFMA) --
// C -= A B in FP32 on the matrix cores, all three column-major with one
// leading dimension ld (the LU's A22 -= A21 U12: A is m x k, B is k x n).
// One 256-thread workgroup computes a 128 x 128 tile of C: each wavefront a
// 64 x 64 block as 2 x 2 v_mfma_f32_32x32x2f32 accumulators (16 floats per
// lane each).  K advances in chunks of 16 staged through two LDS buffers: the
// A chunk k-major as in memory (rows contiguous), the B chunk transposed to
// k-major rows padded by 4 words so its column-wise stores spread over the
// banks; the next chunk's global loads are issued before the current chunk's
// MFMAs.  Operand layout of the 32x32x2 instruction: lane l supplies
// A[l % 32][l / 32] and B[l / 32][l % 32] of the 32 x 2 and 2 x 32 slices;
// accumulator element v of lane l is C[8 (v / 4) + 4 (l / 32) + v % 4][l % 32].
// The product is formed transposed (B's columns as the instruction's rows), so
// that a store of one element by 32 lanes is 32 consecutive rows of a column.
// Blocks map to tiles XCD-aware (consecutive tiles of one XCD share A rows).
constexpr int GM_TM = 128, GM_TN = 128, GM_TK = 16;
constexpr int GM_LDB = GM_TN + 4;
typedef float f32x16 __attribute__((ext_vector_type(16)));

__global__ void __launch_bounds__(256) k_gemm_sub_f32(const float* __restrict__ A, const float* __restrict__ B,
                                                       float* __restrict__ C, int ld, int m, int n, int k) {
    __shared__ float As[2][GM_TK][GM_TM];
    __shared__ float Bs[2][GM_TK][GM_LDB];
    const int tiles_m = (m + GM_TM - 1) / GM_TM, tiles_n = (n + GM_TN - 1) / GM_TN;
    const int ntiles = tiles_m * tiles_n;
    // XCD-aware: block b runs on XCD b % 8; XCD x takes tiles [x * per, (x + 1) * per)
    const int nb = gridDim.x, b = blockIdx.x;
    const int per = (nb + 7) / 8;
    const int tile = (b % 8) * per + b / 8;
    if (tile >= ntiles) return;
    const int tm = tile % tiles_m, tn = tile / tiles_m;
    const int row0 = tm * GM_TM, col0 = tn * GM_TN;
    const int t = threadIdx.x, wave = t >> 6, lane = t & 63;
    const int wm = (wave & 1) * 64, wn = (wave >> 1) * 64;
    const bool full = row0 + GM_TM <= m && col0 + GM_TN <= n;
    // global -> register staging: A chunk (128 rows x 16 k): column kk = t / 16,
    // rows 8 (t % 16) .. +8; B chunk (16 k x 128 columns): column t / 2, k
    // 8 (t % 2) .. +8
    const int a_k = t >> 4, a_r = (t & 15) * 8;
    const int b_c = t >> 1, b_k = (t & 1) * 8;
    float ra[8], rb[8];
    auto load = [&](int kb) {
        const int ka = kb + a_k, kbb = kb + b_k;
        const float4* pa = reinterpret_cast<const float4*>(A + (size_t)ka * ld + row0 + a_r);
        const float4 a0 = pa[0], a1 = pa[1];
        ra[0] = a0.x; ra[1] = a0.y; ra[2] = a0.z; ra[3] = a0.w; ra[4] = a1.x; ra[5] = a1.y; ra[6] = a1.z; ra[7] = a1.w;
        const float4* pb = reinterpret_cast<const float4*>(B + (size_t)min(col0 + b_c, n - 1) * ld + kbb);
        const float4 b0 = pb[0], b1 = pb[1];
        rb[0] = b0.x; rb[1] = b0.y; rb[2] = b0.z; rb[3] = b0.w; rb[4] = b1.x; rb[5] = b1.y; rb[6] = b1.z; rb[7] = b1.w;
    };
    auto store = [&](int buf) {
        float4* da = reinterpret_cast<float4*>(&As[buf][a_k][a_r]);
        da[0] = make_float4(ra[0], ra[1], ra[2], ra[3]);
        da[1] = make_float4(ra[4], ra[5], ra[6], ra[7]);
        for (int i = 0; i < 8; ++i) Bs[buf][b_k + i][b_c] = rb[i];
    };
    f32x16 acc[2][2];
    for (int i = 0; i < 2; ++i)
        for (int j = 0; j < 2; ++j)
            for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;
    const int nk = (k + GM_TK - 1) / GM_TK;
    load(0);
    store(0);
    __syncthreads();
    const int lr = lane & 31, lk = lane >> 5;
    for (int c = 0; c < nk; ++c) {
        const int buf = c & 1;
        if (c + 1 < nk) load((c + 1) * GM_TK);
#pragma unroll
        for (int kk = 0; kk < GM_TK; kk += 2) {
            const float a0 = As[buf][kk + lk][wm + lr], a1 = As[buf][kk + lk][wm + 32 + lr];
            const float b0 = Bs[buf][kk + lk][wn + lr], b1 = Bs[buf][kk + lk][wn + 32 + lr];
            acc[0][0] = __builtin_amdgcn_mfma_f32_32x32x2f32(b0, a0, acc[0][0], 0, 0, 0);
            acc[0][1] = __builtin_amdgcn_mfma_f32_32x32x2f32(b1, a0, acc[0][1], 0, 0, 0);
            acc[1][0] = __builtin_amdgcn_mfma_f32_32x32x2f32(b0, a1, acc[1][0], 0, 0, 0);
            acc[1][1] = __builtin_amdgcn_mfma_f32_32x32x2f32(b1, a1, acc[1][1], 0, 0, 0);
        }
        if (c + 1 < nk) {
            store(buf ^ 1);   // the other buffer: its last readers finished before the previous barrier
        }
        __syncthreads();
    }
    // C -= acc
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int row = row0 + wm + i * 32 + lr, cb = col0 + wn + j * 32 + 4 * lk;
            float* pc = C + (size_t)cb * ld + row;
            if (full) {
                float cv[16];
#pragma unroll
                for (int v = 0; v < 16; ++v) cv[v] = pc[(size_t)(8 * (v / 4) + v % 4) * ld];
#pragma unroll
                for (int v = 0; v < 16; ++v) pc[(size_t)(8 * (v / 4) + v % 4) * ld] = cv[v] - acc[i][j][v];
            } else {
#pragma unroll
                for (int v = 0; v < 16; ++v) {
                    const int dc = 8 * (v / 4) + v % 4;
                    if (row < m && cb + dc < n) pc[(size_t)dc * ld] -= acc[i][j][v];
                }
            }
        }
}

hipError_t launch_gemm_sub_f32(hipStream_t s, const float* A, const float* B, float* C, int ld, int m, int n, int k) {
    if (m <= 0 || n <= 0 || k <= 0) return hipSuccess;
    const int tiles = ((m + GM_TM - 1) / GM_TM) * ((n + GM_TN - 1) / GM_TN);
    const int nb = ((tiles + 7) / 8) * 8;
    hipLaunchKernelGGL(k_gemm_sub_f32, dim3(nb), dim3(256), 0, s, A, B, C, ld, m, n, k);
    return hipGetLastError();
}

__global__ void k_panel_reset(unsigned long long* keys, unsigned long long* vals, unsigned long long* prow, int* perm,
                              int* src, int* dst, int n, int nwg, unsigned* abort_flag, unsigned* trsv_abort,
                              int* info) {
    const int stride = gridDim.x * blockDim.x, i0 = blockIdx.x * blockDim.x + threadIdx.x;
    // the words carry the column sequence j0 + j + 1, which repeats from one
    // factorisation to the next
    for (int q = i0; q < 2 * KEY_STRIDE * nwg; q += stride) keys[q] = 0ull;
    for (int q = i0; q < 2 * SUB * nwg; q += stride) vals[q] = 0ull;
    for (int q = i0; q < 2 * SUB * LU_NB; q += stride) prow[q] = 0ull;
    // no interchanges in any panel, for one that gives up before it writes its own
    for (int q = i0; q < n; q += stride) {
        perm[q] = q;
        src[q] = dst[q] = q % LU_NB;
    }
    if (i0 == 0) {
        *abort_flag = 0u;
        *trsv_abort = 0u;   // a new factorisation also re-arms the triangular solves
        *info = 0;
    }
}

template <typename T>
hipError_t dalloc(T** p, size_t count) {
    return hipMalloc((void**)p, std::max<size_t>(count, 1) * sizeof(T));
}

}  // namespace

// ======================================================= dense solver ====
struct afx_dense {
    int n = 0, lda = 0;
    hipStream_t s = nullptr;
    // look-ahead of the factorisation: the update of the columns past the
    // next panel runs on s2 while s factors that panel
    hipStream_t s2 = nullptr;
    hipEvent_t ev_panel = nullptr, ev_near = nullptr, ev_far = nullptr;
    double* A64 = nullptr;     // row-major n x n
    float* A32 = nullptr;      // column-major lda x n, LU in place
    int* ipiv = nullptr;       // followed by src and dst
    int* perm = nullptr;
    double *b = nullptr, *x = nullptr, *r = nullptr, *rowabs = nullptr;
    float* y = nullptr;
    int *src = nullptr, *dst = nullptr;   // every panel's interchanges as a whole (k_panel_lu)
    unsigned long long* keys = nullptr;   // candidates of the panel's workgroups, followed by vals and prow
    unsigned long long* vals = nullptr;   // and their values, value | column sequence
    unsigned long long* prow = nullptr;   // pivot rows of a sub-panel, value | column sequence
    unsigned* pabort = nullptr;
    int* info = nullptr;   // followed by pabort
    float *Linv = nullptr, *Uinv = nullptr;   // inverses of the 128 x 128 diagonal blocks
    unsigned *tk = nullptr, *abort = nullptr;   // triangular-solve tickets and abort flag
    unsigned long long* yx = nullptr;            // published solution elements: value | epoch << 32
    unsigned tk_base = 0, epoch = 0;
    int nblk = 0;
    bool anorm_known = false;   // state->anorm is |A|inf of the current FP64 matrix
    SolveState* state = nullptr;
    struct Results {            // what factor and solve read back
        SolveState solve;
        int info;
        unsigned aborted;
    };
    afx::HostMemory results;
    Results* host() const { return static_cast<Results*>(results.get()); }
    unsigned spin_limit = SPIN_LIMIT;   // of the panel's waits
    bool factored = false;
    ~afx_dense() {
        for (void* p : {(void*)A64, (void*)A32, (void*)ipiv, (void*)perm, (void*)b, (void*)x, (void*)r,
                        (void*)rowabs, (void*)state, (void*)y, (void*)keys,
                        (void*)info, (void*)Linv, (void*)Uinv, (void*)tk,
                        (void*)yx, (void*)abort})
            if (p) (void)hipFree(p);
        if (ev_panel) (void)hipEventDestroy(ev_panel);
        if (ev_near) (void)hipEventDestroy(ev_near);
        if (ev_far) (void)hipEventDestroy(ev_far);
        if (s) (void)hipStreamDestroy(s);
        if (s2) (void)hipStreamDestroy(s2);
    }
};

namespace {

int dense_init(afx_dense* h, int n) {
    if (n <= 0) return api_fail(AFX_EARG, "matrix order must be positive");
    if ((n + PANEL_R - 1) / PANEL_R > MAX_PANEL_WG)
        return api_fail(AFX_EUNSUP, "matrix order " + std::to_string(n) + " exceeds the panel kernel's " +
                                        std::to_string(MAX_PANEL_WG * PANEL_R));
    int dev = 0, coop = 0;
    VCHK(hipGetDevice(&dev));
    VCHK(hipDeviceGetAttribute(&coop, hipDeviceAttributeCooperativeLaunch, dev));
    if (!coop) return api_fail(AFX_EUNSUP, "device does not support cooperative launches");
    h->n = n;
    h->lda = ((n + 31) / 32) * 32 + 32;   // padded so that columns do not alias HBM channels
    VCHK(hipStreamCreateWithFlags(&h->s, hipStreamNonBlocking));
    VCHK(hipStreamCreateWithFlags(&h->s2, hipStreamNonBlocking));
    VCHK(hipEventCreateWithFlags(&h->ev_panel, hipEventDisableTiming));
    VCHK(hipEventCreateWithFlags(&h->ev_near, hipEventDisableTiming));
    VCHK(hipEventCreateWithFlags(&h->ev_far, hipEventDisableTiming));
    const size_t nn = (size_t)n;
    VCHK(dalloc(&h->A64, nn * nn));
    VCHK(dalloc(&h->A32, (size_t)h->lda * nn + LU_NB));   // (the update reads whole tiles of rows)
    VCHK(dalloc(&h->ipiv, 3 * nn));
    h->src = h->ipiv + nn;
    h->dst = h->src + nn;
    VCHK(dalloc(&h->perm, nn));
    VCHK(dalloc(&h->b, nn));
    VCHK(dalloc(&h->x, nn));
    VCHK(dalloc(&h->r, nn));
    VCHK(dalloc(&h->rowabs, nn));
    VCHK(dalloc(&h->state, 1));
    VCHK(h->results.alloc(sizeof(afx_dense::Results)));
    VCHK(dalloc(&h->y, nn));
    const size_t nwg = (nn + PANEL_R - 1) / PANEL_R;
    VCHK(dalloc(&h->keys, 2 * nwg * KEY_STRIDE + 2 * nwg * SUB + 2 * SUB * LU_NB));
    h->vals = h->keys + 2 * nwg * KEY_STRIDE;
    h->prow = h->vals + 2 * nwg * SUB;
    VCHK(dalloc(&h->info, 2));
    h->pabort = reinterpret_cast<unsigned*>(h->info + 1);
    h->nblk = (n + LU_NB - 1) / LU_NB;
    VCHK(dalloc(&h->Linv, (size_t)h->nblk * LU_NB * LU_NB));
    VCHK(dalloc(&h->Uinv, (size_t)h->nblk * LU_NB * LU_NB));
    VCHK(dalloc(&h->tk, 1));
    VCHK(dalloc(&h->yx, h->n));
    VCHK(dalloc(&h->abort, 1));
    VCHK(hipMemsetAsync(h->tk, 0, sizeof(unsigned), h->s));
    VCHK(hipMemsetAsync(h->yx, 0, (size_t)h->n * sizeof(unsigned long long), h->s));
    VCHK(hipMemsetAsync(h->abort, 0, sizeof(unsigned), h->s));
    VCHK(hipStreamSynchronize(h->s));
    return AFX_OK;
}

int dense_factor(afx_dense* h, int32_t* info_out) {
    const int n = h->n, lda = h->lda;
    hipStream_t s = h->s;
    h->factored = false;
    dim3 tg((n + 63) / 64, (n + 63) / 64);
    k_to_cm32<<<tg, 256, 0, s>>>(h->A64, n, h->A32, lda);
    VCHK(hipGetLastError());
    k_panel_reset<<<64, 256, 0, s>>>(h->keys, h->vals, h->prow, h->perm, h->src, h->dst, n,
                                     (n + PANEL_R - 1) / PANEL_R, h->pabort, h->abort, h->info);
    VCHK(hipGetLastError());
    // Right-looking blocked LU with a look-ahead of one panel.  After panel
    // k (columns [j0, c1)) is factored on s, s2 interchanges the rows of the
    // columns past the next panel ([c2, n)), solves their block row and applies
    // step k's update, while s does the same for the next panel's columns
    // [c1, c2) alone and factors that panel.  s waits for the far update of
    // step k - 1 before its own of step k, since that one brought [c1, c2) up to
    // step k - 1; the column sets the two streams touch at the same time are
    // disjoint.  The far product is held back until the near one is done and
    // behind the interchanges of the columns left of the panel (and of the
    // permutation), so that the next panel's workgroups, which need a compute
    // unit's LDS each, find their places before it fills the chip: behind it a
    // panel of 64 workgroups waited out all of the product (1300 us for one of
    // 560).
    float* A = h->A32;
    for (int j0 = 0; j0 < n; j0 += LU_NB) {
        const int nbc = std::min(LU_NB, n - j0);
        const int m = n - j0;
        const int nwg = (m + PANEL_R - 1) / PANEL_R;
        if (nwg == 1) {   // waits for no other workgroup: needs no cooperative launch
            k_panel_lu<<<1, 256, 0, s>>>(A, lda, m, nbc, j0, h->ipiv, h->src, h->dst, h->keys, h->vals, h->prow,
                                         h->pabort, h->spin_limit, h->info);
            VCHK(hipGetLastError());
        } else {
            int ldai = lda, mi = m, nbci = nbc, j0i = j0;
            void* args[] = {&A,       &ldai,    &mi,      &nbci,    &j0i,       &h->ipiv, &h->src,
                            &h->dst,  &h->keys, &h->vals, &h->prow, &h->pabort, &h->spin_limit,
                            &h->info};
            VCHK(hipLaunchCooperativeKernel((const void*)k_panel_lu, dim3(nwg), dim3(256), args, 0, s));
        }
        const int c1 = j0 + nbc, c2 = std::min(n, c1 + LU_NB), rest = n - c1;
        const float* A21 = A + (size_t)j0 * lda + c1;
        VCHK(hipEventRecord(h->ev_panel, s));
        VCHK(hipStreamWaitEvent(h->s2, h->ev_panel, 0));
        if (c2 < n) {
            constexpr int CPW = 8;
            k_swap_solve<CPW, true><<<(n - c2 + 4 * CPW - 1) / (4 * CPW), 256, 0, h->s2>>>(A, lda, c2, n, j0, nbc, h->src,
                                                                                        h->dst, nullptr);
            VCHK(hipGetLastError());
        }
        if (c1 < n) {
            constexpr int CPW = 2;
            if (j0 > 0) VCHK(hipStreamWaitEvent(s, h->ev_far, 0));   // step k - 1 on [c1, c2)
            k_swap_solve<CPW, true><<<(c2 - c1 + 4 * CPW - 1) / (4 * CPW), 256, 0, s>>>(A, lda, c1, c2, j0, nbc, h->src,
                                                                                     h->dst, nullptr);
            VCHK(hipGetLastError());
            VCHK(launch_gemm_sub_f32(s, A21, A + (size_t)c1 * lda + j0, A + (size_t)c1 * lda + c1, lda, rest, c2 - c1,
                                     nbc));
        }
        VCHK(hipEventRecord(h->ev_near, s));
        VCHK(hipStreamWaitEvent(h->s2, h->ev_near, 0));
        k_swap_solve<1, false><<<(j0 + 1 + 3) / 4, 256, 0, h->s2>>>(A, lda, 0, j0, j0, nbc, h->src, h->dst,
                                                                    reinterpret_cast<float*>(h->perm));
        VCHK(hipGetLastError());
        if (c2 < n) {
            VCHK(launch_gemm_sub_f32(h->s2, A21, A + (size_t)c2 * lda + j0, A + (size_t)c2 * lda + c1, lda, rest, n - c2,
                                     nbc));
        }
        VCHK(hipEventRecord(h->ev_far, h->s2));
    }
    k_tri_inv<<<dim3(h->nblk, 2), 256, 0, s>>>(h->A32, lda, n, h->Linv, h->Uinv);
    VCHK(hipGetLastError());
    VCHK(hipEventRecord(h->ev_far, h->s2));
    VCHK(hipStreamWaitEvent(s, h->ev_far, 0));
    VCHK(hipMemcpyAsync(&h->host()->info, h->info, 2 * sizeof(int), hipMemcpyDeviceToHost, s));
    VCHK(hipStreamSynchronize(s));
    const int info = h->host()->info;
    if (h->host()->aborted) return api_fail(AFX_EHIP, "LU panel: pivot exchange timed out (workgroups not co-resident)");
    if (info_out) *info_out = info;
    h->factored = info == 0;
    if (info) return api_fail(AFX_EARG, "matrix is singular in FP32: zero pivot at column " + std::to_string(info - 1));
    return AFX_OK;
}

// FP64 iterative refinement: x = 0 (or the caller's x when warm); repeat r = b - A x (FP64), stop when the
// normwise backward error |r| / (|A| |x| + |b|) <= tol, else x += U^-1 L^-1 P r.  The decisions are taken on
// the device (SolveState) and steps are queued two at a time: a wait after each, with its copies back, took
// a third of a solve of order 1 280, and a step that turns out not to be needed costs its four launches.
int dense_solve_dev(afx_dense* h, const double* b_dev, double* x_dev, double tol, int max_iter, bool warm,
                    afx_solve_info* info) {
    if (!h->factored) return api_fail(AFX_ESTATE, "no factorisation: call factor first");
    const int n = h->n, nb = h->nblk;
    hipStream_t s = h->s;
    if (tol <= 0.0) tol = std::sqrt((double)n) * 1.1102230246251565e-16;
    if (max_iter <= 0) max_iter = 30;
    if (!warm) VCHK(hipMemsetAsync(x_dev, 0, n * sizeof(double), s));
    const bool need_norm = !h->anorm_known;
    auto evaluate = [&](int it) {
        double* rowabs = it == 0 && need_norm ? h->rowabs : nullptr;
        k_resid64<<<(n + 4 * RES_ROWS - 1) / (4 * RES_ROWS), 256, 0, s>>>(h->A64, n, x_dev, b_dev, h->r, rowabs,
                                                                         it > 0 ? h->state : nullptr);
        k_refine_check<<<1, 1024, 0, s>>>(h->r, x_dev, b_dev, rowabs, n, it, tol, max_iter, h->abort, h->state);
    };
    evaluate(0);
    SolveState& st = h->host()->solve;
    for (int it = 0;;) {
        for (int q = 0; q < 2 && it < max_iter; ++q) {
            k_trsv<true><<<nb, LU_NB * TRSV_G, 0, s>>>(h->A32, h->lda, h->Linv, h->r, h->perm, h->y, nullptr, n, nb, h->tk,
                                                      h->tk_base, h->yx, ++h->epoch, h->abort, h->state);
            h->tk_base += (unsigned)nb;
            k_trsv<false><<<nb, LU_NB * TRSV_G, 0, s>>>(h->A32, h->lda, h->Uinv, nullptr, nullptr, h->y, x_dev, n, nb, h->tk,
                                                       h->tk_base, h->yx, ++h->epoch, h->abort, h->state);
            h->tk_base += (unsigned)nb;
            evaluate(++it);
        }
        VCHK(hipGetLastError());
        VCHK(hipMemcpyAsync(&st, h->state, sizeof(st), hipMemcpyDeviceToHost, s));
        VCHK(hipStreamSynchronize(s));
        if (st.done) break;
    }
    if (st.aborted) {
        // the timed-out launch left the solution words incomplete: the
        // factorisation is discarded, and the next factor call clears the
        // flag (k_panel_reset)
        h->factored = false;
        return api_fail(AFX_EHIP, "triangular solve: a block wait timed out (factor again before solving)");
    }
    h->anorm_known = true;
    if (info) {
        *info = afx_solve_info{};
        info->iterations = st.it;
        info->converged = st.converged;
        info->backward_error = st.backward;
        info->contraction = st.contraction;
    }
    return AFX_OK;
}

}  // namespace

// ================================================================ VLM =====
struct afx_vlm {
    int nn = 0, nr = 0, ns = 0;
    std::vector<double> xyz;
    std::vector<int> rn, soff;
    afx_vlm_flow flow{};
    bool flow_set = false, built = false, solved = false, have_gamma = false;
    afx_dense* dense = nullptr;
    double *d_nodes = nullptr, *d_corner = nullptr, *d_wcorner = nullptr, *d_colloc = nullptr,
           *d_normal = nullptr, *d_rhs = nullptr, *d_gamma = nullptr, *d_rforce = nullptr, *d_sforce = nullptr;
    int *d_rn = nullptr, *d_soff = nullptr, *d_rst = nullptr;
    double* d_salpha = nullptr;
    afx::HostMemory staged;    // nodes on their way in, angles and forces
    double* stage() const { return static_cast<double*>(staged.get()); }
    ~afx_vlm() {
        for (void* p : {(void*)d_nodes, (void*)d_corner, (void*)d_wcorner, (void*)d_colloc, (void*)d_normal,
                        (void*)d_rhs, (void*)d_gamma, (void*)d_rforce, (void*)d_sforce, (void*)d_rn, (void*)d_soff,
                        (void*)d_rst, (void*)d_salpha})
            if (p) (void)hipFree(p);
        delete dense;
    }
};

namespace {
double flow_kfac(double alpha_deg) {
    // vortexRing::computeCollocationPoint (panel.cpp:111-120): the branch
    // condition keeps k = 1 for every angle below 1e-6 degrees
    if (alpha_deg < 1e-6 && alpha_deg > -1e6) return 1.0;
    const double a = alpha_deg * M_PI / 180.0;
    return alpha_deg * M_PI / (180.0 * std::sin(a));
}
}  // namespace

extern "C" {

int afx_dense_create(int32_t n, afx_dense** out) {
    if (!out) return api_fail(AFX_EARG, "null argument");
    auto* h = new afx_dense();
    int rc = dense_init(h, n);
    if (rc) { delete h; return rc; }
    *out = h;
    return AFX_OK;
}

int afx_dense_destroy(afx_dense* h) {
    delete h;
    return AFX_OK;
}

int afx_dense_set(afx_dense* h, const double* a) {
    if (!h || !a) return api_fail(AFX_EARG, "null argument");
    VCHK(hipMemcpyAsync(h->A64, a, (size_t)h->n * h->n * sizeof(double), hipMemcpyHostToDevice, h->s));
    VCHK(hipStreamSynchronize(h->s));
    h->anorm_known = false;
    h->factored = false;
    return AFX_OK;
}

int afx_dense_factor(afx_dense* h, int32_t* info) {
    if (!h) return api_fail(AFX_EARG, "null argument");
    return dense_factor(h, info);
}

int afx_dense_solve(afx_dense* h, const double* b, double tol, int32_t max_iter, double* x, afx_solve_info* info) {
    if (!h || !b || !x) return api_fail(AFX_EARG, "null argument");
    const int n = h->n;
    VCHK(hipMemcpyAsync(h->b, b, n * sizeof(double), hipMemcpyHostToDevice, h->s));
    int rc = dense_solve_dev(h, h->b, h->x, tol, max_iter, false, info);
    if (rc) return rc;
    VCHK(hipMemcpyAsync(x, h->x, n * sizeof(double), hipMemcpyDeviceToHost, h->s));
    VCHK(hipStreamSynchronize(h->s));
    return AFX_OK;
}

// Test hook: raise the triangular solves' abort flag as a wait that timed
// out raises it.  The host side of that case follows: the next solve fails
// and discards the factorisation, and the next factor clears the flag
// (k_panel_reset).  No kernel runs here.
int afx_dense_raise_abort(afx_dense* h) {
    if (!h) return api_fail(AFX_EARG, "null argument");
    const unsigned one = 1u;
    VCHK(hipMemcpyAsync(h->abort, &one, sizeof(unsigned), hipMemcpyHostToDevice, h->s));
    VCHK(hipStreamSynchronize(h->s));
    return AFX_OK;
}

// Test hook: the panels' waits give up after `polls` polls (0: the kernels' own
// limit), so that a factorisation takes the way of a timed-out wait with every
// kernel still ending normally.
int afx_dense_limit_polls(afx_dense* h, uint32_t polls) {
    if (!h) return api_fail(AFX_EARG, "null argument");
    h->spin_limit = polls ? std::min(polls, SPIN_LIMIT) : SPIN_LIMIT;
    return AFX_OK;
}

int afx_dense_get_lu(afx_dense* h, float* lu, int32_t* ipiv) {
    if (!h) return api_fail(AFX_EARG, "null argument");
    const int n = h->n;
    if (lu) VCHK(hipMemcpy2DAsync(lu, n * sizeof(float), h->A32, h->lda * sizeof(float), n * sizeof(float), n,
                                  hipMemcpyDeviceToHost, h->s));
    if (ipiv) VCHK(hipMemcpyAsync(ipiv, h->ipiv, n * sizeof(int), hipMemcpyDeviceToHost, h->s));
    VCHK(hipStreamSynchronize(h->s));
    return AFX_OK;
}

int afx_vlm_create(int32_t n_nodes, const double* xyz, int32_t n_stations, const int32_t* soff,
                   const int32_t* ring_nodes, afx_vlm** out) {
    if (!xyz || !soff || !ring_nodes || !out) return api_fail(AFX_EARG, "null argument");
    if (n_nodes <= 0 || n_stations <= 0) return api_fail(AFX_EARG, "empty lattice");
    if (soff[0] != 0) return api_fail(AFX_EARG, "station_offsets[0] must be 0");
    for (int s = 0; s < n_stations; ++s)
        if (soff[s + 1] <= soff[s]) return api_fail(AFX_EARG, "every station needs at least one ring");
    const int nr = soff[n_stations];
    for (int k = 0; k < 4 * nr; ++k)
        if (ring_nodes[k] < 0 || ring_nodes[k] >= n_nodes) return api_fail(AFX_EARG, "ring node id out of range");
    auto* h = new afx_vlm();
    auto bail = [&](int rc) { delete h; return rc; };
    h->nn = n_nodes;
    h->nr = nr;
    h->ns = n_stations;
    h->xyz.assign(xyz, xyz + 3 * (size_t)n_nodes);
    h->rn.assign(ring_nodes, ring_nodes + 4 * (size_t)nr);
    h->soff.assign(soff, soff + n_stations + 1);
    h->dense = new afx_dense();
    int rc = dense_init(h->dense, nr);
    if (rc) return bail(rc);
#define VCHK_C(x)                                                                                    \
    do {                                                                                             \
        hipError_t e_ = (x);                                                                         \
        if (e_ != hipSuccess) return bail(hip_fail(#x, e_));                                         \
    } while (0)
    VCHK_C(dalloc(&h->d_nodes, 3 * (size_t)n_nodes));
    VCHK_C(dalloc(&h->d_corner, 12 * (size_t)nr));
    VCHK_C(dalloc(&h->d_wcorner, 12 * (size_t)n_stations));
    VCHK_C(dalloc(&h->d_colloc, 3 * (size_t)nr));
    VCHK_C(dalloc(&h->d_normal, 3 * (size_t)nr));
    VCHK_C(dalloc(&h->d_rhs, nr));
    VCHK_C(dalloc(&h->d_gamma, nr));
    VCHK_C(dalloc(&h->d_rforce, 3 * (size_t)nr));
    VCHK_C(dalloc(&h->d_sforce, 3 * (size_t)n_stations));
    VCHK_C(dalloc(&h->d_rn, 4 * (size_t)nr));
    VCHK_C(dalloc(&h->d_soff, n_stations + 1));
    VCHK_C(dalloc(&h->d_rst, nr));
    VCHK_C(dalloc(&h->d_salpha, n_stations));
    VCHK_C(h->staged.alloc(sizeof(double) *
                           std::max(3 * (size_t)n_nodes, 3 * ((size_t)nr + n_stations) + n_stations)));
    std::vector<int> rst(nr);
    for (int st = 0; st < n_stations; ++st)
        for (int k = soff[st]; k < soff[st + 1]; ++k) rst[k] = st;
    hipStream_t s = h->dense->s;
    VCHK_C(hipMemcpyAsync(h->d_nodes, xyz, 3 * (size_t)n_nodes * sizeof(double), hipMemcpyHostToDevice, s));
    VCHK_C(hipMemcpyAsync(h->d_rn, ring_nodes, 4 * (size_t)nr * sizeof(int), hipMemcpyHostToDevice, s));
    VCHK_C(hipMemcpyAsync(h->d_soff, soff, (n_stations + 1) * sizeof(int), hipMemcpyHostToDevice, s));
    VCHK_C(hipMemcpyAsync(h->d_rst, rst.data(), nr * sizeof(int), hipMemcpyHostToDevice, s));
    VCHK_C(hipStreamSynchronize(s));
#undef VCHK_C
    *out = h;
    return AFX_OK;
}

int afx_vlm_destroy(afx_vlm* h) {
    delete h;
    return AFX_OK;
}

int afx_vlm_counts(const afx_vlm* h, int32_t* nn, int32_t* nr, int32_t* ns) {
    if (!h) return api_fail(AFX_EARG, "null argument");
    if (nn) *nn = h->nn;
    if (nr) *nr = h->nr;
    if (ns) *ns = h->ns;
    return AFX_OK;
}

int afx_vlm_set_flow(afx_vlm* h, const afx_vlm_flow* f) {
    if (!h || !f) return api_fail(AFX_EARG, "null argument");
    if (!(f->vinf > 0.0) || !(f->rho > 0.0) || !(f->sref > 0.0) || !(f->cref > 0.0))
        return api_fail(AFX_EARG, "vinf, rho, sref and cref must be positive");
    if (f->core_radius < 0.0) return api_fail(AFX_EARG, "core radius must be >= 0");
    h->flow = *f;
    if (!(h->flow.wake_length > 0.0)) h->flow.wake_length = 100.0 * f->cref;   // solver.cpp:36
    h->flow_set = true;
    h->built = h->solved = false;
    return AFX_OK;
}

int afx_vlm_set_nodes(afx_vlm* h, const double* xyz) {
    const int rc = afx::vlm_queue_nodes(h, xyz);
    if (rc) return rc;
    VCHK(hipStreamSynchronize(h->dense->s));
    return AFX_OK;
}

}  // extern "C"

int afx::vlm_queue_nodes(afx_vlm* h, const double* xyz) {
    if (!h || !xyz) return api_fail(AFX_EARG, "null argument");
    std::copy(xyz, xyz + 3 * (size_t)h->nn, h->xyz.begin());
    VCHK(hipStreamSynchronize(h->dense->s));   // the stage is free
    std::copy(h->xyz.begin(), h->xyz.end(), h->stage());
    VCHK(hipMemcpyAsync(h->d_nodes, h->stage(), 3 * (size_t)h->nn * sizeof(double), hipMemcpyHostToDevice, h->dense->s));
    h->built = h->solved = false;
    return AFX_OK;
}

extern "C" {

int afx_vlm_get_nodes(const afx_vlm* h, double* xyz) {
    if (!h || !xyz) return api_fail(AFX_EARG, "null argument");
    std::copy(h->xyz.begin(), h->xyz.end(), xyz);
    return AFX_OK;
}

int afx_vlm_get_rings(const afx_vlm* h, int32_t* ring_nodes, int32_t* soff) {
    if (!h) return api_fail(AFX_EARG, "null argument");
    if (ring_nodes) std::copy(h->rn.begin(), h->rn.end(), ring_nodes);
    if (soff) std::copy(h->soff.begin(), h->soff.end(), soff);
    return AFX_OK;
}

int afx_vlm_build(afx_vlm* h) {
    const int rc = afx::vlm_queue_build(h);
    if (rc) return rc;
    VCHK(hipStreamSynchronize(h->dense->s));
    return AFX_OK;
}

}  // extern "C"

int afx::vlm_queue_build(afx_vlm* h) {
    if (!h) return api_fail(AFX_EARG, "null argument");
    if (!h->flow_set) return api_fail(AFX_ESTATE, "flow not set");
    const afx_vlm_flow& f = h->flow;
    const double a = f.alpha_deg * M_PI / 180.0;
    const double vx = f.vinf * std::cos(a), vy = 0.0, vz = f.vinf * std::sin(a);
    const double kf = flow_kfac(f.alpha_deg);
    const int nr = h->nr, ns = h->ns;
    hipStream_t s = h->dense->s;
    k_ring_geom<<<(nr + 127) / 128, 128, 0, s>>>(h->d_nodes, h->d_rn, nr, kf, vx, vy, vz, h->d_corner, h->d_colloc,
                                                 h->d_normal, h->d_rhs);
    k_wake<<<(ns + 127) / 128, 128, 0, s>>>(h->d_corner, h->d_soff, ns, f.wake_length, std::cos(a), 0.0, std::sin(a),
                                            h->d_wcorner);
    dim3 g((nr + 63) / 64, (nr + 63) / 64);
    k_aic<<<g, 256, 0, s>>>(h->d_colloc, h->d_normal, h->d_corner, nr, f.core_radius, h->dense->A64);
    const long long nw = (long long)nr * ns;
    k_aic_wake<<<(unsigned)((nw + 255) / 256), 256, 0, s>>>(h->d_colloc, h->d_normal, h->d_wcorner, h->d_soff, ns,
                                                            nr, f.core_radius, h->dense->A64);
    VCHK(hipGetLastError());
    h->dense->anorm_known = false;
    h->built = true;
    h->solved = false;
    return AFX_OK;
}

extern "C" {

int afx_vlm_factor(afx_vlm* h) {
    if (!h) return api_fail(AFX_EARG, "null argument");
    if (!h->built) return api_fail(AFX_ESTATE, "matrix not built");
    int32_t info = 0;
    return dense_factor(h->dense, &info);
}

int afx_vlm_solve(afx_vlm* h, double tol, int32_t max_iter, int32_t warm, double* gamma, afx_solve_info* info) {
    if (!h) return api_fail(AFX_EARG, "null argument");
    if (!h->built) return api_fail(AFX_ESTATE, "matrix not built");
    afx_solve_info inf{};
    int rc = dense_solve_dev(h->dense, h->d_rhs, h->d_gamma, tol, max_iter, warm != 0 && h->have_gamma, &inf);
    if (rc) return rc;
    if (info) *info = inf;
    if (gamma) {
        VCHK(hipMemcpyAsync(gamma, h->d_gamma, h->nr * sizeof(double), hipMemcpyDeviceToHost, h->dense->s));
        VCHK(hipStreamSynchronize(h->dense->s));
    }
    h->solved = h->have_gamma = true;
    return AFX_OK;
}

int afx_vlm_forces(afx_vlm* h, double* ring_force, double* station_force, double* coeffs) {
    if (!h) return api_fail(AFX_EARG, "null argument");
    if (!h->solved) return api_fail(AFX_ESTATE, "no solution: call afx_vlm_solve first");
    const afx_vlm_flow& f = h->flow;
    const double a = f.alpha_deg * M_PI / 180.0;
    const double vx = f.vinf * std::cos(a), vz = f.vinf * std::sin(a);
    hipStream_t s = h->dense->s;
    k_forces<<<(h->ns + 127) / 128, 128, 0, s>>>(h->d_corner, h->d_gamma, h->d_soff, h->ns, f.rho, vx, 0.0, vz,
                                                 h->d_rforce, h->d_sforce);
    VCHK(hipGetLastError());
    const size_t nsf = 3 * (size_t)h->ns, nrf = 3 * (size_t)h->nr;
    const double *sf = h->stage(), *rf = sf + nsf;
    VCHK(hipMemcpyAsync(h->stage(), h->d_sforce, nsf * sizeof(double), hipMemcpyDeviceToHost, s));
    if (ring_force)
        VCHK(hipMemcpyAsync(h->stage() + nsf, h->d_rforce, nrf * sizeof(double), hipMemcpyDeviceToHost, s));
    VCHK(hipStreamSynchronize(s));
    if (ring_force) std::copy(rf, rf + nrf, ring_force);
    if (station_force) std::copy(sf, sf + nsf, station_force);
    if (coeffs) {
        // lift axis = freestream x unit-y (input.cpp:46-52), stream axis = freestream
        const double q = 0.5 * f.rho * f.vinf * f.vinf;
        const double lx = -std::sin(a), lz = std::cos(a);
        double cl = 0.0, cy = 0.0, cd = 0.0;
        for (int st = 0; st < h->ns; ++st) {
            const double* F = &sf[3 * st];
            cl += (F[0] * lx + F[2] * lz) / (q * f.sref);
            cy += F[1] / (q * f.sref);
            cd += (F[0] * std::cos(a) + F[2] * std::sin(a)) / (q * f.sref);
        }
        coeffs[0] = cl;
        coeffs[1] = cy;
        coeffs[2] = cd;
    }
    return AFX_OK;
}

}  // extern "C"

namespace {
constexpr double VLM_CLA_DEG = 0.109662271123215082635482531259185634553432464599609375;   // 2 pi per radian

// mlinterp 1D (libs/headeronly/mlinterp): linear inside, end values outside
double interp1(const double* xd, const double* yd, int n, double x) {
    if (n == 1 || x <= xd[0]) return yd[0];
    if (x >= xd[n - 1]) return yd[n - 1];
    int lo = 0, hi = n - 2;
    while (lo <= hi) {
        const int mid = lo + (hi - lo) / 2;
        if (x < xd[mid]) hi = mid - 1;
        else if (x >= xd[mid + 1]) lo = mid + 1;
        else {
            const double w = (xd[mid + 1] - x) / (xd[mid + 1] - xd[mid]);
            return w * yd[mid] + (1.0 - w) * yd[mid + 1];
        }
    }
    return yd[n - 1];
}

// database::table::coefficients (database.cpp:192-242): each section's
// airfoil at alpha, then across the span
void polar_coeffs(const afx_polar& P, double alpha, double span, double* out3) {
    std::vector<double> c[3];
    for (int q = 0; q < P.n_sections; ++q) {
        const int a = P.section_airfoil[q];
        const int o = P.offsets[a], n = P.offsets[a + 1] - o;
        c[0].push_back(interp1(P.alpha_deg + o, P.cl + o, n, alpha));
        c[1].push_back(interp1(P.alpha_deg + o, P.cd + o, n, alpha));
        c[2].push_back(interp1(P.alpha_deg + o, P.cmy + o, n, alpha));
    }
    for (int k = 0; k < 3; ++k) out3[k] = interp1(P.section_span, c[k].data(), P.n_sections, span);
}
}  // namespace

extern "C" {

int afx_vlm_nonlinear_solve(afx_vlm* h, const afx_polar* P, double relaxation, double tol, int32_t max_iter,
                            afx_nonlinear_info* info, double* station_alpha, double* station_cl) {
    if (!h || !P) return api_fail(AFX_EARG, "null argument");
    if (!h->flow_set) return api_fail(AFX_ESTATE, "flow not set");
    if (P->n_airfoils < 1 || P->n_sections < 1 || !P->offsets || !P->alpha_deg || !P->cl || !P->cd || !P->cmy ||
        !P->section_airfoil || !P->section_span)
        return api_fail(AFX_EARG, "polar table is empty");
    for (int a = 0; a < P->n_airfoils; ++a)
        if (P->offsets[a + 1] <= P->offsets[a]) return api_fail(AFX_EARG, "an airfoil polar has no rows");
    for (int q = 0; q < P->n_sections; ++q)
        if (P->section_airfoil[q] < 0 || P->section_airfoil[q] >= P->n_airfoils)
            return api_fail(AFX_EARG, "section airfoil index out of range");
    const afx_vlm_flow& f = h->flow;
    const int ns = h->ns;
    int rc = afx::vlm_queue_build(h);
    if (rc) return rc;
    if ((rc = afx_vlm_factor(h))) return rc;
    // station geometry (wingStation / wing, surface.cpp): area = sum of ring
    // areas (panel.cpp:64-72), leading-edge segment of the first ring, span
    // location (wing::computeSpan) normalised from the first station
    std::vector<double> area(ns, 0.0), le(3 * (size_t)ns), spanloc(ns);
    auto node = [&](int id, int d) { return h->xyz[3 * (size_t)id + d]; };
    double span = 0.0;
    for (int st = 0; st < ns; ++st) {
        for (int k = h->soff[st]; k < h->soff[st + 1]; ++k) {
            double c[3] = {0, 0, 0};
            for (int a = 0; a < 4; ++a)
                for (int d = 0; d < 3; ++d) c[d] += node(h->rn[4 * k + a], d) / 4.0;
            for (int a = 0; a < 4; ++a) {
                const int i0 = h->rn[4 * k + a], i1 = h->rn[4 * k + ((a + 1) & 3)];
                const double dl[3] = {node(i1, 0) - node(i0, 0), node(i1, 1) - node(i0, 1), node(i1, 2) - node(i0, 2)};
                const double ce[3] = {c[0] - node(i0, 0), c[1] - node(i0, 1), c[2] - node(i0, 2)};
                const double x = dl[1] * ce[2] - dl[2] * ce[1], y = dl[2] * ce[0] - dl[0] * ce[2],
                             z = dl[0] * ce[1] - dl[1] * ce[0];
                area[st] += 0.5 * std::sqrt(x * x + y * y + z * z);
            }
        }
        const int k0 = h->soff[st];
        for (int d = 0; d < 3; ++d) le[3 * st + d] = node(h->rn[4 * k0 + 1], d) - node(h->rn[4 * k0], d);
        const double len = std::sqrt(le[3 * st] * le[3 * st] + le[3 * st + 1] * le[3 * st + 1] +
                                     le[3 * st + 2] * le[3 * st + 2]);
        span += len;
        spanloc[st] = span - 0.5 * len;
    }
    for (int st = ns - 1; st >= 0; --st) spanloc[st] = (spanloc[st] - spanloc[0]) / span;
    const double q = 0.5 * f.rho * f.vinf * f.vinf;
    std::vector<double> alpha(ns, f.alpha_deg), clinv(ns);
    double *sf = h->stage(), *angles = sf + 3 * (size_t)ns;   // (free after each wait of the loop)
    VCHK(hipStreamSynchronize(h->dense->s));
    hipStream_t s = h->dense->s;
    auto lift_axis = [&](int st, double* ax) {   // unit(V(alpha_s) x dl_LE)
        const double a = alpha[st] * M_PI / 180.0, vx = std::cos(a), vz = std::sin(a);
        const double* d = &le[3 * st];
        ax[0] = 0.0 * d[2] - vz * d[1];
        ax[1] = vz * d[0] - vx * d[2];
        ax[2] = vx * d[1] - 0.0 * d[0];
        const double n = std::sqrt(ax[0] * ax[0] + ax[1] * ax[1] + ax[2] * ax[2]);
        for (int k = 0; k < 3; ++k) ax[k] /= n;
    };
    afx_nonlinear_info inf{};
    int iter = 0;
    double residual = 0.0;
    do {
        std::copy(alpha.begin(), alpha.end(), angles);
        VCHK(hipMemcpyAsync(h->d_salpha, angles, ns * sizeof(double), hipMemcpyHostToDevice, s));
        k_rhs_stations<<<(h->nr + 127) / 128, 128, 0, s>>>(h->d_normal, h->d_rst, h->nr, f.vinf, h->d_salpha, h->d_rhs);
        VCHK(hipGetLastError());
        afx_solve_info si{};
        if ((rc = dense_solve_dev(h->dense, h->d_rhs, h->d_gamma, 0.0, 30, iter > 0, &si))) return rc;
        if (!si.converged) return api_fail(AFX_EARG, "vortex-lattice refinement did not converge");
        h->solved = h->have_gamma = true;
        k_forces_stations<<<(ns + 127) / 128, 128, 0, s>>>(h->d_corner, h->d_gamma, h->d_soff, ns, f.rho, f.vinf,
                                                           h->d_salpha, h->d_sforce);
        VCHK(hipGetLastError());
        VCHK(hipMemcpyAsync(sf, h->d_sforce, 3 * (size_t)ns * sizeof(double), hipMemcpyDeviceToHost, s));
        VCHK(hipStreamSynchronize(s));
        residual = 0.0;
        for (int st = 0; st < ns; ++st) {
            double ax[3];
            lift_axis(st, ax);
            clinv[st] = (sf[3 * st] * ax[0] + sf[3 * st + 1] * ax[1] + sf[3 * st + 2] * ax[2]) / (q * area[st]);
            const double aoa_eff = clinv[st] / VLM_CLA_DEG - alpha[st] + f.alpha_deg;
            double c3[3];
            polar_coeffs(*P, aoa_eff, spanloc[st], c3);
            alpha[st] += relaxation * (c3[0] - clinv[st]) / VLM_CLA_DEG;
            const double r = (c3[0] - clinv[st]) / c3[0];
            residual += r * r;
        }
        residual = std::sqrt(residual);
        ++iter;
    } while (residual > tol && iter <= max_iter);
    // nonlinear::steady::computeForces (solver.cpp:434-476): viscous section
    // coefficients at the final effective angles
    const double A = f.alpha_deg * M_PI / 180.0;
    const double lx = -std::sin(A), lz = std::cos(A);
    double cl = 0.0, cd = 0.0, cy = 0.0;
    for (int st = 0; st < ns; ++st) {
        const double aoa_eff = clinv[st] / VLM_CLA_DEG - alpha[st] + f.alpha_deg;
        double c3[3], ax[3];
        polar_coeffs(*P, aoa_eff, spanloc[st], c3);
        lift_axis(st, ax);
        const double scl = c3[0] * (ax[0] * lx + ax[2] * lz);
        cl += scl * area[st] / f.sref;
        cy += c3[0] * ax[1] * area[st] / f.sref;
        cd += c3[1] * area[st] / f.sref;
        if (station_cl) station_cl[st] = scl;
    }
    if (station_alpha) std::copy(alpha.begin(), alpha.end(), station_alpha);
    inf.iterations = iter;
    inf.converged = residual <= tol;
    inf.residual = residual;
    inf.cl = cl;
    inf.cd = cd;
    inf.cy = cy;
    if (info) *info = inf;
    return AFX_OK;
}

int afx_vlm_get_aic(afx_vlm* h, double* aic) {
    if (!h || !aic) return api_fail(AFX_EARG, "null argument");
    if (!h->built) return api_fail(AFX_ESTATE, "matrix not built");
    VCHK(hipMemcpyAsync(aic, h->dense->A64, (size_t)h->nr * h->nr * sizeof(double), hipMemcpyDeviceToHost,
                        h->dense->s));
    VCHK(hipStreamSynchronize(h->dense->s));
    return AFX_OK;
}

int afx_vlm_get_system(afx_vlm* h, double* rhs, double* gamma, double* colloc, double* normal) {
    if (!h) return api_fail(AFX_EARG, "null argument");
    hipStream_t s = h->dense->s;
    const size_t nr = h->nr;
    if (rhs) VCHK(hipMemcpyAsync(rhs, h->d_rhs, nr * sizeof(double), hipMemcpyDeviceToHost, s));
    if (gamma) VCHK(hipMemcpyAsync(gamma, h->d_gamma, nr * sizeof(double), hipMemcpyDeviceToHost, s));
    if (colloc) VCHK(hipMemcpyAsync(colloc, h->d_colloc, 3 * nr * sizeof(double), hipMemcpyDeviceToHost, s));
    if (normal) VCHK(hipMemcpyAsync(normal, h->d_normal, 3 * nr * sizeof(double), hipMemcpyDeviceToHost, s));
    VCHK(hipStreamSynchronize(s));
    return AFX_OK;
}

}  // extern "C"
