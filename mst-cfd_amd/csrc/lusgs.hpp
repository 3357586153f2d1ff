// Steady driver: matrix-free LU-SGS over a cell colouring.
//
// The factorised operator (D+L) D^-1 (D+U) -- a forward sweep with the lower part, a division by D, a
// backward sweep with the upper part -- is the one SparseSolverNUM::solveILUSGS applies to its
// assembled scalar systems (lusolver/SparseSolverNUM.cpp:144-196).  Here the blocks are never
// assembled; they come from the Rusanov split of the face-flux Jacobian (Jameson & Yoon, AIAA J.
// 25(7), 1987):
//   r_f  = max over the face's cells of |u.S_f| + a |S_f|        (boundary face: its one cell)
//   D_i  = (1/CFL + omega/2) sum_f r_f                            (local step CFL V_i / sum_f r_f)
//   (i,j) block times dQ_j = 1/2 [F_n(Q_j + dQ_j) - F_n(Q_j)] - 1/2 omega r_f dQ_j,
//        n = the outward normal of cell i at f, F_n = sum_d n_d F_d (physical Euler flux)
// L / U hold the neighbours of lower / higher colour; boundary faces enter D only.
//
// Sequential Gauss-Seidel order is replaced by colour order: no two cells of one colour are
// neighbours, so one launch per colour updates all of its cells at once, and the result is the same
// as sweeping the cells one by one in colour order (the order inside a colour does not matter).
//   k_lu_sweep   one lane per cell of one colour; forward: r_f of the cell's faces, D, and
//                dQ* = (-R - sum_L ...) / D; backward: dQ = dQ* - sum_U ... / D, Q_new = Q + dQ
//                (and the admissibility check)
// Both sweeps are gathers over the neighbours of a cell, like the residual's gather; a colour of a few hundred thousand
// cells is two or three waves per SIMD, all in step, so they are bound by their loads' latency and then the solves'.
#pragma once
#include "kernels.hpp"

namespace mstk {

// Cells are addressed by their position t in the colour-sorted list (colour k: positions
// [start_k, start_{k+1})); per (slot, position), slot-major, the sweeps read precomputed records so a
// neighbour costs one round of dependent loads (its state and update) instead of walking
// cell -> face -> neighbour -> colour.
struct LuArgs {
    int64_t nc;
    const int32_t *__restrict__ cells;   // position -> cell
    const int32_t *__restrict__ nb;      // (neighbour << 2) | 1 (lower colour) | 2 (higher colour);
                                         // -1 boundary face, -2 past the last face
    const double *__restrict__ n;        // outward normal of the cell at the slot (area-weighted)
    double *__restrict__ r;              // spectral radius of the slot's face (per iteration)
    double *__restrict__ D;              // diagonal (per iteration)
    const double *__restrict__ Q;        // state at the start of the iteration (cell order)
    const double *__restrict__ R;        // its residual (cell order)
    double *__restrict__ dQ;             // update (cell order)
    double *__restrict__ Qout;
    int *__restrict__ bad;
    double gamma, dscale, omega;         // dscale = 1/CFL + omega/2
    // first-order residual computed by the forward sweep itself (RSCHEME >= 0)
    const uint32_t *__restrict__ finfo;  // per position, byte s: kind | (L/R mask << 3) | (is_c1 << 6) of slot s's face
    Params<double> P;
    // batches: the case of each position, per case its parameters, scheme, gamma and active flag (inactive cases
    // are skipped; the bad flag is per case); G: the face fluxes of LU_R_GATHER
    const int32_t *__restrict__ pcase;
    const Params<double> *__restrict__ Pc;
    const int32_t *__restrict__ scheme;
    const double *__restrict__ gam;
    const uint8_t *__restrict__ active;
    const double *__restrict__ G;
    const int32_t *__restrict__ face;    // (face << 1) | is_c1 per (slot, position)
};

// the finfo words of LuArgs from the face codes and the faces' current kinds and masks (kind < 8, mask < 8): one
// coalesced 4-byte load per cell in the sweeps instead of a code and a dependent gather per slot
template <int U>
__global__ __launch_bounds__(BLOCK) void k_lu_finfo(int64_t nc, int slots, const int32_t *__restrict__ face,
                                                    const int32_t *__restrict__ finfo, uint32_t *__restrict__ out) {
    const int64_t t = (int64_t)blockIdx.x * BLOCK + threadIdx.x;
    if (t >= nc) return;
    uint32_t v = 0;
    for (int s = 0; s < slots && s < 4; s++) {
        const int32_t e = face[(int64_t)s * nc + t];
        if (e < 0) break;
        const int info = finfo[e >> 1];
        v |= ((uint32_t)(info & 7) | (uint32_t)((info >> 4) & 7) << 3 | (uint32_t)(e & 1) << 6) << (8 * s);
    }
    out[t] = v;
}

// one wave per workgroup: a colour is a few hundred 256-lane blocks, an uneven share of the 256 CUs (bf / last forward
// sweep, 150,000 cells: 22.5 / 17.9 us at 256 lanes, 21.3 / 17.8 at 64; 92,000 cells of a batch: 15.7 / 14.2, 15.3 / 13.7)
constexpr int LU_BLOCK = 64;

// residual sources of the forward sweep
constexpr int LU_R_ARRAY = -1;   // read R
constexpr int LU_R_GATHER = -2;  // sum +-G_f of the cell's faces in slot order (the gather kernels' order)
constexpr int LU_R_RUNTIME = -3; // as a scheme (>= 0), chosen per case

template <int DIM>
__device__ __forceinline__ double lu_pressure(const double *q, double gamma) {
    constexpr int NV = DIM + 2;
    double ke = 0;
#pragma unroll
    for (int d = 0; d < DIM; d++) ke += q[1 + d] * q[1 + d];
    return (q[NV - 1] - 0.5 * ke / q[0]) * (gamma - 1);
}

template <int DIM>
__device__ __forceinline__ double lu_radius(const double *q, const double *n, double gamma) {
    double un = 0, s2 = 0;
#pragma unroll
    for (int d = 0; d < DIM; d++) {
        un += q[1 + d] * n[d];
        s2 += n[d] * n[d];
    }
    const double p = lu_pressure<DIM>(q, gamma);
    return fabs(un / q[0]) + sqrt(gamma * p / q[0]) * sqrt(s2);
}

template <int DIM>
__device__ __forceinline__ void lu_flux(const double *q, const double *n, double gamma, double *F) {
    constexpr int NV = DIM + 2;
    double un = 0;
#pragma unroll
    for (int d = 0; d < DIM; d++) un += q[1 + d] * n[d];
    un /= q[0];
    const double p = lu_pressure<DIM>(q, gamma);
    F[0] = q[0] * un;
#pragma unroll
    for (int d = 0; d < DIM; d++) F[1 + d] = q[1 + d] * un + p * n[d];
    F[NV - 1] = (q[NV - 1] + p) * un;
}

// -R of a cell (order 1, cells of <= 4 faces) from its state qc and its neighbours' q: the same face solves
// (face_solve, the c0 outward normal, the c0 side first) summed in slot order as the gather kernels sum them, so R
// is theirs bit for bit.
template <int DIM, int MAXF, int RSCHEME>
__device__ __forceinline__ void lu_solve(const Params<double> &P, const bool roe, const uint32_t finfo,
                                         const int32_t (&code)[MAXF], const double (&nrm)[MAXF][DIM],
                                         const double (&qc)[DIM + 2], const double (&q)[MAXF][DIM + 2],
                                         double (&s)[DIM + 2]) {
    constexpr int NV = DIM + 2;
    double r[NV], cmp[NV];
#pragma unroll
    for (int j = 0; j < NV; j++) r[j] = cmp[j] = 0;
#pragma unroll
    for (int k = 0; k < MAXF; k++) {
        if (code[k] == -2) break;
        const uint32_t e = finfo >> (8 * k);
        const int kind = (int)(e & 7);
        if (kind >= mst::KIND_NONE) continue;  // zero-flux face
        const bool c1side = e & 64;
        double n64[DIM], X[NV], Y[NV], g[NV];
#pragma unroll
        for (int d = 0; d < DIM; d++) n64[d] = c1side ? -nrm[k][d] : nrm[k][d];
#pragma unroll
        for (int j = 0; j < NV; j++) {
            X[j] = (code[k] >= 0 && c1side) ? q[k][j] : qc[j];
            Y[j] = code[k] >= 0 ? (c1side ? qc[j] : q[k][j]) : qc[j];
        }
        face_solve<DIM, (RSCHEME == LU_R_RUNTIME ? SCHEME_RUNTIME : RSCHEME), double>(
            P, RSCHEME == LU_R_RUNTIME ? roe : RSCHEME == MST_SCHEME_ROE, kind, (int)(e >> 3 & 7), n64, X, Y, g);
        accumulate<NV, false>(r, cmp, g, c1side);
    }
#pragma unroll
    for (int j = 0; j < NV; j++) s[j] = -r[j];
}

// s -= a neighbour's off-diagonal term, from its state q, q + dq, dq and the face's radius
template <int DIM>
__device__ __forceinline__ void lu_offdiag(const double *q, const double *qp, const double *dq, const double *n, double r,
                                           double gamma, double omega, double *s) {
    constexpr int NV = DIM + 2;
    double F1[NV], F0[NV];
    lu_flux<DIM>(qp, n, gamma, F1);
    lu_flux<DIM>(q, n, gamma, F0);
#pragma unroll
    for (int j = 0; j < NV; j++) s[j] -= 0.5 * ((F1[j] - F0[j]) - omega * r * dq[j]);
}

// One colour's positions [t0, t0 + n).
// FWD: the spectral radius of each of the cell's faces (max over the face's two cells: the same value
// from either side, exactly, since it depends on the normal only through |u.n| and |n|) and D are
// computed and stored for the backward sweep, then dQ* = (-R - sum_L ...) / D.  The last colour has
// no higher neighbours, so its backward sweep is the identity: LAST also writes Qout, and neither radii nor D.
// Backward (!FWD): dQ = dQ* - sum_U ... / D, Qout = Q + dQ.
// RSCHEME = LU_R_GATHER (forward, cells of <= 4 faces): R is gathered from the face fluxes G.
// RSCHEME a scheme (forward, order 1, cells of <= 4 faces): R of the cell is not read but computed here
// (lu_solve), from the states the sweep loads anyway.
// One cell's sweep (position t, cell c).  P, roe: of the cell's case.
// (Solving each face once, its flux and radius stored by the lower colour's sweep for the higher's, cut colour 1's
// vector instructions from 1,770 to 560 per wave and its time from 18.6 to 17.3 us on 300,000 triangles, but colour
// 0's kernel grew from 22.7 to 24.5 us with the stores, and colour 1 waits for its loads either way.  Not kept.)
template <int DIM, bool FWD, bool LAST, int MAXF, int RSCHEME>
__device__ __forceinline__ void lu_cell(const LuArgs &a, const Params<double> &P, const bool roe, const int64_t t,
                                        const int64_t c) {
    static_assert(RSCHEME == LU_R_ARRAY || (FWD && MAXF <= 4), "computed residual: forward sweeps of small cells");
    constexpr int NV = DIM + 2;
    constexpr bool SOLVE = RSCHEME >= 0 || RSCHEME == LU_R_RUNTIME;
    double s[NV], qc[NV];
    if constexpr (FWD) {
        if constexpr (RSCHEME == LU_R_ARRAY) {
            ldq<NV>(a.R + c * NV, s);
#pragma unroll
            for (int k = 0; k < NV; k++) s[k] = -s[k];
        }
        ldq<NV>(a.Q + c * NV, qc);
    } else {
#pragma unroll
        for (int k = 0; k < NV; k++) s[k] = 0;
    }
    double dqc[NV], D = 0;  // backward: the cell's own update, state and diagonal, read up front
    if constexpr (!FWD) {
        ldq<NV>(a.dQ + c * NV, dqc);
        ldq<NV>(a.Q + c * NV, qc);
        D = a.D[t];
    }
    constexpr int32_t SIDE = FWD ? 1 : 2;
    double rsum = 0;
    if constexpr (MAXF <= 4) {
        // every memory read of the cell's slots is issued before the first is used: two rounds of
        // dependent loads per cell (records, then neighbour states and updates) instead of two per
        // slot.  The arithmetic below runs in the same order as the slot loop further down.
        int32_t code[MAXF], fcode[MAXF];
        double nrm[MAXF][DIM], q[MAXF][NV], dq[MAXF][NV], rr[MAXF];
#pragma unroll
        for (int k = 0; k < MAXF; k++) code[k] = a.nb[(int64_t)k * a.nc + t];
        uint32_t finfo = 0;
        if constexpr (SOLVE) finfo = a.finfo[t];
        if constexpr (RSCHEME == LU_R_GATHER) {
#pragma unroll
            for (int k = 0; k < MAXF; k++) fcode[k] = a.face[(int64_t)k * a.nc + t];
        }
        double gsl[MAXF][NV];  // gathered face fluxes (RSCHEME == LU_R_GATHER)
        if constexpr (RSCHEME == LU_R_GATHER) {
#pragma unroll
            for (int k = 0; k < MAXF; k++)
                if (fcode[k] >= 0) ldq<NV>(a.G + (int64_t)(fcode[k] >> 1) * NV, gsl[k]);
        }
#pragma unroll
        for (int k = 0; k < MAXF; k++) {
            const int64_t i = (int64_t)k * a.nc + t;
            const bool nbr = code[k] >= 0, use = nbr && (code[k] & SIDE);
            const int64_t o = code[k] >> 2;
            if (FWD ? code[k] != -2 : use) {
#pragma unroll
                for (int d = 0; d < DIM; d++) nrm[k][d] = a.n[i * DIM + d];
            }
            if (FWD ? nbr : use) ldq<NV>(a.Q + o * NV, q[k]);
            if (use) ldq<NV>(a.dQ + o * NV, dq[k]);
            if (!FWD && use) rr[k] = a.r[i];
        }
        if constexpr (RSCHEME == LU_R_GATHER) {
            double r[NV], cmp[NV];
#pragma unroll
            for (int j = 0; j < NV; j++) r[j] = cmp[j] = 0;
#pragma unroll
            for (int k = 0; k < MAXF; k++) {
                if (code[k] == -2) break;
                accumulate<NV, false>(r, cmp, gsl[k], fcode[k] & 1);
            }
#pragma unroll
            for (int j = 0; j < NV; j++) s[j] = -r[j];
        }
        if constexpr (SOLVE) lu_solve<DIM, MAXF, RSCHEME>(P, roe, finfo, code, nrm, qc, q, s);
#pragma unroll
        for (int k = 0; k < MAXF; k++) {
            if (code[k] == -2) break;  // the slots after it are padding too
            const bool nbr = code[k] >= 0, use = nbr && (code[k] & SIDE);
            double r;
            if constexpr (FWD) {
                r = lu_radius<DIM>(qc, nrm[k], a.gamma);
                if (nbr) r = fmax(r, lu_radius<DIM>(q[k], nrm[k], a.gamma));
                if constexpr (!LAST) a.r[(int64_t)k * a.nc + t] = r;
                rsum += r;
            } else {
                r = rr[k];
            }
            if (!use) continue;
            double qp[NV];
#pragma unroll
            for (int j = 0; j < NV; j++) qp[j] = q[k][j] + dq[k][j];
            lu_offdiag<DIM>(q[k], qp, dq[k], nrm[k], r, a.gamma, a.omega, s);
        }
    } else {
#pragma unroll
        for (int slot = 0; slot < MAXF; slot++) {
            const int64_t i = (int64_t)slot * a.nc + t;
            const int32_t code = a.nb[i];
            if (code == -2) break;
            if (!FWD && (code < 0 || !(code & SIDE))) continue;
            double nrm[DIM], q[NV];
#pragma unroll
            for (int d = 0; d < DIM; d++) nrm[d] = a.n[i * DIM + d];
            const int64_t o = code >> 2;
            if (code >= 0) ldq<NV>(a.Q + o * NV, q);
            double r;
            if constexpr (FWD) {
                r = lu_radius<DIM>(qc, nrm, a.gamma);
                if (code >= 0) r = fmax(r, lu_radius<DIM>(q, nrm, a.gamma));
                if constexpr (!LAST) a.r[i] = r;
                rsum += r;
                if (code < 0 || !(code & SIDE)) continue;
            } else {
                r = a.r[i];
            }
            double dq[NV], qp[NV];
            ldq<NV>(a.dQ + o * NV, dq);
#pragma unroll
            for (int k = 0; k < NV; k++) qp[k] = q[k] + dq[k];
            lu_offdiag<DIM>(q, qp, dq, nrm, r, a.gamma, a.omega, s);
        }
    }
    if constexpr (FWD) {
        D = a.dscale * rsum;
        if constexpr (!LAST) a.D[t] = D;
    }
    double dq[NV], out[NV];
    if constexpr (FWD) {
#pragma unroll
        for (int k = 0; k < NV; k++) dq[k] = s[k] / D;
    } else {
#pragma unroll
        for (int k = 0; k < NV; k++) dq[k] = dqc[k] + s[k] / D;
    }
    stq<NV>(a.dQ + c * NV, dq);
    if constexpr (!FWD || LAST) {
#pragma unroll
        for (int k = 0; k < NV; k++) out[k] = qc[k] + dq[k];
        stq<NV>(a.Qout + c * NV, out);
        const double p = lu_pressure<DIM>(out, a.gamma);
        if (!(out[0] > 0) || !(p > 0)) a.bad[0] = 1;
    }
}

// f(a, P, roe) with the parameters of position t's case in scalar registers: the lanes of one case at a time (nearly
// always the whole wave), inactive cases left out; a single context (not BATCH) once.
template <bool BATCH, typename F>
__device__ __forceinline__ void lu_per_case(const LuArgs &a, const int64_t t, F f) {
    if constexpr (!BATCH) {
        f(a, a.P, false);
    } else {
        const int32_t cs = a.pcase[t];
        for (bool todo = true; todo;) {
            const int32_t u = __builtin_amdgcn_readfirstlane(cs);
            if (cs != u) continue;
            todo = false;
            if (!a.active[u]) continue;
            LuArgs b = a;
            b.gamma = a.gam[u];
            b.bad += u;
            f(b, a.Pc[u], a.scheme[u] == MST_SCHEME_ROE);
        }
    }
}

template <int DIM, bool FWD, bool LAST, int MAXF, int RSCHEME = LU_R_ARRAY, bool BATCH = false>
__global__ __launch_bounds__(LU_BLOCK) void k_lu_sweep(const LuArgs a, int64_t t0, int64_t n) {
    const int64_t l = block_id() * LU_BLOCK + threadIdx.x;
    if (l >= n) return;
    const int64_t t = t0 + l;
    lu_per_case<BATCH>(a, t, [&](const LuArgs &b, const Params<double> &P, bool roe) {
        lu_cell<DIM, FWD, LAST, MAXF, RSCHEME>(b, P, roe, t, b.cells[t]);
    });
}

// Colour 0's backward sweep of one iteration fused with its forward sweep of the next (first order, the residual
// computed in the forward sweeps, two colours or more).  Colour 0 has no lower neighbours, so its forward sweep needs
// only the cell's and its neighbours' new states.  A neighbour's is the sum Q + dQ that the backward term forms and
// that its own colour stored (the same operation on the same stored values), so nothing is loaded twice and the
// backward update, which nobody reads, is not stored.  The expressions of the two separate launches in their order:
// the same bits.
// 150,000 triangles: 21.3 us as the two sweeps' code in turn, 18.4 so (12 us of bytes at the copy rate; the loads of a
// cell and its divisions and square roots are a serial chain, and all waves run in step).
template <int DIM, int MAXF, int RSCHEME>
__device__ __forceinline__ void lu_cell_bf(const LuArgs &a, const Params<double> &P, const bool roe, const int64_t t,
                                           const int64_t c) {
    constexpr int NV = DIM + 2;
    int32_t code[MAXF];
    double nrm[MAXF][DIM], q[MAXF][NV], dq[MAXF][NV], rr[MAXF], qc[NV], dqc[NV], s[NV];
#pragma unroll
    for (int k = 0; k < MAXF; k++) code[k] = a.nb[(int64_t)k * a.nc + t];
    const uint32_t finfo = a.finfo[t];
    ldq<NV>(a.dQ + c * NV, dqc);
    ldq<NV>(a.Q + c * NV, qc);
    double D = a.D[t];
#pragma unroll
    for (int k = 0; k < MAXF; k++) {
        const int64_t i = (int64_t)k * a.nc + t;
        if (code[k] != -2) {
#pragma unroll
            for (int d = 0; d < DIM; d++) nrm[k][d] = a.n[i * DIM + d];
        }
        if (code[k] >= 0 && (code[k] & 2)) {
            const int64_t o = code[k] >> 2;
            ldq<NV>(a.Q + o * NV, q[k]);
            ldq<NV>(a.dQ + o * NV, dq[k]);
            rr[k] = a.r[i];
        }
    }
#pragma unroll
    for (int j = 0; j < NV; j++) s[j] = 0;
    double qp[MAXF][NV];  // the neighbours' new states
#pragma unroll
    for (int k = 0; k < MAXF; k++) {
        if (!(code[k] >= 0 && (code[k] & 2))) continue;
#pragma unroll
        for (int j = 0; j < NV; j++) qp[k][j] = q[k][j] + dq[k][j];
        lu_offdiag<DIM>(q[k], qp[k], dq[k], nrm[k], rr[k], a.gamma, a.omega, s);
    }
    double dqn[NV], out[NV];
#pragma unroll
    for (int k = 0; k < NV; k++) dqn[k] = dqc[k] + s[k] / D;
#pragma unroll
    for (int k = 0; k < NV; k++) out[k] = qc[k] + dqn[k];
    stq<NV>(a.Qout + c * NV, out);
    const double p = lu_pressure<DIM>(out, a.gamma);
    if (!(out[0] > 0) || !(p > 0)) a.bad[0] = 1;
    // forward, from the new states
#pragma unroll
    for (int k = 0; k < MAXF; k++)
        if (code[k] >= 0 && !(code[k] & 2)) {  // the cell itself, through a periodic face
#pragma unroll
            for (int j = 0; j < NV; j++) qp[k][j] = out[j];
        }
    lu_solve<DIM, MAXF, RSCHEME>(P, roe, finfo, code, nrm, out, qp, s);
    double rsum = 0;
#pragma unroll
    for (int k = 0; k < MAXF; k++) {
        if (code[k] == -2) break;
        double r = lu_radius<DIM>(out, nrm[k], a.gamma);
        if (code[k] >= 0) r = fmax(r, lu_radius<DIM>(qp[k], nrm[k], a.gamma));
        a.r[(int64_t)k * a.nc + t] = r;
        rsum += r;
    }
    D = a.dscale * rsum;
    a.D[t] = D;
#pragma unroll
    for (int k = 0; k < NV; k++) dqn[k] = s[k] / D;
    stq<NV>(a.dQ + c * NV, dqn);
}

template <int DIM, int MAXF, int RSCHEME, bool BATCH = false>
__global__ __launch_bounds__(LU_BLOCK) void k_lu_sweep_bf(const LuArgs a, int64_t t0, int64_t n) {
    const int64_t l = block_id() * LU_BLOCK + threadIdx.x;
    if (l >= n) return;
    const int64_t t = t0 + l;
    lu_per_case<BATCH>(a, t, [&](const LuArgs &b, const Params<double> &P, bool roe) {
        lu_cell_bf<DIM, MAXF, RSCHEME>(b, P, roe, t, b.cells[t]);
    });
}

}  // namespace mstk
