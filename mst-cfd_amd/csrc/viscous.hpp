// Viscous flux: the intent of RhoSolver::updateViscid (rhoSolver/RhoSolver.cpp:371-429), which the
// reference cannot run as written and never adds to the residual (FLAGVISCID 0, include/CONST.h:14).
//   Q_f      the gradient kernel's face values (eta0 interpolation of the face's two cells; a
//            boundary face its cell; the last-interior-face quirk has eta0 = 1)         (:373-378)
//   W_f      = (u_1..u_dim, T) of Q_f, T = e / cv; on a wall face u = 0 (no-slip, adiabatic: the
//            cell's T), the wall the viscous branch of the convective boundary stands for (:160-163)
//   grad W_c = (1/V) sum_f W_f n_out                                                    (:380-391)
//   grad W_f = eta0 grad W_c0 + (1 - eta0) grad W_c1; boundary: grad W_c0                (:392-399)
//   tau_id   = mu (du_i/dx_d + du_d/dx_i) + lam (div u) delta_id                         (:401-413)
//   Fv[d]    = (0, tau_1d .. tau_dim,d, sum_i u_i tau_id + kappa dT/dx_d)                 (:415-419)
// and the face flux becomes G_f - sum_d n_d Fv[d] (the residual sums n_out . (F_conv - Fv)).
//   visc_cell  grad W_c of a cell from its slots' face states (the gradient kernel's slot-major incidence layout)
//   visc_face  grad W_f, W_f, tau, and G_f -= n . Fv
// Two routes, the same arithmetic:
//   patch route (patch tables, every boundary face of a known type): the gradient kernel forms grad W_c beside its
//     face states, from the same loads (k_grad_visc), and the patch kernel subtracts n . Fv from its fluxes in
//     registers: two kernels per stage and no face-flux array (order 1 and the mixed form: k_visc_grad first);
//   face route: k_visc_grad and k_visc_flux after the flux kernel, then the gather.
// All are FP64 gathers over the state (memory-bound, like the inviscid gradient and flux kernels; on meshes of
// a few hundred blocks bound by their latency and their number).
#pragma once
#include "kernels.hpp"

namespace mstk {

struct ViscArgs {
    int64_t nc, nf;
    const int32_t *__restrict__ inc_code;  // (neighbour << 1) | is_c1, -1 boundary, -2 empty
    const int32_t *__restrict__ ell;       // the same slots' (face << 1) | is_c1
    const int32_t *__restrict__ finfo;     // kind | (L/R mask << 4) per face
    const double *__restrict__ inc_w;      // eta0 of the face
    const double *__restrict__ inc_n;      // the cell's outward normal
    const double *__restrict__ vol;
    const int32_t *__restrict__ fc0;
    const int32_t *__restrict__ fc1;       // neighbour (interior / periodic partner cell), -1 boundary
    const double *__restrict__ feta;       // eta0 per face (quirk face: 1)
    const double *__restrict__ fn;         // c0 outward normal
    const double *__restrict__ Q;
    double *__restrict__ gw;               // [nc][dim + 1][dim]
    double *__restrict__ G;                // face fluxes, updated in place
    double mu, lam, kappa, cv;
};

template <int DIM>
__device__ __forceinline__ void visc_w(const double *q, double cv, double (&w)[DIM + 1]) {
    double ke = 0;
#pragma unroll
    for (int d = 0; d < DIM; d++) {
        w[d] = q[1 + d] / q[0];
        ke += q[1 + d] * q[1 + d];
    }
    w[DIM] = (q[DIM + 1] - 0.5 * ke / q[0]) / q[0] / cv;
}

// One slot's part of grad W_c: W of the face state qf (no-slip, adiabatic on a wall) times the outward normal
template <int DIM>
__device__ __forceinline__ void visc_slot(const double (&qf)[DIM + 2], bool wall, const double *n, double cv,
                                          double (&t)[DIM + 1][DIM]) {
    double w[DIM + 1];
    visc_w<DIM>(qf, cv, w);
    if (wall) {
#pragma unroll
        for (int d = 0; d < DIM; d++) w[d] = 0;
    }
#pragma unroll
    for (int k = 0; k < DIM + 1; k++)
#pragma unroll
        for (int d = 0; d < DIM; d++) t[k][d] += w[k] * n[d];
}

// face state of a slot: the gradient kernel's (eta interpolation; a boundary face its cell)
template <int NV>
__device__ __forceinline__ void visc_face_state(int32_t code, double eta, const double (&qc)[NV], const double (&qn)[NV],
                                                double (&qf)[NV]) {
#pragma unroll
    for (int k = 0; k < NV; k++) {
        if (code >= 0)
            qf[k] = (code & 1) ? eta * qn[k] + (1 - eta) * qc[k] : eta * qc[k] + (1 - eta) * qn[k];
        else
            qf[k] = qc[k];
    }
}

template <int DIM>
__device__ __forceinline__ bool visc_wall(const ViscArgs &a, int32_t code, int64_t i) {  // slot entry i
    return code == -1 && (a.finfo[a.ell[i] >> 1] & 15) == mst::KIND_WALL;
}

template <int DIM>
__device__ __forceinline__ void visc_store(const ViscArgs &a, int64_t c, double V, const double (&t)[DIM + 1][DIM]) {
#pragma unroll
    for (int k = 0; k < DIM + 1; k++)
#pragma unroll
        for (int d = 0; d < DIM; d++) a.gw[(c * (DIM + 1) + k) * DIM + d] = t[k][d] / V;
}

template <int DIM, int MAXF>
__global__ __launch_bounds__(BLOCK) void k_visc_grad(const ViscArgs a) {
    constexpr int NV = DIM + 2, NW = DIM + 1;
    const int64_t c = block_id() * BLOCK + threadIdx.x;
    if (c >= a.nc) return;
    double qc[NV], t[NW][DIM];
    ldq<NV>(a.Q + c * NV, qc);
#pragma unroll
    for (int k = 0; k < NW; k++)
#pragma unroll
        for (int d = 0; d < DIM; d++) t[k][d] = 0;
#pragma unroll
    for (int s = 0; s < MAXF; s++) {
        const int64_t i = (int64_t)s * a.nc + c;
        const int32_t code = a.inc_code[i];
        if (code == -2) break;
        double eta = 0, qn[NV], qf[NV], n[DIM];
        if (code >= 0) {
            eta = a.inc_w[i];
            ldq<NV>(a.Q + (int64_t)(code >> 1) * NV, qn);
        }
        visc_face_state<NV>(code, eta, qc, qn, qf);
#pragma unroll
        for (int d = 0; d < DIM; d++) n[d] = a.inc_n[i * DIM + d];
        visc_slot<DIM>(qf, visc_wall<DIM>(a, code, i), n, a.cv, t);
    }
    visc_store<DIM>(a, c, a.vol[c], t);
}

// k_grad (FP64) and k_visc_grad in one pass over a cell's slots
template <int DIM, int MAXF, int LIM>
__global__ __launch_bounds__(BLOCK) void k_grad_visc(const GradArgs<double> a, const ViscArgs v) {
    constexpr int NV = DIM + 2;
    const int64_t c = block_id() * BLOCK + threadIdx.x;
    if (c >= a.nc) return;
    GradIn<DIM, MAXF, double> in;
    double lgr[NV * DIM], dxs[MAXF][DIM], t[NV][DIM], ph[NV], w[DIM + 1][DIM];
    grad_fetch<DIM, MAXF, true, double>(a.Q, cell_view(a), c, c, in, dxs);
#pragma unroll
    for (int k = 0; k < DIM + 1; k++)
#pragma unroll
        for (int d = 0; d < DIM; d++) w[k][d] = 0;
#pragma unroll
    for (int s = 0; s < MAXF; s++) {
        if (in.code[s] == -2) break;
        double qf[NV];
        visc_face_state<NV>(in.code[s], in.eta[s], in.qc, in.qn[s], qf);
        visc_slot<DIM>(qf, visc_wall<DIM>(v, in.code[s], (int64_t)s * a.nc + c), in.n[s], v.cv, w);
    }
    visc_store<DIM>(v, c, in.vol, w);
    const int nfc = grad_eval<DIM, MAXF, LIM, double>(in, dxs, lgr, t, ph);
    grad_records<DIM, MAXF, double>(a, c, nfc, in.qc, lgr, dxs);
}

// G_f -= n . Fv of face f
template <int DIM>
__device__ __forceinline__ void visc_face(const ViscArgs &a, int64_t f, int kind, double (&gf)[DIM + 2]) {
    constexpr int NV = DIM + 2, NW = DIM + 1;
    const int64_t c0 = a.fc0[f], c1 = a.fc1[f];
    double q0[NV], qf[NV], g[NW][DIM];
    ldq<NV>(a.Q + c0 * NV, q0);
    if (c1 >= 0) {
        const double eta = a.feta[f];
        double q1[NV];
        ldq<NV>(a.Q + c1 * NV, q1);
#pragma unroll
        for (int k = 0; k < NV; k++) qf[k] = eta * q0[k] + (1 - eta) * q1[k];
#pragma unroll
        for (int k = 0; k < NW; k++)
#pragma unroll
            for (int d = 0; d < DIM; d++)
                g[k][d] = eta * a.gw[(c0 * NW + k) * DIM + d] + (1 - eta) * a.gw[(c1 * NW + k) * DIM + d];
    } else {
#pragma unroll
        for (int k = 0; k < NV; k++) qf[k] = q0[k];
#pragma unroll
        for (int k = 0; k < NW; k++)
#pragma unroll
            for (int d = 0; d < DIM; d++) g[k][d] = a.gw[(c0 * NW + k) * DIM + d];
    }
    double w[NW];
    visc_w<DIM>(qf, a.cv, w);
    if (c1 < 0 && kind == mst::KIND_WALL) {
#pragma unroll
        for (int d = 0; d < DIM; d++) w[d] = 0;
    }
    double div = 0;
#pragma unroll
    for (int d = 0; d < DIM; d++) div += g[d][d];
#pragma unroll
    for (int d = 0; d < DIM; d++) {
        const double nd = a.fn[f * DIM + d];
        double en = 0;
#pragma unroll
        for (int i = 0; i < DIM; i++) {
            double tau = a.mu * (g[i][d] + g[d][i]);
            if (i == d) tau += a.lam * div;
            gf[1 + i] -= nd * tau;
            en += w[i] * tau;
        }
        gf[NV - 1] -= nd * (en + a.kappa * g[DIM][d]);
    }
}

template <int DIM>
__global__ __launch_bounds__(BLOCK) void k_visc_flux(const ViscArgs a) {
    constexpr int NV = DIM + 2;
    const int64_t f = block_id() * BLOCK + threadIdx.x;
    if (f >= a.nf) return;
    double gf[NV];
    ldq<NV>(a.G + f * NV, gf);
    visc_face<DIM>(a, f, a.finfo[f] & 15, gf);
    stq<NV>(a.G + f * NV, gf);
}

// the patch kernel's addition to a face's flux
template <int DIM>
struct ViscFace {
    ViscArgs v;
    __device__ __forceinline__ void operator()(int64_t f, int kind, double (&g)[DIM + 2]) const { visc_face<DIM>(v, f, kind, g); }
};

}  // namespace mstk
