// kernels.hpp -- gfx950 kernels of the density-based explicit residual path.
//
// Per residual evaluation (one RK stage), on the context's stream:
//   k_grad    (order 2)  one lane per cell: Green-Gauss gradient + limiter -> the reconstructed state
//                        at each of the cell's faces (face-state records)
//   k_flux               one lane per face: its two records (or cell states), ghost state,
//                        dimension-split Roe/AUSM, G_f = sum_d n_d F_d  (c0 outward normal)
//   k_update             one lane per cell: R_c = sum +-G_f over its faces in a fixed order (no float
//                        atomics -> bit-reproducible), then the Euler / SSP-RK stage update
//   k_cell               (cell strategy, replaces k_flux + k_update) one lane per cell: solves its own
//                        faces' Riemann problems, sums them and updates, without a face-flux array
//   k_patch              (patch strategy, replaces k_flux + k_update) one block per patch of cells:
//                        solves the patch's faces once into LDS, then sums and updates per cell
//   k_fused              (fused strategy, replaces all of the above at order 2) the patch kernel with
//                        the gradients of the patch and its halo, and the face states, in the block
// plus k_cfl (CFL time step) and one-block reductions (k_finish) of per-block partials.
//
// Precision forms: T = double is the plain FP64 path (the reference's arithmetic); T = float is the
// mixed form: gradient, limiter and Riemann arithmetic in FP32 on an FP32 shadow of the state and FP32
// limited gradients; the per-axis fluxes are projected on the FP64 normals into FP64 face fluxes (so a
// uniform state cancels exactly around a closed cell), then a compensated FP64 gather and the FP64
// state update.  A periodic pair is one face (its second cell sees the partner face's centre), so the
// two sides always exchange exactly opposite fluxes.
#pragma once
#include <type_traits>

#include "device_common.hpp"
#include "prep.hpp"
#include "riemann.hpp"
#include "transfer.hpp"

// Minimum resident waves per SIMD requested from the compiler for the gradient and flux kernels (a
// register budget: 8 waves = 64 VGPRs, 6 = 80, 5 = 96); 1 leaves the choice to the compiler.
#ifndef MST_GRAD_WAVES
#define MST_GRAD_WAVES 1
#endif
#ifndef MST_FLUX_WAVES
#define MST_FLUX_WAVES 1
#endif
// Fused kernel: patch faces per lane whose ids, kinds and normals are fetched before the gradient
// phase (at least 1), and resident waves per SIMD for 2D FP32 triangles (0: the default of
// fused_waves).
#ifndef MST_FUSED_PF
#define MST_FUSED_PF 2
#endif
#ifndef MST_FUSED_WAVES32
#define MST_FUSED_WAVES32 0
#endif

namespace mstk {

// ------------------------------------------------------------------------------------ face flux
template <typename T>
struct FluxArgs {
    int64_t nf;
    const int32_t *__restrict__ fc0;
    const int32_t *__restrict__ fc1;
    const int32_t *__restrict__ finfo;  // kind | (L/R mask << 4)
    const double *__restrict__ fn;      // c0 outward normal
    const T *__restrict__ Q;            // cell states
    // order 2: the gradient kernel's reconstructed face states (NV values per incidence record) and
    // the records of each face's c0 and c1 sides (-1: none)
    const T *__restrict__ rec;
    const int32_t *__restrict__ frec0;
    const int32_t *__restrict__ frec1;
    double *__restrict__ G;
    Params<T> P;
};

// Inputs of face f's Riemann problem, every memory read of the face (RhoSolver::updateFaceFlux,
// RhoSolver.cpp:90-233, and updateFaceFlux2ndOrder, :234-369): the c0 outward normal, and X, Y = the
// c0- and c1-side states of an interior or periodic face (order 1 the cell states, order 2 the
// reconstructed states the gradient kernel stored for the face's two incidences), or X = the raw
// interior state and Y = its reconstructed face state for a boundary face, whose ghost combines the
// two as the reference does.  Everything is read by face index, so the lanes of the two cells of a
// face (cell strategy) load and then compute bit-identical states.
// s0, s1: the face's entries of the side arrays (frec0, frec1 at order 2, else fc0, fc1), fetched before.
template <int DIM, bool SECOND, typename T>
__device__ __forceinline__ void face_load(const FluxArgs<T> &a, int64_t f, int kind, int32_t s0, int32_t s1,
                                          double (&n64)[DIM], T (&X)[DIM + 2], T (&Y)[DIM + 2]) {
    constexpr int NV = DIM + 2;
#pragma unroll
    for (int d = 0; d < DIM; d++) n64[d] = a.fn[f * DIM + d];
    if (kind == mst::KIND_INTERIOR || kind == mst::KIND_PERIODIC) {
        const T *src = SECOND ? a.rec : a.Q;
        ldq<NV>(src + (int64_t)s0 * NV, X);
        ldq<NV>(src + (int64_t)s1 * NV, Y);
        return;
    }
    ldq<NV>(a.Q + (int64_t)(SECOND ? a.fc0[f] : s0) * NV, X);
    if constexpr (SECOND) {
        ldq<NV>(a.rec + (int64_t)s0 * NV, Y);
    } else {
#pragma unroll
        for (int k = 0; k < NV; k++) Y[k] = X[k];
    }
}

// The same with the indices loaded here: ahead of the branch on the kind (c0's is fetched without waiting for the kind)
// or inside it.  Neither is always the better one; measured in microseconds, ahead / inside, on 820,000 triangles and
// 500,000 quadrilaterals (2D), 663,552 tetrahedra (3D), and batches of 300,000 triangles, 240,000 quadrilaterals and
// 384,000 tetrahedra (kb_, per step):
//   order 1: k_flux 17.4 / 18.5 (FP64), 13.0 / 13.6 (FP32); kb_flux 517 / 511; kb_patch 49.0 / 50.3
//   order 2: k_flux 23.6 / 22.0 (FP64), 33.5 / 31.4 (FP32, 3D); kb_flux 490 / 466; kb_patch 171 / 165
//   cells, FP64 2D: k_cell 38.2 / 40.3, 43.0 / 43.6 (orders 1, 2); kb_cell 375 / 402, 531 / 554
//   cells, FP32 2D: k_cell 28.1 / 27.3, 33.7 / 32.2; kb_cell 357 / 337, 486 / 459
//   cells, 3D: order 1 k_cell 46.3 / 48.3 (FP32), kb_cell 669 / 654; order 2 FP64 k_cell 92.7 / 87.5, kb_cell 1169 / 1037
template <int DIM, bool SECOND, typename T, bool AHEAD = !SECOND>
__device__ __forceinline__ void face_load(const FluxArgs<T> &a, int64_t f, int kind, double (&n64)[DIM],
                                          T (&X)[DIM + 2], T (&Y)[DIM + 2]) {
    constexpr int NV = DIM + 2;
    const bool two = kind == mst::KIND_INTERIOR || kind == mst::KIND_PERIODIC;
    if constexpr (AHEAD) {
        const int32_t s0 = SECOND ? a.frec0[f] : a.fc0[f], s1 = two ? (SECOND ? a.frec1[f] : a.fc1[f]) : -1;
        face_load<DIM, SECOND, T>(a, f, kind, s0, s1, n64, X, Y);
    } else {
#pragma unroll
        for (int d = 0; d < DIM; d++) n64[d] = a.fn[f * DIM + d];
        if (two) {
            if constexpr (SECOND) {
                ldq<NV>(a.rec + (int64_t)a.frec0[f] * NV, X);
                ldq<NV>(a.rec + (int64_t)a.frec1[f] * NV, Y);
            } else {
                ldq<NV>(a.Q + (int64_t)a.fc0[f] * NV, X);
                ldq<NV>(a.Q + (int64_t)a.fc1[f] * NV, Y);
            }
            return;
        }
        ldq<NV>(a.Q + (int64_t)a.fc0[f] * NV, X);
        if constexpr (SECOND) {
            ldq<NV>(a.rec + (int64_t)a.frec0[f] * NV, Y);
        } else {
#pragma unroll
            for (int k = 0; k < NV; k++) Y[k] = X[k];
        }
    }
}

// face_load's AHEAD in the cell kernels
template <int DIM, bool SECOND, typename T>
constexpr bool cell_ahead() {
    return DIM == 2 ? std::is_same<T, double>::value : !SECOND;
}

// Riemann left (A: c0 side) and right (B: c1 side or ghost) states from face_load's inputs; registers only
template <int DIM, typename T>
__device__ __forceinline__ void face_bc(const Params<T> &P, int kind, const T *n, const T (&X)[DIM + 2],
                                        const T (&Rc)[DIM + 2], T (&A)[DIM + 2], T (&B)[DIM + 2]) {
    constexpr int NV = DIM + 2;
    if (kind == mst::KIND_INTERIOR || kind == mst::KIND_PERIODIC) {
#pragma unroll
        for (int k = 0; k < NV; k++) {
            A[k] = X[k];
            B[k] = Rc[k];
        }
        return;
    }
    if (kind == mst::KIND_WALL) {  // RhoSolver.cpp:142-179 / 285-319
#pragma unroll
        for (int k = 0; k < NV; k++) A[k] = B[k] = Rc[k];
        if (P.noslip) {  // viscous wall: the ghost's momentum is the interior's negated (:160-163 / 300-303)
#pragma unroll
            for (int d = 0; d < DIM; d++) B[1 + d] = -A[1 + d];
        } else {
            reflect<DIM>(B, A, n);
        }
    } else if (kind == mst::KIND_SYMMETRY) {  // :184-211 / 322-350 (A keeps the raw interior state)
#pragma unroll
        for (int k = 0; k < NV; k++) {
            A[k] = X[k];
            B[k] = Rc[k];
        }
        reflect<DIM>(B, A, n);
    } else if (kind == mst::KIND_INLET) {  // :121-137 / 265-281
#pragma unroll
        for (int k = 0; k < NV; k++) {
            A[k] = Rc[k];
            B[k] = P.qin[k];
        }
    } else {  // outlet :216-226 / 353-363 (A keeps the raw interior state)
#pragma unroll
        for (int k = 0; k < NV; k++) {
            A[k] = X[k];
            B[k] = Rc[k];
        }
    }
}

// scheme chosen per call (a batch mixes Roe and AUSM cases) instead of per instantiation
constexpr int SCHEME_RUNTIME = -1;

// G_f (c0 outward) from face_load's inputs: ghost/boundary states, dimension-split Riemann solves,
// FP64 projection
template <int DIM, int SCHEME, typename T>
__device__ __forceinline__ void face_solve(const Params<T> &P, bool roe, int kind, int mask, const double (&n64)[DIM],
                                           const T (&X)[DIM + 2], const T (&Y)[DIM + 2], double (&g)[DIM + 2]) {
    constexpr int NV = DIM + 2;
    T n[DIM], A[NV], B[NV];
#pragma unroll
    for (int d = 0; d < DIM; d++) n[d] = (T)n64[d];
    face_bc<DIM, T>(P, kind, n, X, Y, A, B);
    if constexpr (SCHEME == SCHEME_RUNTIME) {
        if (roe)
            riemann_face<DIM, MST_SCHEME_ROE, T>(A, B, n64, mask, P, g);
        else
            riemann_face<DIM, MST_SCHEME_AUSM, T>(A, B, n64, mask, P, g);
    } else {
        riemann_face<DIM, SCHEME, T>(A, B, n64, mask, P, g);
    }
}

// G_f of one face: load, then solve
template <int DIM, int SCHEME, bool SECOND, typename T, bool AHEAD = !SECOND>
__device__ __forceinline__ void face_flux(const FluxArgs<T> &a, int64_t f, int kind, int mask, double (&g)[DIM + 2]) {
    constexpr int NV = DIM + 2;
    double n64[DIM];
    T X[NV], Y[NV];
    face_load<DIM, SECOND, T, AHEAD>(a, f, kind, n64, X, Y);
    face_solve<DIM, SCHEME, T>(a.P, SCHEME == MST_SCHEME_ROE, kind, mask, n64, X, Y, g);
}

// face strategy: one lane per face writes G_f (RhoSolver::updateFaceFlux[2ndOrder])
template <int DIM, int SCHEME, bool SECOND, typename T>
__global__ __launch_bounds__(BLOCK, MST_FLUX_WAVES) void k_flux(const FluxArgs<T> a) {
    constexpr int NV = DIM + 2;
    const int64_t f = block_id() * BLOCK + threadIdx.x;
    if (f >= a.nf) return;
    const int info = a.finfo[f];
    const int kind = info & 15, mask = info >> 4;
    double g[NV];
    if (kind >= mst::KIND_NONE) {  // unknown type (zero flux) or the merged half of a periodic pair
#pragma unroll
        for (int k = 0; k < NV; k++) g[k] = 0;
    } else {
        face_flux<DIM, SCHEME, SECOND, T>(a, f, kind, mask, g);
    }
    stq<NV>(a.G + f * NV, g);
}

// ------------------------------------------------------------------------------------ gradient + limiter
// The gradient's volume input: FP64 the cell volume, FP32 its reciprocal (float) frcp(V), computed
// once per mesh (k_recip_vol) with the arithmetic the FP64 form applies to V.
template <typename T>
using GradVol = typename std::conditional<std::is_same<T, float>::value, float, double>::type;

template <typename T>
struct GradArgs {
    int64_t nc;
    // incidence layout (slot-major, index s*nc + c): (neighbour << 1) | is_c1, -1 boundary face, -2
    // empty slot; FP64: eta of the face, FP32: the difference-form weight; the cell's outward normal;
    // offset x_f - x_c (partner face centre on the c1 side of a periodic pair).  Every load but the
    // neighbour states is coalesced.
    const int32_t *__restrict__ inc_code;
    const T *__restrict__ inc_w;
    const T *__restrict__ inc_n;
    const T *__restrict__ inc_dx;
    const T *__restrict__ Q;
    const GradVol<T> *__restrict__ vol;
    T *__restrict__ rec;  // out: reconstructed face state of every incidence, Q_c + phi grad Q . dx
    double *__restrict__ graw;
    double *__restrict__ phi;
};

// RhoSolver::updateGradFlux (RhoSolver.cpp:430-454) fused with the (new) per-cell limiter.
// FP64: grad = (1/V) sum_f Q_f n_out as the reference, Q_f = eta Q_c0 + (1-eta) Q_c1; FP32: the same
// sum written with differences, (1/V) sum_f w_f (Q_nb - Q_c) n_out (w = 1-eta on the c0 side, eta on
// the c1 side), equal because the outward normals of a closed cell sum to zero, and free of the
// cancellation an FP32 sum of whole states would suffer.
// Where a cell's incidence geometry lives: slot s of the cell at geometry index g is entry s * stride + g
// of code / w / n / dx (n and dx DIM-wide), its volume vol[g].  The cell-ordered arrays have g = c and
// stride nc; a patch's halo reads a packed copy in halo order.
template <typename T>
struct IncView {
    const int32_t *code;
    const T *w, *n, *dx;
    const GradVol<T> *vol;
    int64_t stride;
};

// FP32 in 3D: the difference-form weight is folded into the incidence normal (the FP32 normal array
// holds (float)(w n), k_weighted_normals) and the weights are not read.  The FP64 form sums whole face
// states, which needs the weight alone; 2D FP32 keeps them apart because the 2D fused kernel takes its
// normals from its faces'.
template <int DIM, typename T>
constexpr bool grad_wn() {
    return DIM == 3 && std::is_same<T, float>::value;
}

// The memory reads of one cell's limited gradient.  grad_fetch issues every read before the first is
// used: the slots' codes, weights, normals (unless NRM is false: the caller supplies them) and offsets
// and the volume (independent of each other), then all the neighbour states (an empty or boundary
// slot loads the cell's own state, unused).  That is two dependent load rounds per cell instead of
// one or two per slot.
template <int DIM, int MAXF, typename T>
struct GradIn {
    int32_t code[MAXF];
    T eta[MAXF], n[MAXF][DIM];
    T qc[DIM + 2], qn[MAXF][DIM + 2];
    GradVol<T> vol;
};

template <int DIM, int MAXF, bool NRM, typename T>
__device__ __forceinline__ void grad_fetch(const T *__restrict__ Q, const IncView<T> &a, const int64_t g,
                                           const int64_t c, GradIn<DIM, MAXF, T> &in, T (&dxs)[MAXF][DIM]) {
    constexpr int NV = DIM + 2;
#pragma unroll
    for (int s = 0; s < MAXF; s++) {
        const int64_t i = (int64_t)s * a.stride + g;
        in.code[s] = a.code[i];
        if constexpr (!grad_wn<DIM, T>()) in.eta[s] = a.w[i];
#pragma unroll
        for (int d = 0; d < DIM; d++) {
            if constexpr (NRM) in.n[s][d] = a.n[i * DIM + d];
            dxs[s][d] = a.dx[i * DIM + d];
        }
    }
    in.vol = a.vol[g];
    ldq<NV>(Q + c * NV, in.qc);
#pragma unroll
    for (int s = 0; s < MAXF; s++) {
        const int64_t nb = in.code[s] >= 0 ? (int64_t)(in.code[s] >> 1) : c;
        ldq<NV>(Q + nb * NV, in.qn[s]);
    }
}

// The limited gradient of a cell from its fetched inputs; returns the number of used slots.
template <int DIM, int MAXF, int LIM, typename T>
__device__ __forceinline__ int grad_eval(const GradIn<DIM, MAXF, T> &in, const T (&dxs)[MAXF][DIM],
                                         T (&lgr)[(DIM + 2) * DIM], T (&t)[DIM + 2][DIM], T (&ph)[DIM + 2]) {
    constexpr int NV = DIM + 2;
    constexpr bool F32 = std::is_same<T, float>::value;
    const T(&qc)[NV] = in.qc;
    T qmax[NV], qmin[NV];
#pragma unroll
    for (int k = 0; k < NV; k++) {
        qmax[k] = qmin[k] = qc[k];
#pragma unroll
        for (int d = 0; d < DIM; d++) t[k][d] = 0;
    }
    int nfc = 0;
#pragma unroll
    for (int s = 0; s < MAXF; s++) {
        if (in.code[s] == -2) continue;  // empty slots are the last ones of the cell
        const bool interior = in.code[s] >= 0;
        const bool is1 = interior && (in.code[s] & 1);
        T qf[NV];
        if (interior) {
            if constexpr (F32) {
#pragma unroll
                for (int k = 0; k < NV; k++)
                    qf[k] = grad_wn<DIM, T>() ? in.qn[s][k] - qc[k] : in.eta[s] * (in.qn[s][k] - qc[k]);
            } else {
#pragma unroll
                for (int k = 0; k < NV; k++)
                    qf[k] = is1 ? in.eta[s] * in.qn[s][k] + (1 - in.eta[s]) * qc[k] : in.eta[s] * qc[k] + (1 - in.eta[s]) * in.qn[s][k];
            }
#pragma unroll
            for (int k = 0; k < NV; k++) {
                qmax[k] = fmax(qmax[k], in.qn[s][k]);
                qmin[k] = fmin(qmin[k], in.qn[s][k]);
            }
        } else {
#pragma unroll
            for (int k = 0; k < NV; k++) qf[k] = F32 ? T(0) : qc[k];
        }
#pragma unroll
        for (int k = 0; k < NV; k++)
#pragma unroll
            for (int d = 0; d < DIM; d++) t[k][d] += qf[k] * in.n[s][d];
        nfc = s + 1;
    }
    T iV;
    if constexpr (F32)
        iV = in.vol;
    else
        iV = frcp(in.vol);
#pragma unroll
    for (int k = 0; k < NV; k++) {
        ph[k] = 1;
#pragma unroll
        for (int d = 0; d < DIM; d++) t[k][d] *= iV;
    }
    if constexpr (LIM != MST_LIM_NONE) {
        // Phi = min(1, min_f psi(r_f)) = min(1, psi(min_f r_f)) since psi is increasing: the smallest
        // ratio r = |a|/|delta| is tracked as a fraction (bn/bd) and psi is applied once per field
        T bn[NV], bd[NV];
#pragma unroll
        for (int k = 0; k < NV; k++) {
            bn[k] = 1;
            bd[k] = 0;  // "infinite" ratio: no face limits
        }
#pragma unroll
        for (int s = 0; s < MAXF; s++) {
            if (s >= nfc) break;
#pragma unroll
            for (int k = 0; k < NV; k++) {
                T delta = t[k][0] * dxs[s][0] + t[k][1] * dxs[s][1];
                if constexpr (DIM == 3) delta += t[k][2] * dxs[s][2];
                const T eps = T(1e-12) * (fabs(qmax[k]) + fabs(qmin[k]));
                const T ext = delta > 0 ? qmax[k] : qmin[k];
                const T an = fabs(ext - qc[k]), ad = fabs(delta);
                if (fabs(delta) > eps && (bd[k] == T(0) || an * bd[k] < bn[k] * ad)) {
                    bn[k] = an;
                    bd[k] = ad;
                }
            }
        }
#pragma unroll
        for (int k = 0; k < NV; k++) {
            if (bd[k] == T(0)) continue;
            if constexpr (LIM == MST_LIM_MINMOD)
                ph[k] = bn[k] < bd[k] ? fdiv(bn[k], bd[k]) : T(1);
            else
                ph[k] = fmin(T(1), fdiv(T(2) * bn[k], bd[k] + bn[k]));  // (r+|r|)/(1+|r|) at r = bn/bd >= 0
        }
    }
#pragma unroll
    for (int k = 0; k < NV; k++)
#pragma unroll
        for (int d = 0; d < DIM; d++) lgr[k * DIM + d] = ph[k] * t[k][d];
    return nfc;
}

template <int DIM, int MAXF, int LIM, typename T>
__device__ __forceinline__ int grad_limited(const T *__restrict__ Q, const IncView<T> &a, const int64_t g,
                                           const int64_t c, T (&qc)[DIM + 2], T (&lgr)[(DIM + 2) * DIM],
                                           T (&dxs)[MAXF][DIM], T (&t)[DIM + 2][DIM], T (&ph)[DIM + 2]) {
    GradIn<DIM, MAXF, T> in;
    grad_fetch<DIM, MAXF, true, T>(Q, a, g, c, in, dxs);
    const int nfc = grad_eval<DIM, MAXF, LIM, T>(in, dxs, lgr, t, ph);
#pragma unroll
    for (int k = 0; k < DIM + 2; k++) qc[k] = in.qc[k];
    return nfc;
}

template <typename T>
__device__ __forceinline__ IncView<T> cell_view(const GradArgs<T> &a) {
    return IncView<T>{a.inc_code, a.inc_w, a.inc_n, a.inc_dx, a.vol, a.nc};
}

// reconstructed states at the cell's faces (RhoSolver.cpp:250,254 with the limiter), one record per
// incidence, coalesced over the cells of a slot
template <int DIM, int MAXF, typename T>
__device__ __forceinline__ void grad_records(const GradArgs<T> &a, const int64_t c, int nfc, const T (&qc)[DIM + 2],
                                             const T (&lgr)[(DIM + 2) * DIM], const T (&dxs)[MAXF][DIM]) {
    constexpr int NV = DIM + 2;
#pragma unroll
    for (int s = 0; s < MAXF; s++) {
        if (s >= nfc) break;
        T q[NV];
#pragma unroll
        for (int k = 0; k < NV; k++) q[k] = qc[k];
        recon<DIM>(q, lgr, dxs[s]);
        stq<NV>(a.rec + ((int64_t)s * a.nc + c) * NV, q);
    }
}

// grad_limited, then the cell's face records and the optional raw gradient / limiter outputs
template <int DIM, int MAXF, int LIM, typename T>
__device__ __forceinline__ void grad_cell(const GradArgs<T> &a, const int64_t c) {
    constexpr int NV = DIM + 2;
    T qc[NV], lgr[NV * DIM], dxs[MAXF][DIM], t[NV][DIM], ph[NV];
    const int nfc = grad_limited<DIM, MAXF, LIM, T>(a.Q, cell_view(a), c, c, qc, lgr, dxs, t, ph);
    grad_records<DIM, MAXF, T>(a, c, nfc, qc, lgr, dxs);
    if (a.graw) {
#pragma unroll
        for (int k = 0; k < NV; k++)
#pragma unroll
            for (int d = 0; d < DIM; d++) a.graw[c * NV * DIM + k * DIM + d] = (double)t[k][d];
    }
    if (a.phi) {
#pragma unroll
        for (int k = 0; k < NV; k++) a.phi[c * NV + k] = (double)ph[k];
    }
}

template <int DIM, int MAXF, int LIM, typename T>
__global__ __launch_bounds__(BLOCK, MST_GRAD_WAVES) void k_grad(const GradArgs<T> a) {
    const int64_t c = block_id() * BLOCK + threadIdx.x;
    if (c < a.nc) grad_cell<DIM, MAXF, LIM, T>(a, c);
}

// ------------------------------------------------------------------------------------ gather + update
struct UpdArgs {
    int64_t nc;
    const int32_t *__restrict__ ell;
    const double *__restrict__ G;
    const double *__restrict__ Qs;
    const double *__restrict__ Qn;
    const double *__restrict__ vol;
    const double *__restrict__ sh;  // half sums of |S_d| per cell (CFL)
    const double *__restrict__ dt;  // [0] dt of this stage, when dt_n == 0; else it is the minimum of
    const double *__restrict__ dt_part;  // dt_part[0..dt_n), the previous step's block minima
    int dt_n;
    double ca, cb;
    int stage0;
    // mixed form (FP32 kernels read only the FP32 shadow, so an intermediate stage's FP64 state is
    // needed only by the next stage's update): pre = Qs holds the stage's combination
    // ca Q^n + cb Q_s, and the stage computes Qs - cb dt/V R; wa, wb (wb != 0 on a stage with a
    // successor) = that successor's coefficients: Qout receives wa Q^n + wb Q_{s+1} and Qout32 the
    // shadow of Q_{s+1} itself
    int pre;
    double wa, wb;
    int maxf;       // ELL slots (cell strategy)
    int l2, dtred;  // cell strategy: reduce |R/V|^2 / the CFL time step in this launch
    int check;      // flag rho <= 0 / p <= 0 / NaN in the output (the state that ends a step)
    double gamma, cfl;
    double *__restrict__ Qout;
    float *__restrict__ Qout32;     // FP32 shadow of Qout (mixed form), else null
    double *__restrict__ R;
    double *__restrict__ part_l2;   // per-block partial sums of (R/V)^2: [field][block]
    double *__restrict__ part_dt;   // per-block minimum CFL time step
    int *__restrict__ bad;          // set to 1 when an updated state is not physical
};

// The coefficients of one stage update (host side; copied into UpdArgs): Q_out = ca Q^n + cb (Q_s -
// dt/V R), or Q_s - dt/V R on the first stage (stage0).  Mixed form: pre = Q_s already holds ca Q^n +
// cb Q_s, and (wa, wb), wb != 0 on a stage with a successor, are the successor's coefficients.
struct Stage {
    double ca = 0, cb = 1;
    int stage0 = 1;
    int pre = 0;
    double wa = 0, wb = 0;
};

__host__ inline void set_stage(UpdArgs &a, const Stage &sg) {
    a.ca = sg.ca;
    a.cb = sg.cb;
    a.stage0 = sg.stage0;
    a.pre = sg.pre;
    a.wa = sg.wa;
    a.wb = sg.wb;
}

// mode bits: UPD_STAGE writes the stage update (else only R), UPD_L2 reduces |R/V|^2,
// UPD_DT reduces the CFL time step of the updated state (for the next step); UPD_CHECK (a runtime
// flag, not a kernel variant) checks the output for a non-physical state.  Intermediate RK stages
// are not checked: an SSP stage may leave the admissible set and the step's final combination
// return to it (the reference checks nothing at all).
enum { UPD_RESIDUAL = 0, UPD_STAGE = 1, UPD_L2 = 2, UPD_DT = 4, UPD_CHECK = 8 };

// Block-level reduction of W values: sums, or a min when MIN is set; thread 0..W-1 of the block write
// the results.  A fixed xor butterfly inside each wave (every lane ends with the wave's value), then
// the waves' values in wave order: one barrier after the first instead of one per tree level.  The
// per-block partials are combined by k_finish in block order, so every reduction is bit-reproducible
// (no float atomics, no cross-block fences).
// sh: at least W * NT / 64 doubles of LDS.  The first barrier also orders the block's earlier readers
// of sh before the writes, so a kernel may pass LDS it has finished with.
template <int W, bool MIN, int NT = BLOCK>
__device__ __forceinline__ void block_partial(double (&v)[W], double *__restrict__ out, int64_t stride, double *sh) {
    constexpr int NW = NT / 64;
    static_assert(NT % 64 == 0, "blocks are whole waves");
#pragma unroll
    for (int k = 0; k < W; k++)
#pragma unroll
        for (int m = 32; m > 0; m >>= 1) {
            const double y = __shfl_xor(v[k], m, 64);
            v[k] = MIN ? fmin(v[k], y) : v[k] + y;
        }
    __syncthreads();  // a previous call's readers of sh are done (persistent loops reuse it)
    if ((threadIdx.x & 63) == 0) {
#pragma unroll
        for (int k = 0; k < W; k++) sh[k * NW + (threadIdx.x >> 6)] = v[k];
    }
    __syncthreads();
    if ((int)threadIdx.x < W) {
        double s = sh[threadIdx.x * NW];
#pragma unroll
        for (int w = 1; w < NW; w++) s = MIN ? fmin(s, sh[threadIdx.x * NW + w]) : s + sh[threadIdx.x * NW + w];
        out[threadIdx.x * stride] = s;
    }
}
template <int W, bool MIN, int NT = BLOCK>
__device__ __forceinline__ void block_partial(double (&v)[W], double *__restrict__ out, int64_t stride) {
    __shared__ double sh[W * (NT / 64)];
    block_partial<W, MIN, NT>(v, out, stride, sh);
}

template <int DIM>
__device__ __forceinline__ double local_dt(const double *q, const double *shc, double V, double gamma, double cfl) {
    constexpr int NV = DIM + 2;
    const double ir = 1.0 / q[0];  // one division: the velocities and the pressure multiply by 1/rho
    double ke = 0;
#pragma unroll
    for (int k = 1; k <= DIM; k++) ke += q[k] * q[k];
    const double p = (q[NV - 1] - 0.5 * ke * ir) * (gamma - 1);
    const double snd = sqrt(gamma * p * ir);
    double lam = 0;
#pragma unroll
    for (int d = 0; d < DIM; d++) lam += (fabs(q[1 + d] * ir) + snd) * shc[d];
    const double v = cfl * V / lam;
    return v == v ? v : -1.0;  // a NaN state reports a negative time step
}

// add one face flux to a cell's residual; the mixed form (F32) keeps the rounding error of every
// addition in a Neumaier compensation term
template <int NV, bool F32>
__device__ __forceinline__ void accumulate(double (&r)[NV], double (&cmp)[NV], const double (&g)[NV], bool neg) {
#pragma unroll
    for (int k = 0; k < NV; k++) {
        const double x = neg ? -g[k] : g[k];
        if constexpr (F32) {
            const double t = r[k] + x;
            cmp[k] += fabs(r[k]) >= fabs(x) ? (r[k] - t) + x : (x - t) + r[k];
            r[k] = t;
        } else {
            r[k] += x;
        }
    }
}

// Stage update of cell c from its residual r (RhoSolver::solve, RhoSolver.cpp:57-66, in SSP-RK stage
// form) and the non-physical-state flag; red[] receives this cell's |R/V|^2 (L2) and CFL time step (DT)
// the inputs of cell c's stage update that do not depend on its residual: volume, stage state and
// (after the first stage) the state at the start of the step
template <int NV>
struct StageIn {
    double V, qs[NV], qn[NV];
    double sh[NV - 2];  // the cell's CFL half-sums, on a launch that reduces the time step
};

// The time step of the stage, the same in every lane; the whole wave must be active.  Each wave takes the minimum of
// the block minima itself (a minimum does not depend on the order), with its loads in flight together: on
// meshes of few blocks that costs less than a launch between two steps (STEP_DT_MAX in solver.hip).
__device__ __forceinline__ double stage_dt(const UpdArgs &a) {
    if (a.dt_n == 0) return a.dt[0];
    double v = INFINITY;
    for (int i = threadIdx.x & 63; i < a.dt_n; i += 8 * 64) {
        double x[8];
#pragma unroll
        for (int u = 0; u < 8; u++) x[u] = a.dt_part[i + 64 * u < a.dt_n ? i + 64 * u : i];
#pragma unroll
        for (int u = 0; u < 8; u++) v = fmin(v, x[u]);
    }
    for (int m = 32; m > 0; m >>= 1) v = fmin(v, __shfl_xor(v, m, 64));
    return __hiloint2double(__builtin_amdgcn_readfirstlane(__double2hiint(v)),  // (a scalar: no vector registers)
                            __builtin_amdgcn_readfirstlane(__double2loint(v)));
}

template <int NV, bool F32>
__device__ __forceinline__ void stage_load(const UpdArgs &a, int64_t c, StageIn<NV> &in) {
    in.V = a.vol[c];
    ldq<NV>(a.Qs + c * NV, in.qs);
    if (a.dtred)
#pragma unroll
        for (int d = 0; d < NV - 2; d++) in.sh[d] = a.sh[c * (NV - 2) + d];
    // Q^n: the stage combination (FP64 form), or the successor's combination after the first stage
    const bool pre = F32 && a.pre;
    if (!a.stage0 && (!pre || a.wb != 0)) ldq<NV>(a.Qn + c * NV, in.qn);
}

template <int NV, bool F32>
__device__ __forceinline__ void stage_cell(const UpdArgs &a, int64_t c, double dt, const StageIn<NV> &in, const double (&r)[NV],
                                           double (&red)[NV + 1], const bool L2, const bool DT) {
    constexpr int DIM = NV - 2;
    const double V = in.V;
    const double dtv = dt / V;
    const bool pre = F32 && a.pre;
    double out[NV];
    if (pre) {  // Qs = ca Q^n + cb Q_s (cb = 1 on the first stage: the same arithmetic as below)
        const double h = a.cb * dtv;
#pragma unroll
        for (int k = 0; k < NV; k++) out[k] = in.qs[k] - h * r[k];
    } else if (a.stage0) {
#pragma unroll
        for (int k = 0; k < NV; k++) out[k] = in.qs[k] - dtv * r[k];
    } else {
#pragma unroll
        for (int k = 0; k < NV; k++) out[k] = a.ca * in.qn[k] + a.cb * (in.qs[k] - dtv * r[k]);
    }
    if (pre && a.wb != 0) {
        double w[NV];
#pragma unroll
        for (int k = 0; k < NV; k++) w[k] = a.wa * (a.stage0 ? in.qs[k] : in.qn[k]) + a.wb * out[k];
        stq<NV>(a.Qout + c * NV, w);
    } else {
        stq<NV>(a.Qout + c * NV, out);
    }
    if constexpr (F32) stq<NV>(a.Qout32 + c * NV, out);
    if (a.check) {
        double ke = 0;
#pragma unroll
        for (int k = 1; k < NV - 1; k++) ke += out[k] * out[k];
        const double p = (out[NV - 1] - 0.5 * ke / out[0]) * (a.gamma - 1);
        if (!(out[0] > 0) || !(p > 0)) a.bad[0] = 1;
    }
    if (!(dt > 0)) a.bad[0] = 1;  // a NaN or non-physical state gave no positive CFL time step
    if (L2) {
        const double iV = frcp(V);
#pragma unroll
        for (int k = 0; k < NV; k++) {
            const double x = r[k] * iV;
            red[k] += x * x;
        }
    }
    if (DT) red[NV] = fmin(red[NV], local_dt<DIM>(out, in.sh, V, a.gamma, a.cfl));
}

template <int NV, bool F32>
__device__ __forceinline__ void stage_cell(const UpdArgs &a, int64_t c, double dt, const double (&r)[NV],
                                           double (&red)[NV + 1], const bool L2, const bool DT) {
    StageIn<NV> in;
    stage_load<NV, F32>(a, c, in);
    stage_cell<NV, F32>(a, c, dt, in, r, red, L2, DT);
}

// stage_cell for the lanes of one block, then the block's partials of |R/V|^2 and the CFL time step.
// Every lane of the block must call it (block-level reductions).
// lds (DYN): NV * BLOCK / 64 doubles of the kernel's dynamic LDS for the reductions, in place of a static
// array (which would count against every block's LDS for the whole kernel).
// dt: stage_dt (unused by a residual-only evaluation).  in: the inputs when they are loaded already.
template <int NV, bool STAGE, bool F32, int NT = BLOCK, bool DYN = false>
__device__ __forceinline__ void stage_tail(const UpdArgs &a, int64_t c, bool valid, double dt, const double (&r)[NV],
                                           int64_t blk, const bool L2, const bool DT, const StageIn<NV> *in = nullptr,
                                           double *lds = nullptr) {
    if constexpr (!STAGE) {
        if (valid) stq<NV>(a.R + c * NV, r);
        if (L2) {  // residual-only evaluation with its norms (the implicit steady driver)
            double v[NV];
#pragma unroll
            for (int k = 0; k < NV; k++) v[k] = 0;
            if (valid) {
                const double iV = frcp(a.vol[c]);
#pragma unroll
                for (int k = 0; k < NV; k++) {
                    const double x = r[k] * iV;
                    v[k] = x * x;
                }
            }
            block_partial<NV, false, NT>(v, a.part_l2 + blk, gridDim.x);
        }
        return;
    } else {
        double red[NV + 1];
#pragma unroll
        for (int k = 0; k < NV; k++) red[k] = 0;
        red[NV] = INFINITY;
        if (valid) {
            if (in)
                stage_cell<NV, F32>(a, c, dt, *in, r, red, L2, DT);
            else
                stage_cell<NV, F32>(a, c, dt, r, red, L2, DT);
        }
        if (L2) {  // uniform over the launch
            double v[NV];
#pragma unroll
            for (int k = 0; k < NV; k++) v[k] = red[k];
            if constexpr (DYN)
                block_partial<NV, false, NT>(v, a.part_l2 + blk, gridDim.x, lds);
            else
                block_partial<NV, false, NT>(v, a.part_l2 + blk, gridDim.x);
        }
        if (DT) {
            double v[1] = {red[NV]};
            if constexpr (DYN)
                block_partial<1, true, NT>(v, a.part_dt + blk, 1, lds);
            else
                block_partial<1, true, NT>(v, a.part_dt + blk, 1);
        }
    }
}

// Face strategy, second kernel: RhoSolver::solve gather + update (RhoSolver.cpp:45-68).  R_c sums +-G_f
// over the cell's faces in a fixed order (no float atomics -> bit-reproducible).
template <int NV, int MAXF, int MODE, bool F32>
__global__ __launch_bounds__(BLOCK) void k_update(const UpdArgs a) {
    const int64_t blk = block_id();
    const int64_t c = blk * BLOCK + threadIdx.x;
    const bool valid = c < a.nc;
    const double dt = (MODE & UPD_STAGE) ? stage_dt(a) : 0.0;
    double r[NV], cmp[NV];
#pragma unroll
    for (int k = 0; k < NV; k++) r[k] = cmp[k] = 0;
    if (valid) {
#pragma unroll
        for (int s = 0; s < MAXF; s++) {
            const int32_t e = a.ell[(int64_t)s * a.nc + c];
            if (e < 0) break;
            double gf[NV];
            ldq<NV>(a.G + (int64_t)(e >> 1) * NV, gf);
            accumulate<NV, F32>(r, cmp, gf, e & 1);
        }
        if constexpr (F32) {
#pragma unroll
            for (int k = 0; k < NV; k++) r[k] += cmp[k];
        }
    }
    stage_tail<NV, (MODE & UPD_STAGE) != 0, F32>(a, c, valid, dt, r, blk, (MODE & UPD_L2) != 0, (MODE & UPD_DT) != 0);
}

// Sum over cell c's faces of +-G_f (accumulate: c0 adds, c1 subtracts), slots in order.  The face
// records of a cell are read twice per kernel, once by each of the face's cells; they come from L2 the
// second time only if the two reads are close in time.  For 2D cells of 3 or 4 slots (triangles,
// quadrilaterals) every memory read of all the cell's faces is therefore issued before the first
// Riemann solve (4 dependent load rounds per cell instead of 4 per face), so a face's two reads lie
// about the dispatch distance of its two cells' blocks apart rather than up to a block's lifetime.
// 3D cells and larger ones load face by face: their staged states would halve the resident waves.
template <int DIM, int SCHEME, bool SECOND, typename T, int MAXF>
__device__ __forceinline__ void cell_fluxes(const FluxArgs<T> &fa, const int32_t *__restrict__ ell, int64_t nc,
                                            bool roe, int64_t c, double (&r)[DIM + 2], double (&cmp)[DIM + 2]) {
    constexpr int NV = DIM + 2;
    constexpr bool F32 = std::is_same<T, float>::value;
    // 2D, and FP32 in 3D: every face of the cell is loaded before the first solve.  FP64 3D keeps the
    // per-slot loop (the preloaded form needs 178-200 VGPRs there).  FP32 3D cells in the per-slot
    // loop got outlet fluxes that differ from the face strategy's (measured at order 1: up to 10 % of
    // the flux on every outlet face, against F(Q) n, which every other strategy reproduces): its
    // compiled code (ROCm 7.2, gfx950) leaves the inlet density in the right state's density register
    // on outlet and periodic lanes.  The preloaded form, the same arithmetic, reproduces the face
    // strategy bit for bit.
    if constexpr ((DIM == 2 || F32) && MAXF <= 4) {
        int32_t e[MAXF];
        int kind[MAXF], mask[MAXF];
        double n64[MAXF][DIM];
        T X[MAXF][NV], Y[MAXF][NV];
#pragma unroll
        for (int s = 0; s < MAXF; s++) {  // the slot table is padded to MAXF rows
            e[s] = ell[(int64_t)s * nc + c];
            kind[s] = mst::KIND_NONE;  // empty slot: no flux
            mask[s] = 0;
            if (e[s] >= 0) {
                const int64_t f = e[s] >> 1;
                const int info = fa.finfo[f];
                kind[s] = info & 15;
                mask[s] = info >> 4;
                if (kind[s] < mst::KIND_NONE)
                    face_load<DIM, SECOND, T, cell_ahead<DIM, SECOND, T>()>(fa, f, kind[s], n64[s], X[s], Y[s]);
            }
        }
#pragma unroll
        for (int s = 0; s < MAXF; s++) {
            if (kind[s] >= mst::KIND_NONE) continue;  // empty slot or zero-flux face
            double g[NV];
            face_solve<DIM, SCHEME, T>(fa.P, roe, kind[s], mask[s], n64[s], X[s], Y[s], g);
            accumulate<NV, F32>(r, cmp, g, e[s] & 1);
        }
    } else {
        for (int s = 0; s < MAXF; s++) {
            const int32_t e = ell[(int64_t)s * nc + c];
            if (e < 0) break;
            const int64_t f = e >> 1;
            const int info = fa.finfo[f];
            const int kind = info & 15;
            if (kind >= mst::KIND_NONE) continue;  // zero-flux face
            double n64[DIM];
            T X[NV], Y[NV];
            face_load<DIM, SECOND, T, cell_ahead<DIM, SECOND, T>()>(fa, f, kind, n64, X, Y);
            double g[NV];
            face_solve<DIM, SCHEME, T>(fa.P, roe, kind, info >> 4, n64, X, Y, g);
            accumulate<NV, F32>(r, cmp, g, e & 1);
        }
    }
}

// Cell strategy: flux + gather + update fused, one lane per cell.  Each lane solves the Riemann
// problems of its own faces (an interior face is solved by both of its cells, with bit-identical
// inputs and instructions, so the two cells still receive exactly opposite fluxes) and never writes
// face fluxes to memory: the face-flux array's write and re-read are traded for a second solve.
// Resident waves per SIMD: second-order AUSM in 3D FP64 takes 126 to 130 registers as the code around its solves changes;
// 128 are four waves.
template <int DIM, int SCHEME, bool SECOND, typename T>
constexpr int cell_waves() {
    return DIM == 3 && SECOND && SCHEME == MST_SCHEME_AUSM && !std::is_same<T, float>::value ? 4 : 1;
}

template <int DIM, int SCHEME, bool SECOND, typename T, int MAXF>
__global__ __launch_bounds__(BLOCK, (cell_waves<DIM, SCHEME, SECOND, T>())) void k_cell(const FluxArgs<T> fa, const UpdArgs a) {
    constexpr int NV = DIM + 2;
    constexpr bool F32 = std::is_same<T, float>::value;
    const int64_t blk = block_id();
    const int64_t c = blk * BLOCK + threadIdx.x;
    const bool valid = c < a.nc;
    double r[NV], cmp[NV];
#pragma unroll
    for (int k = 0; k < NV; k++) r[k] = cmp[k] = 0;
    if (valid) {
        cell_fluxes<DIM, SCHEME, SECOND, T, MAXF>(fa, a.ell, a.nc, SCHEME == MST_SCHEME_ROE, c, r, cmp);
        if constexpr (F32) {
#pragma unroll
            for (int k = 0; k < NV; k++) r[k] += cmp[k];
        }
    }
    // (the time step last: held over the solves it cost registers, 3D AUSM FP64 98 / 109 us on 663,552 tetrahedra)
    stage_tail<NV, true, F32>(a, c, valid, stage_dt(a), r, blk, a.l2, a.dtred);
}

// ------------------------------------------------------------------------------------ patch strategy
// With the cells in Hilbert order, the BLOCK cells of a block form a compact patch of the mesh: about
// 9 in 10 of the faces it touches join two of its own cells.  The block solves every face of its
// patch once into LDS (a face on the border of two patches is solved by both, with bit-identical
// inputs), then each lane sums its cell's fluxes from LDS in slot order and updates: one kernel, no
// face-flux array in memory, and about 1.65 Riemann problems per cell instead of the cell strategy's
// three.  The sum is the face strategy's, term for term, so all strategies agree bit for bit.
struct PatchArgs {
    const int32_t *__restrict__ start;  // nblk + 1: each block's range in face
    const int32_t *__restrict__ face;   // the faces of each patch that carry a flux, ascending
    const int16_t *__restrict__ loc;    // slot-major per cell: (local face << 1) | is_c1, -1: no flux
    // the same entries with their faces' kind and L/R mask packed in (face | kind << 26 | mask << 29),
    // so a patch face costs one load instead of two dependent ones; null: read face, then finfo
    const uint32_t *__restrict__ fi;
};

constexpr int FI_SHIFT = 26;

// patch face entry j: its face and finfo word (kind | L/R mask << 4)
__device__ __forceinline__ void patch_face(const PatchArgs &p, const int32_t *__restrict__ finfo, int64_t j, int64_t &f,
                                           int &info) {
    if (p.fi) {
        const uint32_t v = p.fi[j];
        f = (int64_t)(v & ((1u << FI_SHIFT) - 1));
        info = (int)((v >> FI_SHIFT) & 7u) | (int)(v >> (FI_SHIFT + 3)) << 4;
    } else {
        f = p.face[j];
        info = finfo[f];
    }
}

// the packed entries of patch_face, from the face lists and the current finfo (kind < 8, mask < 8)
template <int U>
__global__ __launch_bounds__(BLOCK) void k_pack_faces(int64_t n, const int32_t *__restrict__ face,
                                                      const int32_t *__restrict__ finfo, uint32_t *__restrict__ out) {
    const int64_t i = (int64_t)blockIdx.x * BLOCK + threadIdx.x;
    if (i >= n) return;
    const int32_t f = face[i];
    const int info = finfo[f];
    out[i] = (uint32_t)f | (uint32_t)(info & 7) << FI_SHIFT | (uint32_t)((info >> 4) & 7) << (FI_SHIFT + 3);
}

// The FP32 3D gradient's normals (grad_wn): (float)(w n) per incidence, w = 1 - eta on the c0 side and eta
// on the c1 side of the face, in FP64; boundary and empty slots keep (float) n (unused)
template <int DIM>
__global__ __launch_bounds__(BLOCK) void k_weighted_normals(int64_t n, const int32_t *__restrict__ code,
                                                            const double *__restrict__ eta, const double *__restrict__ nrm,
                                                            float *__restrict__ out) {
    const int64_t i = (int64_t)blockIdx.x * BLOCK + threadIdx.x;
    if (i >= n) return;
    const int32_t cd = code[i];
    const double w = cd >= 0 ? ((cd & 1) ? eta[i] : 1.0 - eta[i]) : 1.0;
#pragma unroll
    for (int d = 0; d < DIM; d++) out[i * DIM + d] = (float)(w * nrm[i * DIM + d]);
}

// The FP32 gradient's volume input: (float) frcp(V) per cell (GradVol)
template <int U>
__global__ __launch_bounds__(BLOCK) void k_recip_vol(int64_t n, const double *__restrict__ vol, float *__restrict__ out) {
    const int64_t c = (int64_t)blockIdx.x * BLOCK + threadIdx.x;
    if (c < n) out[c] = (float)frcp(vol[c]);
}

// sum of the lane's cell's face fluxes from LDS, in slot order (the face strategy's order)
template <int NV, int MAXF, bool F32>
__device__ __forceinline__ void patch_sum(const double *g, int npf, const int (&cl)[MAXF], double (&r)[NV]) {
    double cmp[NV];
#pragma unroll
    for (int k = 0; k < NV; k++) r[k] = cmp[k] = 0;
#pragma unroll
    for (int s = 0; s < MAXF; s++) {
        const int l = cl[s];
        if (l < 0) continue;
        double gf[NV];
#pragma unroll
        for (int k = 0; k < NV; k++) gf[k] = g[k * npf + (l >> 1)];
        accumulate<NV, F32>(r, cmp, gf, l & 1);
    }
    if constexpr (F32) {
#pragma unroll
        for (int k = 0; k < NV; k++) r[k] += cmp[k];
    }
}

// STAGE false: the residual only (R and, with a.l2, its norms), for the implicit steady driver.  NT lanes per patch of
// PC cells: twice as many on meshes of few patches, where the patch's faces then take one pass.  extra: what is
// added to a face's flux (the viscous terms).
// A lane has two or three faces, each a chain of loads (entry, the side's indices, the states) and a long solve: the
// next face's indices are fetched while a face is solved, and the update's inputs before the barrier, where a wave waits
// for the others anyway.  Microseconds per SSP-RK2 step before / with: first order 2D 12.9 / 11.7 (45,000 cells),
// 57.8 / 56.8 (819,200); 3D Roe 23.2 / 22.3 (82,944), 80.7 / 78.9 (663,552); second order 3D AUSM 245.2 / 240.5 (the
// patch kernel alone 62.4 / 55.4 in a profile).  Also fetching the next face's states (46 registers more), or the
// update's inputs before the first face (22), is slower again from a few hundred patches on; so is a bound of 96
// registers on 3D Roe (24 bytes of spill: 101 against 81).
struct NoExtra {
    template <typename G>
    __device__ __forceinline__ void operator()(int64_t, int, G &) const {}
};
template <int DIM, int SCHEME, bool SECOND, typename T, int MAXF, bool STAGE = true, int PC = BLOCK, int NT = PC,
          typename Extra = NoExtra>
__global__ __launch_bounds__(NT) void k_patch(const FluxArgs<T> fa, const UpdArgs a, const PatchArgs p,
                                              const Extra extra = Extra()) {
    constexpr int NV = DIM + 2;
    constexpr bool F32 = std::is_same<T, float>::value;
    extern __shared__ double gsh[];  // NV x npf, component-major: consecutive lanes, consecutive banks
    const int64_t blk = block_id();
    const int32_t f0 = p.start[blk];
    const int npf = p.start[blk + 1] - f0;
    const int64_t c = blk * PC + threadIdx.x;
    const bool valid = (NT == PC || threadIdx.x < PC) && c < a.nc;
    struct Idx {
        int32_t f;
        int info;
        int32_t s0, s1;
    } nx;
    auto fetch = [&](int i, Idx &x) {
        int64_t f;
        patch_face(p, fa.finfo, f0 + i, f, x.info);
        x.f = (int32_t)f;
        x.s0 = SECOND ? fa.frec0[f] : fa.fc0[f];
        x.s1 = SECOND ? fa.frec1[f] : fa.fc1[f];
    };
    if ((int)threadIdx.x < npf) fetch(threadIdx.x, nx);
    for (int i = threadIdx.x; i < npf; i += NT) {
        const Idx x = nx;
        double g[NV], n64[DIM];
        T X[NV], Y[NV];
        face_load<DIM, SECOND, T>(fa, x.f, x.info & 15, x.s0, x.s1, n64, X, Y);
        if (i + NT < npf) fetch(i + NT, nx);
        face_solve<DIM, SCHEME, T>(fa.P, SCHEME == MST_SCHEME_ROE, x.info & 15, x.info >> 4, n64, X, Y, g);
        extra(x.f, x.info & 15, g);
#pragma unroll
        for (int k = 0; k < NV; k++) gsh[k * npf + i] = g[k];
    }
    int cl[MAXF];
#pragma unroll
    for (int s = 0; s < MAXF; s++) cl[s] = valid ? p.loc[(int64_t)s * a.nc + c] : -1;  // padded to MAXF rows
    StageIn<NV> in;
    if (STAGE && valid) stage_load<NV, F32>(a, c, in);
    const double dt = STAGE ? stage_dt(a) : 0.0;
    __syncthreads();
    double r[NV];
    patch_sum<NV, MAXF, F32>(gsh, npf, cl, r);
    stage_tail<NV, STAGE, F32, NT>(a, c, valid, dt, r, blk, a.l2, a.dtred, STAGE ? &in : nullptr);
}

// Order 2 in one kernel: the patch also computes the limited gradients of its own cells and of its
// halo (the cells across its border faces), and keeps the reconstructed face states in LDS instead
// of the global record array, so a stage reads the state and the geometry once and writes only the
// new state.  The halo's gradients are computed by every patch that borders them (a quarter more
// gradient work in 2D), from the same inputs with the same instructions as the gradient kernel, so
// the records, fluxes and sums are bit-identical to the other strategies'.
struct HaloArgs {
    const int32_t *__restrict__ start;  // nblk + 1: each block's range in cell
    const int32_t *__restrict__ cell;   // halo cells of each patch
    const int16_t *__restrict__ loc;    // per halo entry, MAXF slots: (local face << 1) | side, -1: not in the patch
    // the halo cells' incidence geometry copied in halo order (slot-major, entry s * nh + j; k_halo_geo):
    // a patch reads its halo's geometry as coalesced runs, where the cell-ordered arrays would cost a
    // mostly unused line per slot and array for each scattered halo cell.  w, n, dx are of the
    // kernel's real type.
    const int32_t *__restrict__ code;
    const void *w, *n, *dx, *vol;
    int64_t nh;
};

// the packed halo geometry: one lane per halo entry j, a copy of its cell's incidence entries
template <int DIM, typename T>
__global__ __launch_bounds__(BLOCK) void k_halo_geo(int64_t nh, int slots, int64_t nc, const int32_t *__restrict__ hcell,
                                                    IncView<T> src, int32_t *__restrict__ code, T *__restrict__ w,
                                                    T *__restrict__ n, T *__restrict__ dx, GradVol<T> *__restrict__ vol) {
    const int64_t j = (int64_t)blockIdx.x * BLOCK + threadIdx.x;
    if (j >= nh) return;
    const int64_t c = hcell[j];
    for (int s = 0; s < slots; s++) {
        const int64_t i = (int64_t)s * nc + c, o = (int64_t)s * nh + j;
        code[o] = src.code[i];
        w[o] = src.w[i];
#pragma unroll
        for (int d = 0; d < DIM; d++) {
            n[o * DIM + d] = src.n[i * DIM + d];
            dx[o * DIM + d] = src.dx[i * DIM + d];
        }
    }
    vol[j] = src.vol[c];
}

// Host side of the packed halo geometry: the device copies, FP64 always and FP32 for the mixed form.
struct HaloGeo {
    int32_t *code = nullptr;
    double *w = nullptr, *n = nullptr, *dx = nullptr, *vol = nullptr;
    float *w32 = nullptr, *n32 = nullptr, *dx32 = nullptr, *vol32 = nullptr;
    int64_t nh = 0;
    void release() {
        for (void *p : {(void *)code, (void *)w, (void *)n, (void *)dx, (void *)vol, (void *)w32, (void *)n32, (void *)dx32,
                        (void *)vol32})
            if (p) (void)hipFree(p);
        *this = HaloGeo();
    }
    // (re)fills the copies from the cell-ordered arrays (f32.code null: no FP32 form); allocates on
    // first use.  Call after every change of the incidence weights.
    template <int DIM>
    hipError_t fill(int slots, int64_t nc, int64_t nh_, const int32_t *hcell, const IncView<double> &f64,
                    const IncView<float> &f32, hipStream_t st) {
        if (nh_ <= 0) return hipSuccess;
        if (code && nh_ != nh) return hipErrorInvalidValue;  // the copies are sized for one halo list
        const size_t m = (size_t)slots * nh_;
        hipError_t e = hipSuccess;
        auto get = [&](auto **p, size_t count) {
            if (!*p && e == hipSuccess) e = hipMalloc((void **)p, count * sizeof(**p));
        };
        get(&code, m);
        get(&w, m);
        get(&n, m * DIM);
        get(&dx, m * DIM);
        get(&vol, (size_t)nh_);
        if (f32.code) {
            get(&w32, m);
            get(&n32, m * DIM);
            get(&dx32, m * DIM);
            get(&vol32, (size_t)nh_);
        }
        if (e != hipSuccess) {
            release();
            return e;
        }
        nh = nh_;
        const dim3 grid((uint32_t)((nh + BLOCK - 1) / BLOCK));
        hipLaunchKernelGGL((k_halo_geo<DIM, double>), grid, dim3(BLOCK), 0, st, nh, slots, nc, hcell, f64, code, w, n, dx, vol);
        if ((e = hipGetLastError()) != hipSuccess) return e;
        if (f32.code) {
            hipLaunchKernelGGL((k_halo_geo<DIM, float>), grid, dim3(BLOCK), 0, st, nh, slots, nc, hcell, f32, code, w32,
                               n32, dx32, vol32);
            e = hipGetLastError();
        }
        return e;
    }
    template <typename T>
    void args(HaloArgs &h) const {
        constexpr bool F32 = std::is_same<T, float>::value;
        h.code = code;
        h.w = F32 ? (const void *)w32 : (const void *)w;
        h.n = F32 ? (const void *)n32 : (const void *)n;
        h.dx = F32 ? (const void *)dx32 : (const void *)dx;
        h.vol = F32 ? (const void *)vol32 : (const void *)vol;
        h.nh = nh;
    }
};

// LDS of the fused kernels for npf faces: the two sides' face states and the fluxes, double[NV][npf].
// Each face's flux overwrites its own states, which only the lane that solves the face reads.
// FP64: states T[2][NV][npf], fluxes over the c0-side states, 16 * NV * npf bytes.  FP32: the two
// sides' states of a component side by side (float2[NV][npf]), exactly the bytes of that
// component's FP64 flux, 8 * NV * npf bytes.  With the face normals staged (2D), the c0 outward normals
// of the patch faces follow, double[DIM][npf] (8 * DIM * npf bytes).
template <typename T>
struct FusedLds {
    T *rec;
    double *g;
    double *nrm;
    int npf;
    __device__ FusedLds(double *sh, int npf_, int nv) : npf(npf_) {
        rec = reinterpret_cast<T *>(sh);
        g = sh;
        nrm = sh + (bytes_per_face_field / 8) * nv * npf_;
    }
    __device__ T &r(int side, int k, int l, int nv) {
        if constexpr (std::is_same<T, double>::value)
            return rec[(side * nv + k) * npf + l];
        else
            return rec[((k * npf + l) << 1) + side];
    }
    static constexpr int bytes_per_face_field = std::is_same<T, double>::value ? 16 : 8;
};

// Whether the fused kernel stages its patch faces' normals in LDS (2D: a patch cell's incidence
// normal is then read from there, + or - its face's normal, instead of from the incidence arrays)
template <int DIM>
constexpr bool fused_lds_normals() {
    return DIM == 2;
}

// dynamic LDS bytes of the fused kernel for patches of at most max_pf faces
inline size_t fused_lds_bytes(int dim, int nv, int max_pf, bool f32, bool staged_normals) {
    const size_t states = (size_t)(f32 ? 8 : 16) * nv * max_pf;
    return states + (staged_normals ? (size_t)8 * dim * max_pf : 0);
}

// Order 2, FP32 records (the mixed form): the patch kernel with its face states staged in LDS.  Each
// lane copies its cell's slot records into the LDS slots of their faces (one coalesced run per slot),
// the halo's lanes the outside sides of the border faces; the faces are then solved from LDS as in the
// fused kernel.  It reads neither the faces' record indices nor, for interior faces, their cells, and
// each record once per patch; the inputs of every face's solve are the records k_flux would read, so
// the results are bit-identical.  LDS: the fused kernel's FP32 layout, 8 * NV bytes per face (the
// size of the FP64 fluxes that overwrite them).
template <int DIM, int SCHEME, int MAXF, int PC = BLOCK, int NT = PC>
__global__ __launch_bounds__(NT) void k_patch_rec(const FluxArgs<float> fa, const UpdArgs a, const PatchArgs p,
                                                     const HaloArgs h) {
    constexpr int NV = DIM + 2;
    extern __shared__ double gsh[];
    const int64_t blk = block_id();
    const int32_t f0 = p.start[blk];
    const int npf = p.start[blk + 1] - f0;
    FusedLds<float> L(gsh, npf, NV);
    const int64_t c = blk * PC + threadIdx.x;
    const bool valid = (NT == PC || threadIdx.x < PC) && c < a.nc;
    int cl[MAXF];
#pragma unroll
    for (int s = 0; s < MAXF; s++) cl[s] = valid ? p.loc[(int64_t)s * a.nc + c] : -1;
    const int32_t h0 = h.start[blk];
    const int nh = h.start[blk + 1] - h0;
#pragma unroll
    for (int s = 0; s < MAXF; s++) {
        const int l = cl[s];
        if (l < 0) continue;
        float q[NV];
        ldq<NV>(fa.rec + ((int64_t)s * a.nc + c) * NV, q);
#pragma unroll
        for (int k = 0; k < NV; k++) L.r(l & 1, k, l >> 1, NV) = q[k];
    }
    // (lanes past the patch's cells take the halo beside them)
    for (int j = NT > PC ? (int)threadIdx.x - PC : threadIdx.x; j < nh; j += NT > PC ? NT - PC : NT) {
        if (NT > PC && j < 0) break;
        const int64_t hc = h.cell[h0 + j];
#pragma unroll
        for (int s = 0; s < MAXF; s++) {
            const int l = h.loc[(int64_t)(h0 + j) * MAXF + s];
            if (l < 0) continue;
            float q[NV];
            ldq<NV>(fa.rec + ((int64_t)s * a.nc + hc) * NV, q);
#pragma unroll
            for (int k = 0; k < NV; k++) L.r(l & 1, k, l >> 1, NV) = q[k];
        }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < npf; i += NT) {
        int64_t f;
        int info;
        patch_face(p, fa.finfo, f0 + i, f, info);
        const int kind = info & 15;
        double n64[DIM];
#pragma unroll
        for (int d = 0; d < DIM; d++) n64[d] = fa.fn[f * DIM + d];
        float X[NV], Y[NV];
        if (kind == mst::KIND_INTERIOR || kind == mst::KIND_PERIODIC) {
#pragma unroll
            for (int k = 0; k < NV; k++) {
                X[k] = L.r(0, k, i, NV);
                Y[k] = L.r(1, k, i, NV);
            }
        } else {
            ldq<NV>(fa.Q + (int64_t)fa.fc0[f] * NV, X);
#pragma unroll
            for (int k = 0; k < NV; k++) Y[k] = L.r(0, k, i, NV);
        }
        double g[NV];
        face_solve<DIM, SCHEME, float>(fa.P, SCHEME == MST_SCHEME_ROE, kind, info >> 4, n64, X, Y, g);
#pragma unroll
        for (int k = 0; k < NV; k++) L.g[k * npf + i] = g[k];
    }
    StageIn<NV> in;
    if (valid) stage_load<NV, true>(a, c, in);
    const double dt = stage_dt(a);
    __syncthreads();
    double r[NV];
    patch_sum<NV, MAXF, true>(L.g, npf, cl, r);
    stage_tail<NV, true, true, NT>(a, c, valid, dt, r, blk, a.l2, a.dtred, &in);
}

// Resident waves per SIMD requested for the fused kernel, where the bound costs no more than a register
// of spill: FP64 triangles with Roe or unlimited AUSM 4 (at most 128 VGPRs; the compiler would keep 3
// and the kernel, bound by its dependent load rounds, runs about 15 % slower), FP32 triangles 6 (at
// most 80 VGPRs; with the gradient's loads all issued up front, 7 waves spill 12 registers and run
// 7 % slower), other 2D FP32 cells 4.  Elsewhere the bound would spill, so the compiler chooses.
template <int DIM, int SCHEME, int LIM, typename T, int MAXF>
constexpr int fused_waves() {
    if constexpr (DIM != 2) return 1;
    if constexpr (sizeof(T) == 4) return MAXF == 3 ? (MST_FUSED_WAVES32 > 0 ? MST_FUSED_WAVES32 : 6) : 4;
    return ((SCHEME == MST_SCHEME_ROE || LIM == MST_LIM_NONE) && MAXF == 3) ? 4 : 1;
}

// Phases of one patch in the fused form, for a block of NT lanes: the limited gradients of the
// patch cells [cb, ce) and of the patch's halo, their face states into LDS, then the fluxes of the
// patch faces (p.face from f0) into L.g.  Ends with a barrier.  cl receives the lane's cell's slot
// entries ((local face << 1) | side, -1: none) for the caller's sums.  roe picks the scheme when
// SCHEME is SCHEME_RUNTIME.  pre() runs between the gradient and the flux phases, when the gradient's
// registers are free: the caller fetches its update's inputs there, so their latency overlaps the
// face solves.  NT = 2 PC: the lanes past the patch's cells take the halo's gradients at the same time, and
// the patch's faces take one pass.
template <int DIM, int SCHEME, int LIM, typename T, int MAXF, bool NRM_LDS = false, int PC = BLOCK, int NT = PC, typename Pre>
__device__ __forceinline__ void fused_patch(const GradArgs<T> &ga, const FluxArgs<T> &fa, bool roe, const PatchArgs &p,
                                            const HaloArgs &h, int64_t patch, int64_t cb, int64_t ce, int64_t nc,
                                            int32_t f0, FusedLds<T> &L, int (&cl)[MAXF], Pre pre) {
    constexpr int NV = DIM + 2;
    const int npf = L.npf;
    // Inputs of the later phases that do not depend on the gradients are fetched first, so their
    // latency overlaps the gradient phase: each lane's first PF patch faces (face, kind, normal), its
    // cell's slot entries and its first halo cell.
    constexpr int PF = NT > PC ? 1 : MST_FUSED_PF;
    int64_t pf_f[PF];
    int pf_info[PF];
    double pf_n[PF][DIM];
#pragma unroll
    for (int q = 0; q < PF; q++) {
        const int i = threadIdx.x + q * NT;
        pf_f[q] = -1;
        pf_info[q] = 0;
        if (i < npf) {
            patch_face(p, fa.finfo, f0 + i, pf_f[q], pf_info[q]);
#pragma unroll
            for (int d = 0; d < DIM; d++) pf_n[q][d] = fa.fn[pf_f[q] * DIM + d];
        }
    }
    const int64_t c = cb + threadIdx.x;
    const bool mine = (NT == PC || threadIdx.x < PC) && c < ce;
#pragma unroll
    for (int s = 0; s < MAXF; s++) cl[s] = mine ? p.loc[(int64_t)s * nc + c] : -1;
    // limited gradients of the patch cells, then of the halo cells; face states into LDS
    const int32_t h0 = h.start[patch];
    const int next = PC + (h.start[patch + 1] - h0);  // the patch's cells, then its halo
    // the lane's first halo cell (a wide block: of the lanes past the patch's cells)
    const int j0 = NT > PC ? (int)threadIdx.x - PC : (int)threadIdx.x;
    const int32_t hc = (NT == PC || j0 >= 0) && PC + j0 < next ? h.cell[h0 + j0] : 0;
    const IncView<T> own = cell_view(ga);
    const IncView<T> hv{h.code, static_cast<const T *>(h.w), static_cast<const T *>(h.n),
                        static_cast<const T *>(h.dx), static_cast<const GradVol<T> *>(h.vol), h.nh};
    if constexpr (NRM_LDS) {
        // The patch cells' reads first (their normals excepted), then the patch faces' normals into
        // LDS, a barrier, and each incidence normal from LDS: + the face's normal on its c0 side, - on
        // its c1 side, which is how the incidence arrays hold it.  A slot whose face carries no flux
        // (not a patch face) reads the incidence array.
        GradIn<DIM, MAXF, T> gin;
        T dxs[MAXF][DIM];
        if (mine) grad_fetch<DIM, MAXF, false, T>(ga.Q, own, c, c, gin, dxs);
#pragma unroll
        for (int q = 0; q < PF; q++) {
            const int i = threadIdx.x + q * NT;
            if (i < npf)
#pragma unroll
                for (int d = 0; d < DIM; d++) L.nrm[d * npf + i] = pf_n[q][d];
        }
        for (int i = threadIdx.x + PF * NT; i < npf; i += NT) {
            const int64_t f = p.face[f0 + i];
#pragma unroll
            for (int d = 0; d < DIM; d++) L.nrm[d * npf + i] = fa.fn[f * DIM + d];
        }
        __syncthreads();
        if (mine) {
#pragma unroll
            for (int s = 0; s < MAXF; s++) {
                const int l = cl[s];
                if (l >= 0) {
#pragma unroll
                    for (int d = 0; d < DIM; d++) {
                        const double v = L.nrm[d * npf + (l >> 1)];
                        gin.n[s][d] = (T)((l & 1) ? -v : v);
                    }
                } else if (gin.code[s] != -2) {
#pragma unroll
                    for (int d = 0; d < DIM; d++) gin.n[s][d] = own.n[((int64_t)s * nc + c) * DIM + d];
                }
            }
            T lgr[NV * DIM], t[NV][DIM], ph[NV];
            const int nfc = grad_eval<DIM, MAXF, LIM, T>(gin, dxs, lgr, t, ph);
#pragma unroll
            for (int s = 0; s < MAXF; s++) {
                if (s >= nfc) break;
                const int l = cl[s];
                if (l < 0) continue;
                T q[NV];
#pragma unroll
                for (int k = 0; k < NV; k++) q[k] = gin.qc[k];
                recon<DIM>(q, lgr, dxs[s]);
#pragma unroll
                for (int k = 0; k < NV; k++) L.r(l & 1, k, l >> 1, NV) = q[k];
            }
        }
    }
    for (int i0 = NRM_LDS && NT == PC ? PC : 0; i0 < next; i0 += NT) {
        const int i = i0 + (int)threadIdx.x;
        if (i >= next) break;
        if (NRM_LDS && NT > PC && i < PC) continue;  // done above
        int64_t cc, g;
        const int16_t *lp;
        int64_t stride;
        const bool halo = NT == PC ? i0 > 0 : i >= PC;
        if (!halo) {
            cc = cb + i;
            if (cc >= ce) continue;
            g = cc;
            lp = p.loc + cc;
            stride = nc;
        } else {
            g = h0 + i - PC;
            cc = i < 2 * PC ? hc : h.cell[g];
            lp = h.loc + g * MAXF;
            stride = 1;
        }
        T qc[NV], lgr[NV * DIM], dxs[MAXF][DIM], t[NV][DIM], ph[NV];
        const int nfc = grad_limited<DIM, MAXF, LIM, T>(ga.Q, halo ? hv : own, g, cc, qc, lgr, dxs, t, ph);
#pragma unroll
        for (int s = 0; s < MAXF; s++) {
            if (s >= nfc) break;
            const int l = lp[s * stride];
            if (l < 0) continue;
            T q[NV];
#pragma unroll
            for (int k = 0; k < NV; k++) q[k] = qc[k];
            recon<DIM>(q, lgr, dxs[s]);
#pragma unroll
            for (int k = 0; k < NV; k++) L.r(l & 1, k, l >> 1, NV) = q[k];
        }
    }
    __syncthreads();
    pre();
    // the patch's face fluxes (face_load's inputs from LDS: both sides' states, or for a boundary
    // face the raw interior state from memory and its reconstructed state)
    for (int q = 0, i = threadIdx.x; i < npf; q++, i += NT) {
        int64_t f;
        int info;
        double n64[DIM];
        if (q < PF) {
            f = pf_f[q];
            info = pf_info[q];
            if constexpr (!NRM_LDS)
#pragma unroll
                for (int d = 0; d < DIM; d++) n64[d] = pf_n[q][d];
        } else {
            patch_face(p, fa.finfo, f0 + i, f, info);
            if constexpr (!NRM_LDS)
#pragma unroll
                for (int d = 0; d < DIM; d++) n64[d] = fa.fn[f * DIM + d];
        }
        if constexpr (NRM_LDS)
#pragma unroll
            for (int d = 0; d < DIM; d++) n64[d] = L.nrm[d * npf + i];
        const int kind = info & 15;
        T X[NV], Y[NV];
        if (kind == mst::KIND_INTERIOR || kind == mst::KIND_PERIODIC) {
#pragma unroll
            for (int k = 0; k < NV; k++) {
                X[k] = L.r(0, k, i, NV);
                Y[k] = L.r(1, k, i, NV);
            }
        } else {
            ldq<NV>(fa.Q + (int64_t)fa.fc0[f] * NV, X);
#pragma unroll
            for (int k = 0; k < NV; k++) Y[k] = L.r(0, k, i, NV);
        }
        double g[NV];
        face_solve<DIM, SCHEME, T>(fa.P, SCHEME == SCHEME_RUNTIME ? roe : SCHEME == MST_SCHEME_ROE, kind, info >> 4,
                                   n64, X, Y, g);
#pragma unroll
        for (int k = 0; k < NV; k++) L.g[k * npf + i] = g[k];
    }
    __syncthreads();
}

template <int DIM, int SCHEME, int LIM, typename T, int MAXF, int PC = BLOCK, int NT = PC>
__global__ __launch_bounds__(NT, (NT > PC ? 2 : fused_waves<DIM, SCHEME, LIM, T, MAXF>())) void k_fused(
    const GradArgs<T> ga, const FluxArgs<T> fa, const UpdArgs a, const PatchArgs p, const HaloArgs h) {
    constexpr int NV = DIM + 2;
    constexpr bool F32 = std::is_same<T, float>::value;
    extern __shared__ double sh[];
    const int64_t blk = block_id();
    const int32_t f0 = p.start[blk];
    FusedLds<T> L(sh, p.start[blk + 1] - f0, NV);
    const int64_t cb = blk * PC, ce = cb + PC < a.nc ? cb + PC : a.nc;
    int cl[MAXF];
    const int64_t c = cb + threadIdx.x;
    const bool valid = (NT == PC || threadIdx.x < PC) && c < a.nc;
    StageIn<NV> in;
    double dt = 0;
    fused_patch<DIM, SCHEME, LIM, T, MAXF, fused_lds_normals<DIM>(), PC, NT>(ga, fa, SCHEME == MST_SCHEME_ROE, p, h, blk, cb,
                                                                          ce, a.nc, f0, L, cl, [&]() {
        dt = stage_dt(a);
        if (valid) stage_load<NV, F32>(a, c, in);
    });
    double r[NV];
    patch_sum<NV, MAXF, F32>(L.g, L.npf, cl, r);
    // (sh: at least NV * NT / 64 doubles)
    stage_tail<NV, true, F32, NT, true>(a, c, valid, dt, r, blk, a.l2, a.dtred, &in, sh);
}

// ------------------------------------------------------------------------------------ reductions
// CFL: dt_c = cfl V / sum_d (|u_d| + a) Shalf_d (new; the reference's DT is fixed, time/Time.cpp:62)
template <int DIM>
__global__ __launch_bounds__(BLOCK) void k_cfl(int64_t nc, const double *__restrict__ Q,
                                               const double *__restrict__ vol, const double *__restrict__ sh,
                                               double gamma, double cfl, double *__restrict__ part_dt) {
    constexpr int NV = DIM + 2;
    const int64_t blk = block_id();
    const int64_t c = blk * BLOCK + threadIdx.x;
    double v[1] = {INFINITY};
    if (c < nc) {
        double q[NV];
        ldq<NV>(Q + c * NV, q);
        v[0] = local_dt<DIM>(q, sh + c * DIM, vol[c], gamma, cfl);
    }
    block_partial<1, true>(v, part_dt + blk, 1);
}

// Time::goNextTimeStep monitor (time/Time.cpp:69-76): max |new-old|/old, values that do not compare
// greater are skipped.  Block b strides over the cells b*BLOCK + i*gridDim.x*BLOCK, so a grid smaller
// than the cell count works too; part receives one partial per block and field.
template <int NV>
__global__ __launch_bounds__(BLOCK) void k_maxrel(int64_t nc, const double *__restrict__ Qnew,
                                                  const double *__restrict__ Qold, double *__restrict__ part) {
    const int64_t blk = block_id();
    double v[NV];
#pragma unroll
    for (int k = 0; k < NV; k++) v[k] = 0;
    for (int64_t c = blk * BLOCK + threadIdx.x; c < nc; c += (int64_t)gridDim.x * BLOCK) {
        double a[NV], b[NV];
        ldq<NV>(Qnew + c * NV, a);
        ldq<NV>(Qold + c * NV, b);
#pragma unroll
        for (int k = 0; k < NV; k++) {
            const double x = fabs(a[k] - b[k]) / b[k];
            if (v[k] < x) v[k] = x;
        }
    }
    __shared__ double s[NV][BLOCK];
#pragma unroll
    for (int k = 0; k < NV; k++) s[k][threadIdx.x] = v[k];
    __syncthreads();
    for (int w = BLOCK / 2; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w)
#pragma unroll
            for (int k = 0; k < NV; k++)
                if (s[k][threadIdx.x] < s[k][threadIdx.x + w]) s[k][threadIdx.x] = s[k][threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x < NV) part[threadIdx.x * (int64_t)gridDim.x + blk] = s[threadIdx.x][0];
}

// part[k][b] = the sum of the partials of block b's SUB_PATCH patches in order (n patches), which is the partial of
// a block of BLOCK cells bit for bit: block_partial adds its waves' sums in this order
template <int U>
__global__ __launch_bounds__(BLOCK) void k_join_partials(int64_t n, int64_t nb, int nv, const double *__restrict__ sub,
                                                         double *__restrict__ part) {
    const int64_t i = (int64_t)blockIdx.x * BLOCK + threadIdx.x;
    if (i >= nb * nv) return;
    const int64_t k = i / nb, b = i % nb;
    constexpr int R = BLOCK / SUB_PATCH;
    double v = sub[k * n + b * R];
    for (int r = 1; r < R && b * R + r < n; r++) v += sub[k * n + b * R + r];
    part[i] = v;
}

// Finish of the per-block partials.  Slot k is a sum (kind 0), a min (kind 1) or a max (kind 2).
// Block b reduces the partials [b*chunk, (b+1)*chunk): every thread walks its share with a fixed
// stride, then a fixed butterfly inside each wave and a fixed pass over the waves, so the result is
// bit-reproducible.  With mid set (first level of a two-level finish) block b writes its raw result
// to mid[k*gridDim.x + b]; otherwise (one block) it writes dst[k] (post: sqrt(v / count)).
constexpr int FIN = 1024;
constexpr int FIN_CHUNK = 1024;  // partials per block of the first level
struct FinArgs {
    const double *src[12];
    int kind[12];
    double *dst[12];
    int post[12];  // 1: sqrt(v / count)
    int n;
    int64_t nblk, chunk;
    double count;
    double *mid;
};

__device__ __forceinline__ double fin_op(int kind, double a, double b) {
    return kind == 0 ? a + b : (kind == 1 ? fmin(a, b) : (a < b ? b : a));
}

static __global__ __launch_bounds__(FIN) void k_finish(const FinArgs a) {
    constexpr int MAXW = 12;
    __shared__ double s[MAXW][FIN / 64];
    double acc[MAXW];
#pragma unroll
    for (int k = 0; k < MAXW; k++) acc[k] = (k < a.n && a.kind[k] == 1) ? INFINITY : 0.0;
    const int64_t i0 = (int64_t)blockIdx.x * a.chunk;
    const int64_t i1 = i0 + a.chunk < a.nblk ? i0 + a.chunk : a.nblk;
    for (int64_t i = i0 + threadIdx.x; i < i1; i += FIN) {
#pragma unroll
        for (int k = 0; k < MAXW; k++)
            if (k < a.n) acc[k] = fin_op(a.kind[k], acc[k], a.src[k][i]);
    }
#pragma unroll
    for (int k = 0; k < MAXW; k++) {
        if (k < a.n) {
            for (int m = 32; m > 0; m >>= 1) acc[k] = fin_op(a.kind[k], acc[k], __shfl_xor(acc[k], m, 64));
            if ((threadIdx.x & 63) == 0) s[k][threadIdx.x >> 6] = acc[k];
        }
    }
    __syncthreads();
    if ((int)threadIdx.x < a.n) {
        const int k = threadIdx.x;
        double v = s[k][0];
        for (int w = 1; w < FIN / 64; w++) v = fin_op(a.kind[k], v, s[k][w]);
        if (a.mid)
            a.mid[(int64_t)k * gridDim.x + blockIdx.x] = v;
        else
            a.dst[k][0] = a.post[k] ? sqrt(v / a.count) : v;
    }
}

// One minimum (the CFL time step) over n partials in one block: each lane's eight loads are in flight
// together.  A minimum does not depend on the combining order, so this equals k_finish's result.
template <int U>
__global__ __launch_bounds__(FIN) void k_finish_min(const double *__restrict__ src, int64_t n, double *__restrict__ dst) {
    __shared__ double s[FIN / 64];
    double v = INFINITY;
    for (int64_t i = threadIdx.x; i < n; i += 8 * FIN) {
        double x[8];
#pragma unroll
        for (int u = 0; u < 8; u++) x[u] = i + u * FIN < n ? src[i + u * FIN] : INFINITY;
#pragma unroll
        for (int u = 0; u < 8; u++) v = fmin(v, x[u]);
    }
    for (int m = 32; m > 0; m >>= 1) v = fmin(v, __shfl_xor(v, m, 64));
    if ((threadIdx.x & 63) == 0) s[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < FIN / 64; w++) v = fmin(v, s[w]);
        dst[0] = v;
    }
}

// The W maxima of k_maxrel's partials (all >= 0, no NaN: any order) to the host's board in one block of NT lanes, U loads
// per field of each lane in flight together: n <= U NT is one round of the memory's latency, so MONITOR_GRID bounds
// k_maxrel's partials by 8 FIN.  (U = 1 up to two rounds: 0.5 us less than eight
// loads that are mostly masked out.)  28 partials: 4 us where k_finish takes 8 and a stream synchronisation and a copy followed;
// the whole call on 2M / 8M / 24.5M triangles: 35 / 113 / 287 us (41 / 143 / 440 with 256 lanes of one load each).
constexpr int64_t MONITOR_GRID = 8 * FIN;
template <int W, int NT, int U>
__global__ __launch_bounds__(NT) void k_finish_max(const double *__restrict__ part, int64_t n, Board *__restrict__ b,
                                                   uint32_t seq) {
    __shared__ double s[W][NT / 64];
    double v[W];
#pragma unroll
    for (int k = 0; k < W; k++) v[k] = 0;
    for (int64_t i = threadIdx.x; i < n; i += U * NT) {
        double x[W][U];
#pragma unroll
        for (int k = 0; k < W; k++)
#pragma unroll
            for (int u = 0; u < U; u++) x[k][u] = i + u * NT < n ? part[k * n + i + u * NT] : 0;
#pragma unroll
        for (int k = 0; k < W; k++)
#pragma unroll
            for (int u = 0; u < U; u++)
                if (v[k] < x[k][u]) v[k] = x[k][u];
    }
#pragma unroll
    for (int k = 0; k < W; k++) {
        for (int m = 32; m > 0; m >>= 1) {
            const double x = __shfl_xor(v[k], m, 64);
            if (v[k] < x) v[k] = x;
        }
        if ((threadIdx.x & 63) == 0) s[k][threadIdx.x >> 6] = v[k];
    }
    __syncthreads();
    if ((int)threadIdx.x < W) {
        double m = s[threadIdx.x][0];
        for (int w = 1; w < NT / 64; w++)
            if (m < s[threadIdx.x][w]) m = s[threadIdx.x][w];
        b->mon[threadIdx.x] = m;
        __threadfence_system();
    }
    __syncthreads();
    if (threadIdx.x == 0) __hip_atomic_store(&b->seq, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// ------------------------------------------------------------------------------------ warm start
// features (cell centre, conditions) for the network and the decoding of its outputs
//   y = (log(rho/rho_inf), u_1/|u_inf|, .., u_dim/|u_inf|, log(p/p_inf)),  rho_inf = 1, p_inf = 1/gamma,
//   |u_inf| = the first condition (the freestream Mach number: a_inf = 1)
// which gives a positive density and pressure for any finite output.
struct WarmArgs {
    int64_t nc;
    const double *cxc;
    int n_cond;
    float cond[8];
    double mach, gamma;
    float *feat;
    const float *Y;
    double *Q;
    int *bad;
};

template <int DIM>
__global__ __launch_bounds__(BLOCK) void k_warm_features(const WarmArgs w) {
    const int64_t c = (int64_t)blockIdx.x * BLOCK + threadIdx.x;
    if (c >= w.nc) return;
    const int n_in = DIM + w.n_cond;
    for (int d = 0; d < DIM; d++) w.feat[c * n_in + d] = (float)w.cxc[c * DIM + d];
    for (int k = 0; k < w.n_cond; k++) w.feat[c * n_in + DIM + k] = w.cond[k];
}

template <int DIM>
__global__ __launch_bounds__(BLOCK) void k_warm_decode(const WarmArgs w) {
    constexpr int NV = DIM + 2;
    const int64_t c = (int64_t)blockIdx.x * BLOCK + threadIdx.x;
    if (c >= w.nc) return;
    const float *y = w.Y + c * NV;
    const double rho = exp((double)y[0]);
    const double p = exp((double)y[NV - 1]) / w.gamma;
    double ke = 0, q[NV];
    q[0] = rho;
    for (int d = 0; d < DIM; d++) {
        const double u = w.mach * (double)y[1 + d];
        q[1 + d] = rho * u;
        ke += u * u;
    }
    q[NV - 1] = p / (w.gamma - 1) + 0.5 * rho * ke;
    bool ok = rho > 0 && p > 0 && rho < INFINITY && p < INFINITY;
    for (int k = 0; k < NV; k++) ok = ok && q[k] == q[k];
    if (!ok) w.bad[0] = 1;
    stq<NV>(w.Q + c * NV, q);
}

// FP32 shadow of a state (mixed form), after the host writes the FP64 state
static __global__ __launch_bounds__(BLOCK) void k_shadow(int64_t n, const double *__restrict__ Q, float *__restrict__ Q32) {
    const int64_t i = (int64_t)blockIdx.x * BLOCK + threadIdx.x;
    if (i < n) Q32[i] = (float)Q[i];
}

// plain streaming copy: the reference point that scales rocprofv3 FETCH_SIZE / WRITE_SIZE to bytes
static __global__ __launch_bounds__(BLOCK) void k_copy(int64_t n2, const double2 *__restrict__ src,
                                                double2 *__restrict__ dst) {
    const int64_t i = (int64_t)blockIdx.x * BLOCK + threadIdx.x;
    if (i < n2) dst[i] = src[i];
}

// batched flux-scheme plugin: F = solverAll(dir) after set(QL, QR)
template <int DIM, int SCHEME>
__global__ __launch_bounds__(BLOCK) void k_riemann(int64_t n, const double *__restrict__ QL,
                                                   const double *__restrict__ QR, const int32_t *__restrict__ dir,
                                                   double *__restrict__ F, Params<double> P) {
    constexpr int NV = DIM + 2;
    const int64_t i = (int64_t)blockIdx.x * BLOCK + threadIdx.x;
    if (i >= n) return;
    double A[NV], B[NV], nrm[DIM], g[NV];
#pragma unroll
    for (int k = 0; k < NV; k++) {
        A[k] = QL[i * NV + k];
        B[k] = QR[i * NV + k];
    }
    const int d0 = dir[i];
#pragma unroll
    for (int d = 0; d < DIM; d++) nrm[d] = d == d0 ? 1.0 : 0.0;
    riemann_face<DIM, SCHEME, double>(A, B, nrm, (1 << DIM) - 1, P, g);
#pragma unroll
    for (int k = 0; k < NV; k++) F[i * NV + k] = g[k];
}

}  // namespace mstk
