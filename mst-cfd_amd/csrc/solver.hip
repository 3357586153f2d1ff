// solver.hip -- device context behind include/mstcfd.h: SoA device arrays, launch sequences of the
// residual path (kernels.hpp), state transfer in the reference's AllData layout, timing.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <string>
#include <vector>

#include "context.hpp"
#include "lusgs.hpp"
#include "viscous.hpp"
#include "mlp.hpp"
#include "mstcfd.h"

namespace mst {
const std::string &last_error();
}

namespace {

int check_config(const mst_config *c) {
    if (!c) return mst::fail(MST_E_ARG, "null config");
    if (c->scheme != MST_SCHEME_ROE && c->scheme != MST_SCHEME_AUSM) return mst::fail(MST_E_ARG, "bad scheme");
    if (c->order != 1 && c->order != 2) return mst::fail(MST_E_ARG, "order must be 1 or 2");
    if (c->limiter < MST_LIM_NONE || c->limiter > MST_LIM_VANLEER) return mst::fail(MST_E_ARG, "bad limiter");
    if (c->rk < 1 || c->rk > 3) return mst::fail(MST_E_ARG, "rk must be 1, 2 or 3");
    if (c->precision != MST_PREC_FP64 && c->precision != MST_PREC_MIXED) return mst::fail(MST_E_ARG, "bad precision");
    if (!(c->gamma > 1) || !(c->entropy_delta > 0) || c->eor < 0 || c->cfl < 0)
        return mst::fail(MST_E_ARG, "bad gamma / entropy_delta / eor / cfl");
    if (!(c->q_inlet[0] > 0)) return mst::fail(MST_E_ARG, "inlet density must be positive");
    if (!(c->mu >= 0) || !(c->kappa >= 0) || !std::isfinite(c->mu) || !std::isfinite(c->kappa) ||
        !std::isfinite(c->lam))
        return mst::fail(MST_E_ARG, "viscous coefficients must be finite, mu and kappa >= 0");
    if ((c->mu > 0 || c->kappa > 0) && !(c->cv > 0)) return mst::fail(MST_E_ARG, "viscous runs need cv > 0");
    return MST_OK;
}

}  // namespace

namespace {

// FP32 shadow of state buffer i (mixed form), made on demand after a host write
int ensure_shadow(mst_ctx *x, int i) {
    if (!x->mixed || x->shadow_ok[i]) return MST_OK;
    int rc = launch(x, -1, k_shadow, x->nc * x->nv, x->nc * x->nv, (const double *)x->Q[i], x->Q32[i]);
    if (rc) return rc;
    x->shadow_ok[i] = true;
    return MST_OK;
}

template <int DIM, typename T>
int run_grad_t(mst_ctx *x, int isrc, bool debug) {
    const GradArgs<T> a = grad_args<T>(x, isrc, debug);
    const int lim = x->cfg.limiter;
#define MST_GRAD(MF)                                                                                    \
    if (lim == MST_LIM_NONE) return launch(x, MST_K_GRAD, k_grad<DIM, MF, MST_LIM_NONE, T>, x->nc, a);     \
    if (lim == MST_LIM_MINMOD) return launch(x, MST_K_GRAD, k_grad<DIM, MF, MST_LIM_MINMOD, T>, x->nc, a); \
    return launch(x, MST_K_GRAD, k_grad<DIM, MF, MST_LIM_VANLEER, T>, x->nc, a);
    if (x->slots == 3) { MST_GRAD(3) }
    if (x->slots == 4) { MST_GRAD(4) }
    MST_GRAD(8)
#undef MST_GRAD
}

int run_grad(mst_ctx *x, int isrc, bool debug) {
    int rc = ensure_shadow(x, isrc);
    if (rc) return rc;
    if (x->mixed) return x->dim == 2 ? run_grad_t<2, float>(x, isrc, debug) : run_grad_t<3, float>(x, isrc, debug);
    return x->dim == 2 ? run_grad_t<2, double>(x, isrc, debug) : run_grad_t<3, double>(x, isrc, debug);
}

template <int DIM, typename T>
int run_flux_t(mst_ctx *x, int isrc) {
    const FluxArgs<T> a = flux_args<T>(x, isrc);
    const bool second = x->cfg.order >= 2;
    if (x->cfg.scheme == MST_SCHEME_ROE)
        return second ? launch(x, MST_K_FLUX, k_flux<DIM, MST_SCHEME_ROE, true, T>, x->nf, a)
                      : launch(x, MST_K_FLUX, k_flux<DIM, MST_SCHEME_ROE, false, T>, x->nf, a);
    return second ? launch(x, MST_K_FLUX, k_flux<DIM, MST_SCHEME_AUSM, true, T>, x->nf, a)
                  : launch(x, MST_K_FLUX, k_flux<DIM, MST_SCHEME_AUSM, false, T>, x->nf, a);
}

// viscous gradients of the cells of state isrc
int run_visc_grad(mst_ctx *x, int isrc) {
    const ViscArgs a = visc_args(x, isrc);
    if (x->dim == 2)
        return x->slots == 3 ? launch(x, MST_K_VISC, k_visc_grad<2, 3>, x->nc, a)
                             : (x->slots == 4 ? launch(x, MST_K_VISC, k_visc_grad<2, 4>, x->nc, a)
                                              : launch(x, MST_K_VISC, k_visc_grad<2, 8>, x->nc, a));
    return x->slots == 4 ? launch(x, MST_K_VISC, k_visc_grad<3, 4>, x->nc, a)
                         : launch(x, MST_K_VISC, k_visc_grad<3, 8>, x->nc, a);
}

// viscous terms of state isrc subtracted from the face fluxes (after the flux kernel)
int run_viscous(mst_ctx *x, int isrc) {
    const int rc = run_visc_grad(x, isrc);
    if (rc) return rc;
    const ViscArgs a = visc_args(x, isrc);
    return x->dim == 2 ? launch(x, MST_K_VISC, k_visc_flux<2>, x->nf, a) : launch(x, MST_K_VISC, k_visc_flux<3>, x->nf, a);
}

// gradients of a viscous stage on the patch route: face states and viscous gradients in one kernel (order 2, FP64)
template <int DIM, int MF>
int run_grad_visc_t(mst_ctx *x, int isrc) {
    const GradArgs<double> g = grad_args<double>(x, isrc, false);
    const ViscArgs v = visc_args(x, isrc);
    if (x->cfg.limiter == MST_LIM_NONE) return launch(x, MST_K_GRAD, k_grad_visc<DIM, MF, MST_LIM_NONE>, x->nc, g, v);
    if (x->cfg.limiter == MST_LIM_MINMOD) return launch(x, MST_K_GRAD, k_grad_visc<DIM, MF, MST_LIM_MINMOD>, x->nc, g, v);
    return launch(x, MST_K_GRAD, k_grad_visc<DIM, MF, MST_LIM_VANLEER>, x->nc, g, v);
}

int run_grad_visc(mst_ctx *x, int isrc) {
    if (x->cfg.order >= 2 && !x->mixed) {
        if (x->dim == 2) return x->slots == 3 ? run_grad_visc_t<2, 3>(x, isrc) : run_grad_visc_t<2, 4>(x, isrc);
        return run_grad_visc_t<3, 4>(x, isrc);
    }
    int rc = MST_OK;
    if (x->cfg.order >= 2) rc = run_grad(x, isrc, false);
    return rc ? rc : run_visc_grad(x, isrc);
}

// residual evaluation up to the face fluxes: gradient + limiter (order 2), the flux kernel, and the
// viscous terms when the configuration has them
int run_face_flux(mst_ctx *x, int isrc) {
    x->g_of = -1;
    int rc = ensure_shadow(x, isrc);
    if (rc) return rc;
    if (x->cfg.order >= 2) {
        rc = run_grad(x, isrc, false);
        if (rc) return rc;
    }
    if (x->mixed)
        rc = x->dim == 2 ? run_flux_t<2, float>(x, isrc) : run_flux_t<3, float>(x, isrc);
    else
        rc = x->dim == 2 ? run_flux_t<2, double>(x, isrc) : run_flux_t<3, double>(x, isrc);
    if (rc || !x->viscous) return rc;
    return run_viscous(x, isrc);
}

// G of the last viscous stage, before G is read or its state or configuration replaced.  The patch route of a viscous
// stage stores no face fluxes, and a viscous context's G is its last stage's whichever route that took: so the
// stage leaves its state's index and the fluxes are formed here, for the few calls that need them.
int ensure_fluxes(mst_ctx *x) { return x->g_of < 0 ? (int)MST_OK : run_face_flux(x, x->g_of); }

template <int NV, bool GT>
int run_update_t(mst_ctx *x, int mode, int is, int in, const Stage &sg, int iout) {
    const UpdArgs a = upd_args(x, mode, is, in, sg, iout);
    partials(x, mode, x->nblk_c);
#define MST_UPD(MF)                                                                                             \
    switch (mode & ~UPD_CHECK) {                                                                                             \
        case UPD_RESIDUAL: return launch(x, MST_K_UPDATE, k_update<NV, MF, UPD_RESIDUAL, GT>, x->nc, a);        \
        case UPD_L2: return launch(x, MST_K_UPDATE, k_update<NV, MF, UPD_L2, GT>, x->nc, a);                    \
        case UPD_STAGE: return launch(x, MST_K_UPDATE, k_update<NV, MF, UPD_STAGE, GT>, x->nc, a);              \
        case UPD_STAGE | UPD_L2: return launch(x, MST_K_UPDATE, k_update<NV, MF, UPD_STAGE | UPD_L2, GT>, x->nc, a); \
        case UPD_STAGE | UPD_DT: return launch(x, MST_K_UPDATE, k_update<NV, MF, UPD_STAGE | UPD_DT, GT>, x->nc, a); \
        default:                                                                                                \
            return launch(x, MST_K_UPDATE, k_update<NV, MF, UPD_STAGE | UPD_L2 | UPD_DT, GT>, x->nc, a);        \
    }
    if (x->maxf <= 3) { MST_UPD(3) }
    if (x->maxf <= 4) { MST_UPD(4) }
    MST_UPD(8)
#undef MST_UPD
}

int run_update(mst_ctx *x, int mode, int is, int in, const Stage &sg, int iout) {
    int rc;
    if (x->mixed)
        rc = x->nv == 4 ? run_update_t<4, true>(x, mode, is, in, sg, iout)
                        : run_update_t<5, true>(x, mode, is, in, sg, iout);
    else
        rc = x->nv == 4 ? run_update_t<4, false>(x, mode, is, in, sg, iout)
                        : run_update_t<5, false>(x, mode, is, in, sg, iout);
    if (rc == MST_OK && iout >= 0) x->shadow_ok[iout] = x->mixed;
    return rc;
}

// cell strategy: gradient + limiter (order 2), then the fused flux + gather + stage update
template <int DIM, typename T>
int run_cell_t(mst_ctx *x, int mode, int is, int in, const Stage &sg, int iout) {
    const FluxArgs<T> fa = flux_args<T>(x, is);
    const UpdArgs a = upd_args(x, mode, is, in, sg, iout);
    partials(x, mode, x->nblk_c);
    const bool second = x->cfg.order >= 2;
    const bool roe = x->cfg.scheme == MST_SCHEME_ROE;
    // slot count of the padded slot-major table: 3 (triangles), 4 (quadrilaterals, tetrahedra), 8
#define MST_CELL(MF)                                                                                            \
    if (roe)                                                                                                    \
        return second ? launch(x, MST_K_CELL, k_cell<DIM, MST_SCHEME_ROE, true, T, MF>, x->nc, fa, a)           \
                      : launch(x, MST_K_CELL, k_cell<DIM, MST_SCHEME_ROE, false, T, MF>, x->nc, fa, a);         \
    return second ? launch(x, MST_K_CELL, k_cell<DIM, MST_SCHEME_AUSM, true, T, MF>, x->nc, fa, a)              \
                  : launch(x, MST_K_CELL, k_cell<DIM, MST_SCHEME_AUSM, false, T, MF>, x->nc, fa, a);
    if (x->slots == 3) { MST_CELL(3) }
    if (x->slots == 4) { MST_CELL(4) }
    MST_CELL(8)
#undef MST_CELL
}

int resolve_strategy(mst_ctx *x);

// one residual evaluation + stage update (mode includes UPD_STAGE) with the context's strategy
int run_stage(mst_ctx *x, int mode, int is, int in, const Stage &sg, int iout) {
    if (x->resolved < 0) {
        int rc = resolve_strategy(x);
        if (rc) return rc;
    }
    if (x->resolved == MST_STRATEGY_FACE || (x->viscous && !x->visc_patch)) {
        int rc = run_face_flux(x, is);
        if (rc) return rc;
        return run_update(x, mode, is, in, sg, iout);
    }
    int rc = ensure_shadow(x, is);
    if (rc) return rc;
    if (x->viscous) {  // the patch route, whichever of the other strategies is set
        rc = run_grad_visc(x, is);
        if (rc) return rc;
        if (x->mixed)
            rc = x->dim == 2 ? run_patch_t<2, float>(x, mode, is, in, sg, iout)
                             : run_patch_t<3, float>(x, mode, is, in, sg, iout);
        else
            rc = x->dim == 2 ? run_patch_t<2, double>(x, mode, is, in, sg, iout)
                             : run_patch_t<3, double>(x, mode, is, in, sg, iout);
        if (rc == MST_OK && iout >= 0) x->shadow_ok[iout] = x->mixed;
        x->g_of = is;
        return rc;
    }
    if (x->resolved == MST_STRATEGY_FUSED) {
        if (x->mixed)
            rc = x->dim == 2 ? run_fused_t<2, float>(x, mode, is, in, sg, iout)
                             : run_fused_t<3, float>(x, mode, is, in, sg, iout);
        else
            rc = x->dim == 2 ? run_fused_t<2, double>(x, mode, is, in, sg, iout)
                             : run_fused_t<3, double>(x, mode, is, in, sg, iout);
        if (rc == MST_OK && iout >= 0) x->shadow_ok[iout] = x->mixed;
        return rc;
    }
    if (x->cfg.order >= 2) {
        rc = run_grad(x, is, false);
        if (rc) return rc;
    }
    if (x->resolved == MST_STRATEGY_PATCH) {
        if (x->mixed)
            rc = x->dim == 2 ? run_patch_t<2, float>(x, mode, is, in, sg, iout)
                             : run_patch_t<3, float>(x, mode, is, in, sg, iout);
        else
            rc = x->dim == 2 ? run_patch_t<2, double>(x, mode, is, in, sg, iout)
                             : run_patch_t<3, double>(x, mode, is, in, sg, iout);
    } else if (x->mixed) {
        rc = x->dim == 2 ? run_cell_t<2, float>(x, mode, is, in, sg, iout)
                         : run_cell_t<3, float>(x, mode, is, in, sg, iout);
    } else {
        rc = x->dim == 2 ? run_cell_t<2, double>(x, mode, is, in, sg, iout)
                         : run_cell_t<3, double>(x, mode, is, in, sg, iout);
    }
    if (rc == MST_OK && iout >= 0) x->shadow_ok[iout] = x->mixed;
    return rc;
}

// finish of f's partials: one block when they are few, else a first level of FIN_CHUNK-partial
// blocks into fin_mid and one block over those (fixed partition: bit-reproducible)
int launch_finish(mst_ctx *x, FinArgs f) {
    f.chunk = f.nblk;
    f.mid = nullptr;
    // sums keep one fixed two-level order above 2 FIN_CHUNK partials (bit-reproducible norms); a lone
    // minimum (the CFL time step) does not depend on the order: one block, one launch, up to
    // 16 FIN_CHUNK partials
    if (f.n == 1 && f.kind[0] == 1 && f.post[0] == 0 && f.nblk <= 16 * FIN_CHUNK) {
        hipLaunchKernelGGL(k_finish_min<0>, dim3(1), dim3(FIN), 0, x->stream, f.src[0], f.nblk, f.dst[0]);
        HIPCHK(hipGetLastError());
        return MST_OK;
    }
    if (f.nblk > 2 * FIN_CHUNK) {
        const int64_t g = (f.nblk + FIN_CHUNK - 1) / FIN_CHUNK;
        FinArgs a = f;
        a.chunk = FIN_CHUNK;
        a.mid = x->fin_mid;
        hipLaunchKernelGGL(k_finish, dim3((uint32_t)g), dim3(FIN), 0, x->stream, a);
        HIPCHK(hipGetLastError());
        for (int k = 0; k < f.n; k++) f.src[k] = x->fin_mid + k * g;
        f.nblk = g;
        f.chunk = g;
    }
    hipLaunchKernelGGL(k_finish, dim3(1), dim3(FIN), 0, x->stream, f);
    HIPCHK(hipGetLastError());
    return MST_OK;
}

// one finish: L2 norms (nl2 fields) and/or the minimum time step, from the per-block partials.  The norms are always
// sums over the partials of blocks of BLOCK cells, whichever patches the kernel had.
int run_finish(mst_ctx *x, int nl2, int want_dt) {
    FinArgs f;
    memset(&f, 0, sizeof(f));
    const int64_t nb = x->nblk_c;
    f.nblk = nb;
    f.count = (double)x->nc;
    const double *part = x->part;
    if (nl2 && x->l2_cnt != nb) {
        double *joined = x->part + x->n_patch * x->nv;
        hipLaunchKernelGGL(k_join_partials<0>, dim3((uint32_t)((nb * nl2 + BLOCK - 1) / BLOCK)), dim3(BLOCK), 0, x->stream,
                           x->l2_cnt, nb, nl2, part, joined);
        HIPCHK(hipGetLastError());
        part = joined;
    }
    for (int k = 0; k < nl2; k++) {
        f.src[f.n] = part + k * nb;
        f.kind[f.n] = 0;
        f.dst[f.n] = x->scal + 1 + k;
        f.post[f.n] = 1;
        f.n++;
    }
    if (want_dt) {
        const int64_t nd = x->dt_cnt[x->dt_to];
        if (nl2 && nd != nb) {  // the partials of other blocks: a finish of its own
            int rc = launch_finish(x, f);
            if (rc) return rc;
            memset(&f, 0, sizeof(f));
            f.count = (double)x->nc;
        }
        f.nblk = nd;
        f.src[f.n] = x->pdt[x->dt_to];
        f.kind[f.n] = 1;
        f.dst[f.n] = x->scal;
        f.post[f.n] = 0;
        f.n++;
    }
    return launch_finish(x, f);
}

int run_cfl(mst_ctx *x, const double *Qsrc, double cfl) {
    double *pdt = x->pdt[x->dt_to];
    partials(x, UPD_DT, x->nblk_c);
    int rc = x->dim == 2 ? launch(x, MST_K_DT, k_cfl<2>, x->nc, x->nc, Qsrc, (const double *)x->cvol,
                                  (const double *)x->cshalf, x->cfg.gamma, cfl, pdt)
                         : launch(x, MST_K_DT, k_cfl<3>, x->nc, x->nc, Qsrc, (const double *)x->cvol,
                                  (const double *)x->cshalf, x->cfg.gamma, cfl, pdt);
    if (rc) return rc;
    return run_finish(x, 0, 1);
}

template <typename T>
int dalloc(T **p, size_t n) {
    if (n == 0) n = 1;
    HIPCHK(hipMalloc((void **)p, n * sizeof(T)));
    return MST_OK;
}
template <typename T>
int dupload(T **p, const std::vector<T> &v) {
    int rc = dalloc(p, v.size());
    if (rc) return rc;
    if (!v.empty()) HIPCHK(hipMemcpy(*p, v.data(), v.size() * sizeof(T), hipMemcpyHostToDevice));
    return MST_OK;
}

// device arrays of the mixed form (allocated the first time a mixed configuration is set)
int alloc_mixed(mst_ctx *x) {
    if (x->rec32) return MST_OK;
    for (int i = 0; i < 4; i++) {
        int rc = dalloc(&x->Q32[i], x->nc * x->nv);
        if (rc) return rc;
        x->shadow_ok[i] = false;
    }
    return dalloc(&x->rec32, (int64_t)x->slots * x->nc * x->nv);
}

// incidence arrays from the padded ELL table: code, signed normal, offset (FP64, and FP32 copies
// in the mixed form); the weights follow the configuration (upload_incidence_weights)
int build_incidence(mst_ctx *x) {
    const mst::Prepared &P = x->prep.P;
    const int dim = x->dim;
    const int64_t n = (int64_t)x->slots * x->nc;
    std::vector<int32_t> code(n, -2);
    std::vector<double> nrm(n * dim, 0.0), dx(n * dim, 0.0);
    for (int s = 0; s < x->slots; s++)
        for (int64_t c = 0; c < x->nc; c++) {
            const int64_t i = (int64_t)s * x->nc + c;
            if (mst::incidence(P, s, c, code[i], &nrm[i * dim], &dx[i * dim]) >= 0) x->n_inc++;
        }
    // records of each face's sides: the incidence (s, c) whose table entry is the face
    std::vector<int32_t> r0(x->nf, -1), r1(x->nf, -1);
    for (int s = 0; s < P.maxf; s++)
        for (int64_t c = 0; c < x->nc; c++) {
            const int32_t e = P.ell[(int64_t)s * x->nc + c];
            if (e < 0) continue;
            ((e & 1) ? r1 : r0)[e >> 1] = (int32_t)((int64_t)s * x->nc + c);
        }
    int rc = dupload(&x->inc_code, code);
    if (!rc) rc = dupload(&x->inc_n, nrm);
    if (!rc) rc = dupload(&x->inc_dx, dx);
    if (!rc) rc = dalloc(&x->inc_w, n);
    if (!rc) rc = dupload(&x->frec0, r0);
    if (!rc) rc = dupload(&x->frec1, r1);
    return rc;
}

// cells per patch of the current configuration (the sweeps stand at mst_ctx::patch_cells)
int patch_cells(const mst_ctx *x) {
    const bool sub = x->nblk_c <= SUB_PATCH_MAX[x->dim - 2] && (x->dim == 2 || x->cfg.precision != MST_PREC_MIXED);
    return sub ? SUB_PATCH : BLOCK;
}

// Patch tables: for each patch of patch_cells consecutive cells, the faces that carry a flux into one of its
// cells (ascending; a face joining two of its cells once), and for each cell slot (local index << 1) |
// is_c1, or -1 for an empty slot or a zero-flux face; and each patch's halo for the fused kernel.
// The kernels keep a patch's face states and fluxes in LDS, so the strategies need at most 4 slots and
// 16 * NV bytes per face of the largest patch within 64 KiB.
// Built at creation, and again by a configuration whose patches have another size.
int build_patches(mst_ctx *x) {
    const mst::Prepared &P = x->prep.P;
    x->patch_ok = x->fused_ok = false;
    for (void **b : {(void **)&x->pstart, (void **)&x->pface, (void **)&x->pfi, (void **)&x->ploc, (void **)&x->hstart,
                     (void **)&x->hcell, (void **)&x->hloc}) {
        if (*b) (void)hipFree(*b);
        *b = nullptr;
    }
    x->hg.release();
    x->hg_dirty = true;
    x->patch_cells = patch_cells(x);
    x->n_patch = (x->nc + x->patch_cells - 1) / x->patch_cells;
    if (x->slots > 4) return MST_OK;
    const int64_t nc = x->nc, pc = x->patch_cells, nb = x->n_patch;
    std::vector<int32_t> start(nb + 1, 0), face, list, hstart(nb + 1, 0), hcell, halo;
    std::vector<int16_t> loc((size_t)x->slots * nc, -1), hloc;
    face.reserve((size_t)(nc * 2));
    size_t max_pf = 0, max_bf = 0;
    auto faces_of = [&](int64_t ca, int64_t cz) {  // list = the flux-carrying faces of cells [ca, cz)
        list.clear();
        for (int s = 0; s < P.maxf; s++)
            for (int64_t c = ca; c < cz; c++) {
                const int32_t e = P.ell[(int64_t)s * nc + c];
                if (e >= 0 && P.fkind[e >> 1] < mst::KIND_NONE) list.push_back(e >> 1);
            }
        std::sort(list.begin(), list.end());
        list.erase(std::unique(list.begin(), list.end()), list.end());
    };
    for (int64_t ca = 0; ca < nc; ca += BLOCK) {  // what a mesh may run does not depend on the size of its patches
        faces_of(ca, std::min<int64_t>(nc, ca + BLOCK));
        max_bf = std::max(max_bf, list.size());
    }
    // the fused kernel keeps 16 * NV bytes per patch face in LDS (the patch kernel half of that)
    if (max_bf * x->nv * 16 > 65536) return MST_OK;
    for (int64_t b = 0; b < nb; b++) {
        const int64_t ca = b * pc, cz = std::min(nc, ca + pc);
        faces_of(ca, cz);
        max_pf = std::max(max_pf, list.size());
        for (int s = 0; s < P.maxf; s++)
            for (int64_t c = ca; c < cz; c++) {
                const int32_t e = P.ell[(int64_t)s * nc + c];
                if (e < 0 || P.fkind[e >> 1] >= mst::KIND_NONE) continue;
                const int64_t l = std::lower_bound(list.begin(), list.end(), e >> 1) - list.begin();
                loc[(size_t)s * nc + c] = (int16_t)((l << 1) | (e & 1));
            }
        start[b] = (int32_t)face.size();
        face.insert(face.end(), list.begin(), list.end());
        // halo: the other cell of every patch face with one cell outside the patch, and for each of its
        // slots the local index of the slot's face when the face is one of the patch's
        halo.clear();
        for (const int32_t f : list) {
            if (P.fkind[f] != mst::KIND_INTERIOR && P.fkind[f] != mst::KIND_PERIODIC) continue;
            for (const int32_t c : {P.fc0[f], P.fc1[f]})
                if (c < ca || c >= cz) halo.push_back(c);
        }
        std::sort(halo.begin(), halo.end());
        halo.erase(std::unique(halo.begin(), halo.end()), halo.end());
        hstart[b] = (int32_t)hcell.size();
        for (const int32_t c : halo) {
            hcell.push_back(c);
            for (int s = 0; s < x->slots; s++) {
                const int32_t e = s < P.maxf ? P.ell[(int64_t)s * nc + c] : -1;
                int16_t v = -1;
                if (e >= 0 && P.fkind[e >> 1] < mst::KIND_NONE) {
                    const auto it = std::lower_bound(list.begin(), list.end(), e >> 1);
                    if (it != list.end() && *it == (e >> 1)) v = (int16_t)(((it - list.begin()) << 1) | (e & 1));
                }
                hloc.push_back(v);
            }
        }
    }
    start[nb] = (int32_t)face.size();
    hstart[nb] = (int32_t)hcell.size();
    int rc = dupload(&x->pstart, start);
    if (!rc) rc = dupload(&x->pface, face);
    if (!rc && x->nf < ((int64_t)1 << FI_SHIFT)) rc = dalloc(&x->pfi, face.size());  // packed by upload_config
    if (!rc) rc = dupload(&x->ploc, loc);
    if (!rc) rc = dupload(&x->hstart, hstart);
    if (!rc) rc = dupload(&x->hcell, hcell);
    if (!rc) rc = dupload(&x->hloc, hloc);
    if (rc) return rc;
    x->n_halo = (int64_t)hcell.size();
    x->max_pf = (int)max_pf;
    x->n_psolve = (int64_t)face.size();
    x->patch_ok = true;
    x->fused_ok = fused_lds_bytes(x->dim, x->nv, (int)max_bf, false, x->dim == 2) <= 65536;
    return MST_OK;
}

// per incidence: FP64 eta of the face (with the last-interior-face quirk), FP32 the difference-form
// weight (1 - eta on the c0 side, eta on the c1 side)
int upload_incidence_weights(mst_ctx *x, const std::vector<double> &eta) {
    const mst::Prepared &P = x->prep.P;
    const int64_t n = (int64_t)x->slots * x->nc;
    std::vector<double> w(n, 0.0);
    std::vector<float> w32(x->mixed ? n : 0, 0.f);
    for (int s = 0; s < P.maxf; s++)
        for (int64_t c = 0; c < x->nc; c++) {
            const int32_t e = P.ell[(int64_t)s * x->nc + c];
            if (e < 0) continue;
            const int64_t i = (int64_t)s * x->nc + c;
            w[i] = eta[e >> 1];
            if (x->mixed) {
                const float ef = (float)eta[e >> 1];
                w32[i] = (e & 1) ? ef : 1.0f - ef;
            }
        }
    HIPCHK(hipMemcpy(x->inc_w, w.data(), sizeof(double) * n, hipMemcpyHostToDevice));
    if (x->mixed) {
        if (!x->inc_w32) {
            const int dim = x->dim;
            int rc = dalloc(&x->inc_w32, n);
            if (rc) return rc;
            std::vector<double> h(n * dim);
            std::vector<float> f(n * dim);
            for (auto pr : {std::make_pair(x->inc_n, &x->inc_n32), std::make_pair(x->inc_dx, &x->inc_dx32)}) {
                if (dim == 3 && pr.second == &x->inc_n32) {  // weighted normals, filled below
                    rc = dalloc(&x->inc_n32, n * dim);
                    if (rc) return rc;
                    continue;
                }
                HIPCHK(hipMemcpy(h.data(), pr.first, sizeof(double) * h.size(), hipMemcpyDeviceToHost));
                for (size_t k = 0; k < h.size(); k++) f[k] = (float)h[k];
                rc = dupload(pr.second, f);
                if (rc) return rc;
            }
            rc = dalloc(&x->ivol32, x->nc);
            if (rc) return rc;
            hipLaunchKernelGGL(k_recip_vol<0>, dim3((uint32_t)((x->nc + BLOCK - 1) / BLOCK)), dim3(BLOCK), 0, x->stream,
                               x->nc, (const double *)x->cvol, x->ivol32);
            HIPCHK(hipGetLastError());
        }
        HIPCHK(hipMemcpy(x->inc_w32, w32.data(), sizeof(float) * n, hipMemcpyHostToDevice));
        if (x->dim == 3) {  // the FP32 3D gradient reads the weights folded into its normals
            hipLaunchKernelGGL(k_weighted_normals<3>, dim3((uint32_t)((n + BLOCK - 1) / BLOCK)), dim3(BLOCK), 0, x->stream,
                               n, (const int32_t *)x->inc_code, (const double *)x->inc_w, (const double *)x->inc_n,
                               x->inc_n32);
            HIPCHK(hipGetLastError());
        }
    }
    x->hg_dirty = true;
    return MST_OK;
}

// the LU-SGS sweeps' face words, from the current kinds and masks (nothing before the colours are built)
int lu_finfo(mst_ctx *x) {
    if (!x->lu_info) return MST_OK;
    hipLaunchKernelGGL(k_lu_finfo<0>, dim3((uint32_t)((x->nc + BLOCK - 1) / BLOCK)), dim3(BLOCK), 0, x->stream, x->nc,
                       x->slots, (const int32_t *)x->lu_face, (const int32_t *)x->finfo, x->lu_info);
    HIPCHK(hipGetLastError());
    return MST_OK;
}

int upload_config(mst_ctx *x) {
    std::vector<int32_t> mask;
    mst::lr_masks(x->prep.P, x->cfg.compat, mask);
    std::vector<int32_t> info(x->nf);
    for (int64_t i = 0; i < x->nf; i++) info[i] = x->prep.P.fkind[i] | (mask[i] << 4);
    HIPCHK(hipMemcpy(x->finfo, info.data(), sizeof(int32_t) * x->nf, hipMemcpyHostToDevice));
    if (x->pfi && x->n_psolve > 0) {  // the patch face entries with the new kinds and masks
        const int64_t n = x->n_psolve;
        hipLaunchKernelGGL(k_pack_faces<0>, dim3((uint32_t)((n + BLOCK - 1) / BLOCK)), dim3(BLOCK), 0, x->stream, n,
                           (const int32_t *)x->pface, (const int32_t *)x->finfo, x->pfi);
        HIPCHK(hipGetLastError());
    }
    int rc = lu_finfo(x);
    if (rc) return rc;
    std::vector<double> eta = x->prep.P.feta;
    if ((x->cfg.compat & MST_COMPAT_GRAD_LASTINT) && x->prep.P.quirk_face >= 0) eta[x->prep.P.quirk_face] = 1.0;
    HIPCHK(hipMemcpy(x->feta, eta.data(), sizeof(double) * x->nf, hipMemcpyHostToDevice));
    x->p64 = make_params<double>(x->cfg);
    x->p32 = make_params<float>(x->cfg);
    x->mixed = x->cfg.precision == MST_PREC_MIXED;
    x->viscous = x->cfg.mu > 0 || x->cfg.kappa > 0;
    // (a face of unknown type is in no patch list, but its cell's viscous flux counts: the face route)
    x->visc_patch = x->patch_ok && std::find(x->prep.P.fkind.begin(), x->prep.P.fkind.end(), (int32_t)mst::KIND_NONE) ==
                                       x->prep.P.fkind.end();
    if (x->viscous && !x->gw) {
        rc = dalloc(&x->gw, (size_t)(x->nc * (x->dim + 1) * x->dim));
        if (rc) return rc;
    }
    if (x->mixed) {
        rc = alloc_mixed(x);
        if (rc) return rc;
        for (int i = 0; i < 4; i++) x->shadow_ok[i] = false;
    }
    return upload_incidence_weights(x, eta);
}

void release(mst_ctx *x) {
    if (!x) return;
    void *bufs[] = {x->fc0, x->fc1, x->finfo, x->ell, x->fn, x->fxf, x->pxf, x->feta, x->cvol, x->cxc,
                    x->cshalf, x->Q[0], x->Q[1], x->Q[2], x->Q[3], x->G, x->rec, x->graw, x->phi, x->R,
                    x->scal, x->part, x->fin_mid, x->bad, x->Q32[0], x->Q32[1], x->Q32[2], x->Q32[3], x->rec32,
                    x->frec0, x->frec1, x->inc_code, x->inc_w, x->inc_n, x->inc_dx, x->inc_w32, x->inc_n32,
                    x->inc_dx32, x->ivol32, x->pstart, x->pface, x->pfi, x->ploc, x->hstart, x->hcell, x->hloc,
                    x->lu_cells, x->lu_nb, x->lu_face, x->lu_info, x->lu_n, x->lu_r, x->lu_D, x->lu_dQ, x->gw, x->cnew, x->pdt[0], x->pdt[1]};
    for (void *b : bufs)
        if (b) (void)hipFree(b);
    x->hg.release();
    x->link.release();
    for (int k = 0; k < MST_K_COUNT; k++)
        for (auto &pr : x->ev[k]) {
            (void)hipEventDestroy(pr.first);
            (void)hipEventDestroy(pr.second);
        }
    for (auto e : x->pool) (void)hipEventDestroy(e);
    if (x->board) (void)hipHostFree(x->board);
    if (x->stream) (void)hipStreamDestroy(x->stream);
    delete x;
}

int fetch_cells(mst_ctx *x, const double *dsrc, int width, double *out) {
    HIPCHK(x->link.fetch(x->stream, x->nc, width, x->cnew, dsrc, out));
    return MST_OK;
}

// max |new - old| / old per field
template <int NV>
int run_monitor(mst_ctx *x, double *out) {
    const int64_t n = std::min(x->nblk_c, MONITOR_GRID);
    int rc = launch(x, -1, k_maxrel<NV>, n * BLOCK, x->nc, (const double *)x->Q[x->inew], (const double *)x->Q[x->iold],
                    x->part);
    if (rc) return rc;
    const uint32_t seq = ++x->board_seq;
    const double *part = x->part;
    if (n <= 2 * BLOCK)
        hipLaunchKernelGGL((k_finish_max<NV, BLOCK, 1>), dim3(1), dim3(BLOCK), 0, x->stream, part, n, x->board, seq);
    else if (n <= 8 * BLOCK)
        hipLaunchKernelGGL((k_finish_max<NV, BLOCK, 8>), dim3(1), dim3(BLOCK), 0, x->stream, part, n, x->board, seq);
    else
        hipLaunchKernelGGL((k_finish_max<NV, FIN, 8>), dim3(1), dim3(FIN), 0, x->stream, part, n, x->board, seq);
    HIPCHK(hipGetLastError());
    HIPCHK(board_wait(x->board, seq, x->stream));
    for (int k = 0; k < NV; k++) out[k] = x->board->mon[k];
    return MST_OK;
}

// scal and the bad flag on the board, after the stream's earlier work
int report(mst_ctx *x, bool take_bad) {
    hipLaunchKernelGGL(k_report, dim3(1), dim3(64), 0, x->stream, (const double *)x->scal, x->bad, (int)take_bad, x->board,
                       ++x->board_seq);
    HIPCHK(hipGetLastError());
    HIPCHK(board_wait(x->board, x->board_seq, x->stream));
    return MST_OK;
}

int check_bad(mst_ctx *x) {
    int rc = report(x, true);
    if (rc) return rc;
    if (x->board->bad) {
        return mst::fail(MST_E_STATE, "non-physical state (rho<=0, p<=0 or NaN, or no positive time step) produced by the update");
    }
    return MST_OK;
}

// LU-SGS: the cell colouring (prep.cpp, lusgs_colours), the cells sorted by colour (ascending inside
// a colour), and per (slot, position) the neighbour record and the cell's outward normal.  Built once
// per context, on the first implicit iteration.
int build_colours(mst_ctx *x) {
    if (x->lu_cells) return MST_OK;
    if (x->nc >= ((int64_t)1 << 29)) return mst::fail(MST_E_UNSUPPORTED, "LU-SGS records hold cell indices below 2^29");
    const auto &P = x->prep.P;
    const int64_t nc = x->nc;
    const int dim = x->dim;
    std::vector<int32_t> col;
    const int ncol = lusgs_colours(P, col);
    std::vector<int64_t> start(ncol + 1, 0);
    for (int64_t c = 0; c < nc; c++) start[col[c] + 1]++;
    for (int k = 0; k < ncol; k++) start[k + 1] += start[k];
    std::vector<int32_t> cells(nc);
    std::vector<int64_t> fill(start.begin(), start.end() - 1);
    for (int64_t c = 0; c < nc; c++) cells[fill[col[c]]++] = (int32_t)c;
    const int64_t slots = x->slots;
    std::vector<int32_t> nb(slots * nc, -2), fcode(slots * nc, -1);
    std::vector<double> nrm(slots * nc * dim, 0.0);
    for (int64_t t = 0; t < nc; t++) {
        const int64_t c = cells[t];
        for (int s = 0; s < P.maxf; s++) {
            const int32_t e = P.ell[(int64_t)s * nc + c];
            if (e < 0) break;
            const int32_t f = e >> 1;
            const bool c1side = e & 1;
            const int32_t o = c1side ? P.fc0[f] : P.fc1[f];
            const int64_t i = (int64_t)s * nc + t;
            for (int d = 0; d < dim; d++) nrm[i * dim + d] = c1side ? -P.fn[(int64_t)f * dim + d] : P.fn[(int64_t)f * dim + d];
            nb[i] = o < 0 ? -1 : ((o << 2) | (col[o] < col[c] ? 1 : 0) | (col[o] > col[c] ? 2 : 0));
            fcode[i] = e;
        }
    }
    int rc = dupload(&x->lu_cells, cells);
    if (rc == MST_OK) rc = dupload(&x->lu_nb, nb);
    if (rc == MST_OK) rc = dupload(&x->lu_face, fcode);
    if (rc == MST_OK) rc = dupload(&x->lu_n, nrm);
    if (rc == MST_OK) rc = dalloc(&x->lu_r, (size_t)(slots * nc));
    if (rc == MST_OK) rc = dalloc(&x->lu_D, (size_t)nc);
    if (rc == MST_OK) rc = dalloc(&x->lu_dQ, (size_t)(nc * x->nv));
    if (rc == MST_OK && !x->R) rc = dalloc(&x->R, (size_t)(nc * x->nv));
    if (rc == MST_OK) rc = dalloc(&x->lu_info, (size_t)nc);
    if (rc == MST_OK) rc = lu_finfo(x);
    if (rc) return rc;
    x->lu_start = start;
    x->lu_colour = std::move(col);
    return MST_OK;
}

// what the sweeps of each colour touch: its cells, their incidences (inc_hi: toward cells of a higher colour), and the
// distinct neighbours of lower and of higher colour
struct LuCount {
    int64_t n = 0, inc = 0, inc_hi = 0, lo = 0, hi = 0;
};

std::vector<LuCount> lu_counts(const mst_ctx *x) {
    const auto &P = x->prep.P;
    const auto &col = x->lu_colour;
    const int64_t nc = x->nc;
    std::vector<LuCount> count(x->lu_start.size() - 1);
    std::vector<int32_t> seen(nc, -1);  // the colour that last counted the cell as a neighbour
    for (size_t k = 0; k < count.size(); k++) count[k].n = x->lu_start[k + 1] - x->lu_start[k];
    for (int s = 0; s < P.maxf; s++)
        for (int64_t c = 0; c < nc; c++) {
            const int32_t e = P.ell[(int64_t)s * nc + c];
            if (e < 0) continue;
            const int32_t o = (e & 1) ? P.fc0[e >> 1] : P.fc1[e >> 1];
            count[col[c]].inc++;
            if (o >= 0 && col[o] > col[c]) count[col[c]].inc_hi++;
        }
    for (size_t k = 0; k < count.size(); k++)  // (a colour at a time: `seen` holds one)
        for (int s = 0; s < P.maxf; s++)
            for (int64_t c = 0; c < nc; c++) {
                const int32_t e = col[c] == (int32_t)k ? P.ell[(int64_t)s * nc + c] : -1;
                if (e < 0) continue;
                const int32_t o = (e & 1) ? P.fc0[e >> 1] : P.fc1[e >> 1];
                if (o < 0 || col[o] == (int32_t)k || seen[o] == (int32_t)k) continue;
                seen[o] = (int32_t)k;
                (col[o] < (int32_t)k ? count[k].lo : count[k].hi)++;
            }
    return count;
}

template <typename K>
int launch_lu(mst_ctx *x, K kernel, const LuArgs &a, int64_t t0, int64_t n) {
    return launch_nt(x, MST_K_LUSGS, kernel, (n + LU_BLOCK - 1) / LU_BLOCK * BLOCK, LU_BLOCK, 0, a, t0, n);
}

// forward launches; RS >= 0: the first-order residual computed by the sweep (scheme RS)
template <int DIM, int MAXF, int RS>
int lu_forward(mst_ctx *x, const LuArgs &a) {
    const int ncol = (int)x->lu_start.size() - 1;
    int rc = MST_OK;
    for (int k = 0; k < ncol && rc == MST_OK; k++) {
        const int64_t t0 = x->lu_start[k], n = x->lu_start[k + 1] - t0;
        rc = k == ncol - 1 ? launch_lu(x, k_lu_sweep<DIM, true, true, MAXF, RS>, a, t0, n)
                           : launch_lu(x, k_lu_sweep<DIM, true, false, MAXF, RS>, a, t0, n);
    }
    return rc;
}

template <int DIM, int MAXF>
int lu_sweeps(mst_ctx *x, const LuArgs &a, bool inline_res) {
    const int ncol = (int)x->lu_start.size() - 1;
    int rc;
    if constexpr (MAXF <= 4) {
        if (inline_res)
            rc = x->cfg.scheme == MST_SCHEME_ROE ? lu_forward<DIM, MAXF, MST_SCHEME_ROE>(x, a)
                                                 : lu_forward<DIM, MAXF, MST_SCHEME_AUSM>(x, a);
        else
            rc = lu_forward<DIM, MAXF, -1>(x, a);
    } else {
        rc = lu_forward<DIM, MAXF, -1>(x, a);
    }
    for (int k = ncol - 2; k >= 0 && rc == MST_OK; k--) {
        const int64_t t0 = x->lu_start[k], n = x->lu_start[k + 1] - t0;
        rc = launch_lu(x, k_lu_sweep<DIM, false, false, MAXF>, a, t0, n);
    }
    return rc;
}

// the sweeps' arguments for the current Old (the iteration's start) and New buffers
LuArgs lu_args(const mst_ctx *x) {
    LuArgs a;
    memset(&a, 0, sizeof(a));  // the batch-only fields (pcase, gam, active, G) stay null: single context
    a.nc = x->nc;
    a.cells = x->lu_cells;
    a.nb = x->lu_nb;
    a.n = x->lu_n;
    a.r = x->lu_r;
    a.D = x->lu_D;
    a.Q = x->Q[x->iold];
    a.R = x->R;
    a.dQ = x->lu_dQ;
    a.Qout = x->Q[x->inew];
    a.bad = x->bad;
    a.gamma = x->cfg.gamma;
    a.omega = x->lu_omega;
    a.dscale = 1.0 / x->lu_cfl + 0.5 * x->lu_omega;
    a.finfo = x->lu_info;
    a.P = x->p64;
    return a;
}

// one LU-SGS iteration: residual of Old (+ its L2 norms when l2 is set), the two sweeps into New
int lu_iteration(mst_ctx *x, bool l2) {
    int rc = MST_OK;
    const int mode = l2 ? UPD_L2 : UPD_RESIDUAL;
    // order 1, FP64, inviscid, cells of <= 4 faces: the forward sweeps compute the residual themselves
    // (the norms of a call's last iteration still come from the residual kernel)
    x->lu_inline = x->cfg.order == 1 && !x->mixed && !x->viscous && x->slots <= 4;
    const bool inline_res = !l2 && x->lu_inline;
    if (inline_res) {
        // nothing to launch before the sweeps
    } else if (x->patch_ok && !x->mixed && !x->viscous) {  // one launch: the patch kernel's residual-only form (same R)
        if (x->cfg.order >= 2) {
            rc = run_grad(x, x->iold, false);
            if (rc) return rc;
        }
        rc = x->dim == 2 ? run_patch_residual_t<2>(x, mode, x->iold) : run_patch_residual_t<3>(x, mode, x->iold);
    } else {
        rc = run_face_flux(x, x->iold);
        if (rc) return rc;
        rc = run_update(x, mode, x->iold, -1, Stage{0, 0}, -1);
    }
    if (rc) return rc;
    if (l2) {
        rc = run_finish(x, x->nv, 0);
        if (rc) return rc;
    }
    const LuArgs a = lu_args(x);
    // the records are padded to the slot count of the device table (3, 4 or 8)
    if (x->dim == 2) {
        if (x->slots == 3) return lu_sweeps<2, 3>(x, a, inline_res);
        if (x->slots == 4) return lu_sweeps<2, 4>(x, a, inline_res);
        return lu_sweeps<2, 8>(x, a, inline_res);
    }
    if (x->slots == 3) return lu_sweeps<3, 3>(x, a, inline_res);
    if (x->slots == 4) return lu_sweeps<3, 4>(x, a, inline_res);
    return lu_sweeps<3, 8>(x, a, inline_res);
}

// n >= 1 consecutive iterations with the residual computed in the forward sweeps (lu_inline, two
// colours or more): colour 0's backward sweep of each iteration but the last runs fused with the next
// iteration's forward sweep of colour 0 (k_lu_sweep_bf), 2 K - 2 launches per iteration for K colours
// instead of 2 K - 1, with the same results.  Each iteration ends with the Old/New swap.
template <int DIM, int MAXF, int RS>
int lu_inline_run(mst_ctx *x, int n) {
    const int ncol = (int)x->lu_start.size() - 1;
    const int64_t n0 = x->lu_start[1] - x->lu_start[0];
    int rc = MST_OK;
    for (int it = 0; it < n && rc == MST_OK; it++) {
        const LuArgs a = lu_args(x);
        for (int k = it == 0 ? 0 : 1; k < ncol && rc == MST_OK; k++) {  // colour 0: done by the fused launch
            const int64_t t0 = x->lu_start[k], m = x->lu_start[k + 1] - t0;
            rc = k == ncol - 1 ? launch_lu(x, k_lu_sweep<DIM, true, true, MAXF, RS>, a, t0, m)
                               : launch_lu(x, k_lu_sweep<DIM, true, false, MAXF, RS>, a, t0, m);
        }
        for (int k = ncol - 2; k >= 1 && rc == MST_OK; k--) {
            const int64_t t0 = x->lu_start[k], m = x->lu_start[k + 1] - t0;
            rc = launch_lu(x, k_lu_sweep<DIM, false, false, MAXF>, a, t0, m);
        }
        if (rc) break;
        rc = it < n - 1 ? launch_lu(x, k_lu_sweep_bf<DIM, MAXF, RS>, a, x->lu_start[0], n0)
                        : launch_lu(x, k_lu_sweep<DIM, false, false, MAXF>, a, x->lu_start[0], n0);
        x->shadow_ok[x->inew] = false;
        std::swap(x->iold, x->inew);
    }
    return rc;
}

template <int DIM, int MAXF>
int lu_inline_run_s(mst_ctx *x, int n) {
    return x->cfg.scheme == MST_SCHEME_ROE ? lu_inline_run<DIM, MAXF, MST_SCHEME_ROE>(x, n)
                                           : lu_inline_run<DIM, MAXF, MST_SCHEME_AUSM>(x, n);
}

int lu_inline_iterations(mst_ctx *x, int n) {
    if (x->dim == 2) return x->slots == 3 ? lu_inline_run_s<2, 3>(x, n) : lu_inline_run_s<2, 4>(x, n);
    return x->slots == 3 ? lu_inline_run_s<3, 3>(x, n) : lu_inline_run_s<3, 4>(x, n);
}


// x->resolved = the fastest of the n candidates: REPS stages of each are timed in each round, outputs to a spare state
// buffer (the Old and New states are untouched).  Stages of a few microseconds: the rounds are queued behind each
// other and the better one counts.  (Three stages from an empty queue, 12 us of launches, picked an 8.5 us kernel over a
// 5.6 us one about every other time.)
int time_strategies(mst_ctx *x, const int *cand, int n, int rounds) {
    constexpr int REPS = 3;
    int spare = 0;
    while (spare == x->iold || spare == x->inew) spare++;
    const bool timing = x->timing;
    x->timing = false;
    hipEvent_t ev[16] = {};
    hipError_t e = hipSuccess;
    int rc = MST_OK;
    for (int k = 0; k < 2 * rounds * n && e == hipSuccess; k++) e = hipEventCreate(&ev[k]);
    for (int k = 0; k < rounds * n && !rc && e == hipSuccess; k++) {
        x->resolved = cand[k % n];
        if (k < n) rc = run_stage(x, UPD_STAGE, x->iold, x->iold, Stage{}, spare);  // warm-up
        if (!rc) e = hipEventRecord(ev[2 * k], x->stream);
        for (int r = 0; r < REPS && !rc; r++) rc = run_stage(x, UPD_STAGE, x->iold, x->iold, Stage{}, spare);
        if (!rc && e == hipSuccess) e = hipEventRecord(ev[2 * k + 1], x->stream);
    }
    x->timing = timing;
    // waits for the trials; they may have flagged their (unchecked) outputs, e.g. with no time step set yet
    if (!rc) rc = report(x, true);
    if (!rc && e == hipSuccess) e = hipEventSynchronize(ev[2 * rounds * n - 1]);
    float best = INFINITY;
    x->resolved = cand[0];
    for (int k = 0; k < rounds * n && !rc && e == hipSuccess; k++) {
        float ms = 0;
        if (hipEventElapsedTime(&ms, ev[2 * k], ev[2 * k + 1]) == hipSuccess && ms < best) {
            best = ms;
            x->resolved = cand[k % n];
        }
    }
    for (hipEvent_t v : ev)
        if (v) (void)hipEventDestroy(v);
    HIPCHK(e);
    return rc;
}

// Blocks up to which AUTO looks no further than the patch kernels, where a mesh has patch tables.  On 20 meshes of 2 to
// 131,072 triangles, quadrilaterals and tetrahedra, both orders, schemes and precisions, viscous or not, a stage of the
// face or the cell strategy took 1.03 to 1.65 times the better of patch and fused (mixed 3D AUSM on 10,368 cells: the
// same, 14.7 us); at 140,000 to 162,000 cells 1.06 to 1.37.  So a first step of order 1, or in 3D FP64, costs no trial
// there, and another of order 2 14 stages: about 150 us, where timing all four well enough took 600 to 1,500.
constexpr int64_t AUTO_PATCH_MAX = 512;

// AUTO: the strategy for this mesh and configuration.  Where more than one can be the fastest, a few stages of each are
// timed (outputs go to a spare state buffer; the Old and New states are untouched).
int resolve_strategy(mst_ctx *x) {
    if (x->strategy != MST_STRATEGY_AUTO) {
        x->resolved = x->strategy;
        return MST_OK;
    }
    const bool few = x->patch_ok && x->nblk_c <= AUTO_PATCH_MAX;
    int cand[4], n = 0;
    if (x->viscous) {  // two routes: the face strategy's, and the patch route under any other
        if (!few || !x->visc_patch) cand[n++] = MST_STRATEGY_FACE;
        if (x->visc_patch) cand[n++] = MST_STRATEGY_PATCH;
    } else {
        if (!few) {
            cand[n++] = MST_STRATEGY_FACE;
            cand[n++] = MST_STRATEGY_CELL;
        }
        if (x->patch_ok) cand[n++] = MST_STRATEGY_PATCH;
        // (order 1: the patch kernel; small FP64 meshes in 3D: 1.00 to 1.39 times the patch kernels' time, so no trial)
        if (x->fused_ok && x->cfg.order >= 2 && (!few || x->dim == 2 || x->mixed)) cand[n++] = MST_STRATEGY_FUSED;
    }
    x->resolved = cand[0];
    if (n > 1) {
        const int rc = time_strategies(x, cand, n, few ? 2 : 1);
        if (rc) return rc;
    }
    if (x->resolved != MST_STRATEGY_FUSED) {  // the fused kernel's halo copy (0.64 N_c entries in 3D) is not kept
        x->hg.release();
        x->hg_dirty = true;
    }
    return MST_OK;
}

}  // namespace

#define CTX_GUARD(x)                                           \
    if (!(x)) return mst::fail(MST_E_ARG, "null context");

// ------------------------------------------------------------------ allocation-free monitor
// The monitor over caller-owned device states, for callers that cannot allocate.  Its only scratch,
// one partial maximum per block and field, lives in the file-scope array below: NOALLOC_GRID blocks
// stride over any number of cells, so the array never grows.  Each device holds its own copy; its
// address is looked up once per device (hipGetSymbolAddress, with that device current) and kept.
// Every block writes its partials before the finish reads them, so nothing needs clearing between
// calls; calls that overlap on one device share the array and race.
namespace {
constexpr int NOALLOC_GRID = 2048;
constexpr int NOALLOC_MAX_DEVICES = 64;
__device__ __align__(256) double scratch[NOALLOC_GRID * 5];
std::mutex noalloc_mu;
double *noalloc_scratch[NOALLOC_MAX_DEVICES];

int noalloc_scratch_ptr(double **out) {
    int dev = -1;
    HIPCHK(hipGetDevice(&dev));
    if (dev < 0 || dev >= NOALLOC_MAX_DEVICES) return mst::fail(MST_E_UNSUPPORTED, "device index out of range");
    std::lock_guard<std::mutex> g(noalloc_mu);
    if (!noalloc_scratch[dev]) {
        void *p = nullptr;
        HIPCHK(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        if (!p) return mst::fail(MST_E_HIP, "hipGetSymbolAddress returned no address for the monitor scratch");
        noalloc_scratch[dev] = static_cast<double *>(p);
    }
    *out = noalloc_scratch[dev];
    return MST_OK;
}
}  // namespace

extern "C" {

int mst_ctx_create(const mst_mesh *m, const mst_config *cfg, mst_ctx **out) {
    if (!m || !out) return mst::fail(MST_E_ARG, "null argument");
    *out = nullptr;
    int rc = check_config(cfg);
    if (rc) return rc;
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev <= 0)
        return mst::fail(MST_E_HIP, "no HIP device available: the residual path runs only on the GPU");
    mst_ctx *x = new (std::nothrow) mst_ctx();
    if (!x) return mst::fail(MST_E_ARG, "out of host memory");
    try {
        rc = mst::prepare(*m, x->prep.P);
    } catch (const std::bad_alloc &) {
        rc = mst::fail(MST_E_ARG, "out of host memory");
    }
    if (rc) {
        delete x;
        return rc;
    }
    if (x->prep.P.bad_cells > 0) {
        rc = mst::fail(MST_E_MESH, std::to_string(x->prep.P.bad_cells) + " cells have non-positive or NaN volume "
                                   "(first: file cell " + std::to_string(x->prep.P.first_bad_cell) + ")");
        delete x;
        return rc;
    }
    const mst::Prepared &P = x->prep.P;
    x->cfg = *cfg;
    x->dim = P.dim;
    x->nv = P.nv;
    x->maxf = P.maxf;
    x->nc = P.nc;
    x->nf = P.nf;
    x->nblk_c = (x->nc + BLOCK - 1) / BLOCK;
    x->nblk_f = (x->nf + BLOCK - 1) / BLOCK;
    x->wide_patch = x->nblk_c <= (x->dim == 3 ? 512 : 256);
#define TRY(e)            \
    do {                  \
        int _r = (e);     \
        if (_r) {         \
            release(x);   \
            return _r;    \
        }                 \
    } while (0)
    if (hipGetDevice(&x->device) != hipSuccess) {
        delete x;
        return mst::fail(MST_E_HIP, "hipGetDevice failed");
    }
    if (hipStreamCreate(&x->stream) != hipSuccess) {
        delete x;
        return mst::fail(MST_E_HIP, "hipStreamCreate failed");
    }
    TRY(dupload(&x->fc0, P.fc0));
    TRY(dupload(&x->fc1, P.fc1));
    TRY(dalloc(&x->finfo, x->nf));
    {
        // the gather loops are instantiated for 3, 4 or 8 slots: pad the slot-major table with empty
        // rows up to that count so an unrolled loop over a full cell never reads past it
        const int64_t slots = x->maxf <= 3 ? 3 : (x->maxf <= 4 ? 4 : 8);
        x->slots = (int)slots;
        if (slots * x->nc >= (int64_t)INT32_MAX) {  // incidence records are indexed in 32 bits
            release(x);
            return mst::fail(MST_E_UNSUPPORTED, "mesh too large: cells x face slots must stay below 2^31");
        }
        std::vector<int32_t> ell(P.ell);
        ell.resize(slots * x->nc, -1);
        TRY(dupload(&x->ell, ell));
    }

    TRY(dupload(&x->fn, P.fn));
    TRY(dupload(&x->fxf, P.fxf));
    TRY(dupload(&x->pxf, P.pxf));
    TRY(dalloc(&x->feta, x->nf));
    TRY(dupload(&x->cvol, P.cvol));
    TRY(dupload(&x->cxc, P.cxc));
    TRY(dupload(&x->cshalf, P.cshalf));
    TRY(dupload(&x->cnew, P.cell_new_of_old));
    x->link.most = x->nc * x->nv;
    for (int i = 0; i < 4; i++) TRY(dalloc(&x->Q[i], x->nc * x->nv));
    TRY(dalloc(&x->G, x->nf * x->nv));
    TRY(dalloc(&x->rec, (int64_t)x->slots * x->nc * x->nv));
    TRY(dalloc(&x->scal, 16));
    // (a configuration may change the size of the patches)
    const int64_t most = x->nblk_c <= SUB_PATCH_MAX[x->dim - 2] ? (x->nc + SUB_PATCH - 1) / SUB_PATCH : x->nblk_c;
    TRY(dalloc(&x->part, std::max(most + x->nblk_c, x->nblk_f) * x->nv + 16));
    for (int i = 0; i < 2; i++) TRY(dalloc(&x->pdt[i], most));
    TRY(dalloc(&x->fin_mid, 12 * (x->nblk_c / FIN_CHUNK + 2)));
    TRY(dalloc(&x->bad, 1));
    if (hipHostMalloc((void **)&x->board, sizeof(Board), hipHostMallocCoherent) != hipSuccess) {
        release(x);
        return mst::fail(MST_E_HIP, "hipHostMalloc failed");
    }
    memset(x->board, 0, sizeof(Board));
    if (hipMemset(x->bad, 0, sizeof(int)) != hipSuccess || hipMemset(x->scal, 0, 16 * sizeof(double)) != hipSuccess ||
        hipMemset(x->rec, 0, sizeof(double) * x->slots * x->nc * x->nv) != hipSuccess) {
        release(x);
        return mst::fail(MST_E_HIP, "hipMemset failed");
    }
    TRY(build_incidence(x));
    TRY(build_patches(x));
    TRY(upload_config(x));
#undef TRY
    *out = x;
    return MST_OK;
}

int mst_ctx_destroy(mst_ctx *ctx) {
    if (!ctx) return MST_OK;
    (void)hipStreamSynchronize(ctx->stream);
    release(ctx);
    return MST_OK;
}

int mst_ctx_set_config(mst_ctx *ctx, const mst_config *cfg) {
    CTX_GUARD(ctx);
    int rc = check_config(cfg);
    if (rc) return rc;
    rc = ensure_fluxes(ctx);
    if (rc) return rc;
    HIPCHK(hipStreamSynchronize(ctx->stream));
    ctx->cfg = *cfg;
    ctx->dt_valid = false;
    if (ctx->strategy == MST_STRATEGY_AUTO) ctx->resolved = -1;  // the best strategy depends on the configuration
    if (ctx->patch_ok && patch_cells(ctx) != ctx->patch_cells) {
        rc = build_patches(ctx);
        if (rc) return rc;
    }
    return upload_config(ctx);
}

const mst_prep *mst_ctx_prep(const mst_ctx *ctx) { return ctx ? &ctx->prep : nullptr; }

int mst_set_state(mst_ctx *ctx, const double *Q, int64_t n_cells) {
    CTX_GUARD(ctx);
    if (!Q || n_cells != ctx->nc) return mst::fail(MST_E_ARG, "state size does not match the mesh");
    if (ctx->g_of == ctx->iold) {
        int rc = ensure_fluxes(ctx);
        if (rc) return rc;
    }
    HIPCHK(ctx->link.put(ctx->stream, ctx->nc, ctx->nv, ctx->cnew, Q, &ctx->Q[ctx->iold], 1));
    ctx->shadow_ok[ctx->iold] = false;
    ctx->dt_valid = false;
    return MST_OK;
}

int mst_get_state(mst_ctx *ctx, double *Q, int64_t n_cells) {
    CTX_GUARD(ctx);
    if (!Q || n_cells != ctx->nc) return mst::fail(MST_E_ARG, "state size does not match the mesh");
    return fetch_cells(ctx, ctx->Q[ctx->iold], ctx->nv, Q);
}

int mst_get_new_state(mst_ctx *ctx, double *Q, int64_t n_cells) {
    CTX_GUARD(ctx);
    if (!Q || n_cells != ctx->nc) return mst::fail(MST_E_ARG, "state size does not match the mesh");
    return fetch_cells(ctx, ctx->Q[ctx->inew], ctx->nv, Q);
}

int mst_set_dt(mst_ctx *ctx, double dt) {
    CTX_GUARD(ctx);
    if (!(dt > 0)) return mst::fail(MST_E_ARG, "dt must be positive");
    hipLaunchKernelGGL(k_store, dim3(1), dim3(1), 0, ctx->stream, ctx->scal, dt);
    HIPCHK(hipGetLastError());
    ctx->dt_valid = false;
    return MST_OK;
}

int mst_face_flux(mst_ctx *ctx) {
    CTX_GUARD(ctx);
    return run_face_flux(ctx, ctx->iold);
}

int mst_residual_update(mst_ctx *ctx) {
    CTX_GUARD(ctx);
    int rc = ensure_fluxes(ctx);
    if (rc) return rc;
    rc = run_update(ctx, UPD_STAGE | UPD_CHECK, ctx->iold, ctx->iold, Stage{}, ctx->inew);
    if (rc) return rc;
    return check_bad(ctx);
}

int mst_solve(mst_ctx *ctx) {
    CTX_GUARD(ctx);
    int rc = run_stage(ctx, UPD_STAGE | UPD_CHECK, ctx->iold, ctx->iold, Stage{}, ctx->inew);
    if (rc) return rc;
    return check_bad(ctx);
}

int mst_set_strategy(mst_ctx *ctx, int strategy) {
    CTX_GUARD(ctx);
    if (strategy != MST_STRATEGY_FACE && strategy != MST_STRATEGY_CELL && strategy != MST_STRATEGY_PATCH &&
        strategy != MST_STRATEGY_FUSED && strategy != MST_STRATEGY_AUTO)
        return mst::fail(MST_E_ARG, "bad strategy");
    if ((strategy == MST_STRATEGY_PATCH || strategy == MST_STRATEGY_FUSED) && !ctx->patch_ok)
        return mst::fail(MST_E_UNSUPPORTED, "patch strategy: needs at most 4 faces per cell and 64 KiB of fluxes per patch");
    if (strategy == MST_STRATEGY_FUSED && !ctx->fused_ok)
        return mst::fail(MST_E_UNSUPPORTED, "fused strategy: a patch's face states exceed 64 KiB of LDS");
    ctx->strategy = strategy;
    ctx->resolved = strategy == MST_STRATEGY_AUTO ? -1 : strategy;
    return MST_OK;
}

int mst_get_strategy(const mst_ctx *ctx, int *strategy) {
    CTX_GUARD(ctx);
    if (!strategy) return mst::fail(MST_E_ARG, "null argument");
    *strategy = ctx->resolved >= 0 ? ctx->resolved : ctx->strategy;
    return MST_OK;
}

int mst_update_new_to_old(mst_ctx *ctx) {
    CTX_GUARD(ctx);
    std::swap(ctx->iold, ctx->inew);
    return MST_OK;
}

// Blocks up to which a step's stages reduce the block minima of its time step (stage_dt) instead of a launch between
// the steps (patches of SUB_PATCH cells count).  Microseconds per SSP-RK2 step, launch / in the stages: 24.7 / 23.6 at 32 blocks, 18.4 / 17.0 at 512 (first
// order), 26.5 / 27.2 at 1013.
constexpr int64_t STEP_DT_MAX = 512;

int mst_step(mst_ctx *ctx, int nsteps) {
    CTX_GUARD(ctx);
    if (nsteps < 0) return mst::fail(MST_E_ARG, "nsteps must be >= 0");
    static const double A2[2] = {0, 0.5}, B2[2] = {1, 0.5};
    static const double A3[3] = {0, 0.75, 1.0 / 3.0}, B3[3] = {1, 0.25, 2.0 / 3.0};
    const int ns = ctx->cfg.rk;
    const double *A = ns == 3 ? A3 : A2, *B = ns == 3 ? B3 : B2;
    const bool cfl = ctx->cfg.cfl > 0;
    for (int it = 0; it < nsteps; it++) {
        int rc;
        double *Qn = ctx->Q[ctx->iold];
        if (cfl && !ctx->dt_valid) {
            rc = run_cfl(ctx, Qn, ctx->cfg.cfl);
            if (rc) return rc;
        }
        // stage buffers: the two spare buffers alternate, the last stage lands in "new"; the first
        // stage of the call's last step reduces |R/V| (the norms are a monitor: one reduction per
        // call), the last stage of every step the CFL time step of the new state (next step's dt)
        int spare[2], w = 0;
        for (int i = 0; i < 4; i++)
            if (i != ctx->iold && i != ctx->inew) spare[w++] = i;
        const bool l2 = it == nsteps - 1;
        // mixed form: a stage that has a successor stores the successor's combination A Q^n + B Q_s in
        // place of its FP64 state (the FP32 kernels read only the shadow), so no later stage reads Q^n
        // again (SSP-RK2: none; RK3: the middle stage).  The viscous kernels read the FP64 stage state.
        const bool pre = ctx->mixed && !ctx->viscous;
        int src = ctx->iold;
        ctx->dt_to = ctx->dt_from == 0 ? 1 : 0;  // (the step's last stage still reads the other one)
        for (int s = 0; s < ns; s++) {
            const int dst = (s == ns - 1) ? ctx->inew : spare[s & 1];
            const int mode = UPD_STAGE | ((l2 && s == 0) ? UPD_L2 : 0) | ((cfl && s == ns - 1) ? UPD_DT : 0) |
                             (s == ns - 1 ? UPD_CHECK : 0);
            Stage sg;
            sg.ca = A[s];
            sg.cb = B[s];
            sg.stage0 = s == 0;
            sg.pre = pre;
            sg.wa = pre && s < ns - 1 ? A[s + 1] : 0;
            sg.wb = pre && s < ns - 1 ? B[s + 1] : 0;
            rc = run_stage(ctx, mode, src, ctx->iold, sg, dst);
            if (rc) break;
            src = dst;
        }
        // the next step's time step: on meshes of few blocks its stages reduce the minima themselves
        ctx->dt_from = -1;
        if (!rc && cfl && !l2 && ctx->dt_cnt[ctx->dt_to] <= STEP_DT_MAX)
            ctx->dt_from = ctx->dt_to;
        else if (!rc && (l2 || cfl))
            rc = run_finish(ctx, l2 ? ctx->nv : 0, cfl ? 1 : 0);
        ctx->dt_valid = cfl && !rc;
        if (rc) return rc;
        std::swap(ctx->iold, ctx->inew);
    }
    return check_bad(ctx);
}

int mst_run_to_steady(mst_ctx *ctx, double tol, int max_steps, int check_every, double *ref, int *steps_done,
                      double *drop) {
    CTX_GUARD(ctx);
    if (!ref || !(tol > 0) || max_steps < 1 || check_every < 1) return mst::fail(MST_E_ARG, "bad arguments");
    const bool lu = ctx->steady == MST_STEADY_LUSGS;
    if (!lu && !(ctx->cfg.cfl > 0))
        return mst::fail(MST_E_ARG, "explicit steady runs advance with the CFL time step (cfl > 0)");
    const int nv = ctx->nv;
    double r[5];
    int steps = 0;
    if (!(ref[0] > 0)) {  // reference: the residual of the first step
        int rc = lu ? mst_lusgs_step(ctx, 1) : mst_step(ctx, 1);
        if (rc) return rc;
        rc = mst_residual_norms(ctx, ref);
        if (rc) return rc;
        steps = 1;
    }
    double ratio = INFINITY;
    while (steps < max_steps) {
        const int k = std::min(check_every, max_steps - steps);
        int rc = lu ? mst_lusgs_step(ctx, k) : mst_step(ctx, k);
        if (rc) return rc;
        steps += k;
        rc = mst_residual_norms(ctx, r);
        if (rc) return rc;
        ratio = 0;
        for (int i = 0; i < nv; i++) ratio = std::max(ratio, ref[i] > 0 ? r[i] / ref[i] : 0.0);
        if (ratio <= tol) break;
    }
    if (steps_done) *steps_done = steps;
    if (drop) *drop = ratio;
    return MST_OK;
}

int mst_set_steady_driver(mst_ctx *ctx, int driver, double cfl, double omega) {
    CTX_GUARD(ctx);
    if (driver != MST_STEADY_EXPLICIT && driver != MST_STEADY_LUSGS)
        return mst::fail(MST_E_ARG, "driver must be MST_STEADY_EXPLICIT or MST_STEADY_LUSGS");
    if (driver == MST_STEADY_LUSGS && (!(cfl > 0) || !(omega > 0) || !std::isfinite(cfl)))
        return mst::fail(MST_E_ARG, "LU-SGS needs a finite cfl > 0 and omega > 0");
    ctx->steady = driver;
    if (driver == MST_STEADY_LUSGS) {
        ctx->lu_cfl = cfl;
        ctx->lu_omega = omega;
    }
    return MST_OK;
}

int mst_lusgs_step(mst_ctx *ctx, int n_iter) {
    CTX_GUARD(ctx);
    if (n_iter < 0) return mst::fail(MST_E_ARG, "n_iter must be >= 0");
    int rc = build_colours(ctx);
    if (rc) return rc;
    ctx->lu_inline = ctx->cfg.order == 1 && !ctx->mixed && !ctx->viscous && ctx->slots <= 4;
    const bool fuse = ctx->lu_inline && ctx->lu_start.size() >= 3;  // two colours or more
    for (int it = 0; it < n_iter;) {
        if (fuse && it < n_iter - 1) {  // the iterations before the call's last, colour 0's sweeps fused
            const int m = n_iter - 1 - it;
            rc = lu_inline_iterations(ctx, m);
            if (rc) return rc;
            it += m;
            continue;
        }
        rc = lu_iteration(ctx, it == n_iter - 1);  // norms of the call's last iteration (a monitor)
        if (rc) return rc;
        ctx->shadow_ok[ctx->inew] = false;
        std::swap(ctx->iold, ctx->inew);
        it++;
    }
    if (n_iter > 0) ctx->dt_valid = false;
    return check_bad(ctx);
}

int mst_lusgs_colours(mst_ctx *ctx, int32_t *colour, int64_t n_cells, int *n_colours) {
    CTX_GUARD(ctx);
    if (!colour || !n_colours || n_cells != ctx->nc) return mst::fail(MST_E_ARG, "size does not match the mesh");
    int rc = build_colours(ctx);
    if (rc) return rc;
    const auto &new_of_old = ctx->prep.P.cell_new_of_old;
    for (int64_t c = 0; c < ctx->nc; c++) colour[c] = ctx->lu_colour[new_of_old[c]];
    *n_colours = (int)ctx->lu_start.size() - 1;
    return MST_OK;
}

int mst_compute_dt(mst_ctx *ctx, double cfl, double *dt) {
    CTX_GUARD(ctx);
    if (!(cfl > 0) || !dt) return mst::fail(MST_E_ARG, "cfl must be positive");
    int rc = run_cfl(ctx, ctx->Q[ctx->iold], cfl);
    if (rc) return rc;
    rc = report(ctx, false);
    if (rc) return rc;
    *dt = ctx->board->scal[0];
    ctx->dt_valid = cfl == ctx->cfg.cfl;
    if (!(*dt > 0)) return mst::fail(MST_E_STATE, "non-physical state: no positive CFL time step");
    return MST_OK;
}

int mst_residual_norms(mst_ctx *ctx, double *out) {
    CTX_GUARD(ctx);
    if (!out) return mst::fail(MST_E_ARG, "null argument");
    int rc = report(ctx, false);
    if (rc) return rc;
    for (int k = 0; k < ctx->nv; k++) out[k] = ctx->board->scal[1 + k];
    return MST_OK;
}

int mst_monitor_maxrel(mst_ctx *ctx, double *out) {
    CTX_GUARD(ctx);
    if (!out) return mst::fail(MST_E_ARG, "null argument");
    return ctx->nv == 4 ? run_monitor<4>(ctx, out) : run_monitor<5>(ctx, out);
}

int mst_monitor_maxrel_noalloc(const double *qnew, const double *qold, int64_t n_cells, int nv, double *out,
                               void *stream) {
    if (!qnew || !qold || !out) return mst::fail(MST_E_ARG, "null device pointer");
    if (nv != 4 && nv != 5) return mst::fail(MST_E_ARG, "nv must be 4 (2D) or 5 (3D)");
    if (n_cells < 1 || n_cells > MST_NOALLOC_MAX_CELLS)
        return mst::fail(MST_E_ARG, "n_cells must be in [1, MST_NOALLOC_MAX_CELLS]");
    if (nv == 4 && (((uintptr_t)qnew | (uintptr_t)qold) & 15u))
        return mst::fail(MST_E_ARG, "2D states must be 16-byte aligned (records are loaded as 16-byte pairs)");
    double *part = nullptr;
    int rc = noalloc_scratch_ptr(&part);
    if (rc) return rc;
    hipStream_t st = static_cast<hipStream_t>(stream);
    const int64_t grid = std::min<int64_t>((n_cells + BLOCK - 1) / BLOCK, NOALLOC_GRID);
    if (nv == 4)
        hipLaunchKernelGGL(k_maxrel<4>, dim3((uint32_t)grid), dim3(BLOCK), 0, st, n_cells, qnew, qold, part);
    else
        hipLaunchKernelGGL(k_maxrel<5>, dim3((uint32_t)grid), dim3(BLOCK), 0, st, n_cells, qnew, qold, part);
    HIPCHK(hipGetLastError());
    FinArgs f;
    memset(&f, 0, sizeof(f));
    f.nblk = grid;  // <= 2 * FIN_CHUNK: one finish block
    f.chunk = grid;
    f.count = 1.0;
    f.n = nv;
    for (int k = 0; k < nv; k++) {
        f.src[k] = part + k * grid;
        f.kind[k] = 2;
        f.dst[k] = out + k;
    }
    hipLaunchKernelGGL(k_finish, dim3(1), dim3(FIN), 0, st, f);
    HIPCHK(hipGetLastError());
    return MST_OK;
}

int mst_ctx_warm_start(mst_ctx *ctx, mst_mlp *mlp, const double *cond, int n_cond) {
    CTX_GUARD(ctx);
    if (!mlp || n_cond < 1 || n_cond > 8 || !cond) return mst::fail(MST_E_ARG, "bad arguments");
    int n_in = 0, n_out = 0;
    mst::mlp_dims(mlp, &n_in, &n_out);
    if (n_in != ctx->dim + n_cond || n_out != ctx->nv)
        return mst::fail(MST_E_ARG, "network sizes do not match (dim + conditions) -> nv");
    if (!(cond[0] > 0)) return mst::fail(MST_E_ARG, "the first condition (freestream Mach number) must be positive");
    if (ctx->g_of != ctx->inew) {  // (every other buffer is written here)
        int rc = ensure_fluxes(ctx);
        if (rc) return rc;
    }
    WarmArgs w;
    w.nc = ctx->nc;
    w.cxc = ctx->cxc;
    w.n_cond = n_cond;
    for (int k = 0; k < 8; k++) w.cond[k] = k < n_cond ? (float)cond[k] : 0.f;
    w.mach = cond[0];
    w.gamma = ctx->cfg.gamma;
    w.Q = ctx->Q[ctx->iold];
    w.bad = ctx->bad;
    // the two spare stage buffers hold the features and the outputs (nothing between calls)
    int spare[2], ns = 0;
    for (int i = 0; i < 4; i++)
        if (i != ctx->iold && i != ctx->inew) spare[ns++] = i;
    const bool fits = sizeof(float) * n_in <= sizeof(double) * ctx->nv;
    float *feat = reinterpret_cast<float *>(ctx->Q[spare[0]]);
    if (!fits) HIPCHK(hipMalloc((void **)&feat, sizeof(float) * ctx->nc * n_in));
    w.feat = feat;
    w.Y = reinterpret_cast<float *>(ctx->Q[spare[1]]);
    int rc = ctx->dim == 2 ? launch(ctx, -1, k_warm_features<2>, ctx->nc, w) : launch(ctx, -1, k_warm_features<3>, ctx->nc, w);
    if (!rc) rc = mst::mlp_forward_device(mlp, feat, ctx->nc, reinterpret_cast<float *>(ctx->Q[spare[1]]), ctx->stream);
    if (!rc)
        rc = ctx->dim == 2 ? launch(ctx, -1, k_warm_decode<2>, ctx->nc, w) : launch(ctx, -1, k_warm_decode<3>, ctx->nc, w);
    if (!fits) {
        const hipError_t e = hipStreamSynchronize(ctx->stream);
        (void)hipFree(feat);
        if (!rc && e != hipSuccess) return mst::fail(MST_E_HIP, hipGetErrorString(e));
    }
    if (rc) return rc;
    for (int i = 0; i < 4; i++) ctx->shadow_ok[i] = false;
    ctx->dt_valid = false;
    return check_bad(ctx);
}

int mst_get_residual(mst_ctx *ctx, double *R, int64_t n_cells) {
    CTX_GUARD(ctx);
    if (!R || n_cells != ctx->nc) return mst::fail(MST_E_ARG, "size does not match the mesh");
    if (!ctx->R) {
        int rc = dalloc(&ctx->R, ctx->nc * ctx->nv);
        if (rc) return rc;
    }
    int rc = run_face_flux(ctx, ctx->iold);
    if (rc) return rc;
    rc = run_update(ctx, UPD_RESIDUAL, -1, -1, Stage{0, 0, 0}, -1);
    if (rc) return rc;
    return fetch_cells(ctx, ctx->R, ctx->nv, R);
}

int mst_get_face_flux(mst_ctx *ctx, double *G, int64_t n_faces) {
    CTX_GUARD(ctx);
    if (!G || n_faces != ctx->nf) return mst::fail(MST_E_ARG, "size does not match the mesh");
    int rc = ensure_fluxes(ctx);
    if (rc) return rc;
    const int nv = ctx->nv;
    std::vector<double> buf(ctx->nf * nv);
    HIPCHK(hipStreamSynchronize(ctx->stream));
    HIPCHK(hipMemcpy(buf.data(), ctx->G, sizeof(double) * buf.size(), hipMemcpyDeviceToHost));
    const auto &new_of_old = ctx->prep.P.face_new_of_old;
    const auto &merged = ctx->prep.P.fmerged_into;
    for (int64_t f = 0; f < ctx->nf; f++) {
        const int64_t i = new_of_old[f];
        for (int k = 0; k < nv; k++)  // the merged half of a periodic pair carries minus its pair's flux
            G[f * nv + k] = merged[i] >= 0 ? -buf[(int64_t)merged[i] * nv + k] : buf[i * nv + k];
    }
    return MST_OK;
}

int mst_get_gradient(mst_ctx *ctx, double *grad, double *phi, int64_t n_cells) {
    CTX_GUARD(ctx);
    if (n_cells != ctx->nc) return mst::fail(MST_E_ARG, "size does not match the mesh");
    if (!ctx->graw) {
        int rc = dalloc(&ctx->graw, ctx->nc * ctx->nv * ctx->dim);
        if (rc) return rc;
        rc = dalloc(&ctx->phi, ctx->nc * ctx->nv);
        if (rc) return rc;
    }
    int rc = run_grad(ctx, ctx->iold, true);
    if (rc) return rc;
    if (grad) {
        rc = fetch_cells(ctx, ctx->graw, ctx->nv * ctx->dim, grad);
        if (rc) return rc;
    }
    if (phi) return fetch_cells(ctx, ctx->phi, ctx->nv, phi);
    return MST_OK;
}

int mst_riemann_flux(const mst_config *cfg, int dim, int64_t n, const double *QL, const double *QR,
                     const int32_t *dir, double *F) {
    int rc = check_config(cfg);
    if (rc) return rc;
    if ((dim != 2 && dim != 3) || n < 0 || (n > 0 && (!QL || !QR || !dir || !F)))
        return mst::fail(MST_E_ARG, "bad arguments");
    for (int64_t i = 0; i < n; i++)
        if (dir[i] < 0 || dir[i] >= dim) return mst::fail(MST_E_ARG, "direction out of range");
    if (n == 0) return MST_OK;
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev <= 0) return mst::fail(MST_E_HIP, "no HIP device available");
    const int nv = dim + 2;
    double *dL = nullptr, *dR = nullptr, *dF = nullptr;
    int32_t *dd = nullptr;
    HIPCHK(hipMalloc((void **)&dL, sizeof(double) * n * nv));
    HIPCHK(hipMalloc((void **)&dR, sizeof(double) * n * nv));
    HIPCHK(hipMalloc((void **)&dF, sizeof(double) * n * nv));
    HIPCHK(hipMalloc((void **)&dd, sizeof(int32_t) * n));
    HIPCHK(hipMemcpy(dL, QL, sizeof(double) * n * nv, hipMemcpyHostToDevice));
    HIPCHK(hipMemcpy(dR, QR, sizeof(double) * n * nv, hipMemcpyHostToDevice));
    HIPCHK(hipMemcpy(dd, dir, sizeof(int32_t) * n, hipMemcpyHostToDevice));
    Params<double> P = make_params<double>(*cfg);
    const uint32_t grid = (uint32_t)((n + BLOCK - 1) / BLOCK);
    if (dim == 2) {
        if (cfg->scheme == MST_SCHEME_ROE)
            hipLaunchKernelGGL((k_riemann<2, MST_SCHEME_ROE>), dim3(grid), dim3(BLOCK), 0, 0, n, dL, dR, dd, dF, P);
        else
            hipLaunchKernelGGL((k_riemann<2, MST_SCHEME_AUSM>), dim3(grid), dim3(BLOCK), 0, 0, n, dL, dR, dd, dF, P);
    } else {
        if (cfg->scheme == MST_SCHEME_ROE)
            hipLaunchKernelGGL((k_riemann<3, MST_SCHEME_ROE>), dim3(grid), dim3(BLOCK), 0, 0, n, dL, dR, dd, dF, P);
        else
            hipLaunchKernelGGL((k_riemann<3, MST_SCHEME_AUSM>), dim3(grid), dim3(BLOCK), 0, 0, n, dL, dR, dd, dF, P);
    }
    hipError_t e = hipGetLastError();
    if (e == hipSuccess) e = hipDeviceSynchronize();
    if (e == hipSuccess) e = hipMemcpy(F, dF, sizeof(double) * n * nv, hipMemcpyDeviceToHost);
    (void)hipFree(dL);
    (void)hipFree(dR);
    (void)hipFree(dF);
    (void)hipFree(dd);
    if (e != hipSuccess) return mst::fail(MST_E_HIP, std::string("riemann kernel: ") + hipGetErrorString(e));
    return MST_OK;
}

int mst_copy_probe(int64_t nbytes, double *ms) {
    if (nbytes < 16 || nbytes % 16) return mst::fail(MST_E_ARG, "nbytes must be a positive multiple of 16");
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev <= 0) return mst::fail(MST_E_HIP, "no HIP device available");
    double2 *a = nullptr, *b = nullptr;
    HIPCHK(hipMalloc((void **)&a, nbytes));
    HIPCHK(hipMalloc((void **)&b, nbytes));
    HIPCHK(hipMemset(a, 0, nbytes));
    const int64_t n2 = nbytes / 16;
    hipEvent_t e0, e1;
    HIPCHK(hipEventCreate(&e0));
    HIPCHK(hipEventCreate(&e1));
    HIPCHK(hipDeviceSynchronize());
    HIPCHK(hipEventRecord(e0, 0));
    hipLaunchKernelGGL(k_copy, dim3((uint32_t)((n2 + BLOCK - 1) / BLOCK)), dim3(BLOCK), 0, 0, n2,
                       (const double2 *)a, b);
    HIPCHK(hipGetLastError());
    HIPCHK(hipEventRecord(e1, 0));
    HIPCHK(hipEventSynchronize(e1));
    float t = 0;
    HIPCHK(hipEventElapsedTime(&t, e0, e1));
    if (ms) *ms = t;
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    (void)hipFree(a);
    (void)hipFree(b);
    return MST_OK;
}

int mst_timing_enable(mst_ctx *ctx, int on) {
    CTX_GUARD(ctx);
    if (on < 0) return mst::fail(MST_E_ARG, "timing: on must be >= 0");
    ctx->timing = on != 0;
    ctx->timing_stride = on > 1 ? on : 1;
    for (int k = 0; k < MST_K_COUNT; k++) ctx->tick[k] = 0;
    return MST_OK;
}

int mst_timing_get(mst_ctx *ctx, int kernel, int64_t *count, double *total_ms) {
    CTX_GUARD(ctx);
    if (kernel < 0 || kernel >= MST_K_COUNT || !count || !total_ms) return mst::fail(MST_E_ARG, "bad kernel id");
    HIPCHK(hipStreamSynchronize(ctx->stream));
    double tot = 0;
    for (auto &pr : ctx->ev[kernel]) {
        float ms = 0;
        HIPCHK(hipEventElapsedTime(&ms, pr.first, pr.second));
        tot += ms;
    }
    *count = (int64_t)ctx->ev[kernel].size();
    *total_ms = tot;
    return MST_OK;
}

int mst_timing_reset(mst_ctx *ctx) {
    CTX_GUARD(ctx);
    HIPCHK(hipStreamSynchronize(ctx->stream));
    for (int k = 0; k < MST_K_COUNT; k++) {
        for (auto &pr : ctx->ev[k]) {
            ctx->pool.push_back(pr.first);
            ctx->pool.push_back(pr.second);
        }
        ctx->ev[k].clear();
    }
    return MST_OK;
}

int mst_sync(mst_ctx *ctx) {
    CTX_GUARD(ctx);
    HIPCHK(hipStreamSynchronize(ctx->stream));
    return MST_OK;
}

// Compulsory HBM traffic of one launch: every array the kernel must touch, once.  r is the size of
// the arithmetic real of the gradient/flux kernels (8 FP64, 4 mixed: FP32 state shadow, normals,
// offsets, limited gradients); face fluxes, the stage states, volumes and centres stay FP64.
int mst_algorithmic_bytes(const mst_ctx *ctx, int kernel, double *bytes) {
    CTX_GUARD(ctx);
    if (!bytes) return mst::fail(MST_E_ARG, "null argument");
    const double nc = (double)ctx->nc, nf = (double)ctx->nf, D = ctx->dim, NV = ctx->nv;
    const bool mixed = ctx->mixed, second = ctx->cfg.order >= 2;
    const double r = mixed ? 4 : 8;
    const double ell = 4.0 * ctx->maxf * nc;
    const double w_inc = mixed && ctx->dim == 3 ? 0 : r;  // incidence weight bytes of the gradient
    const double stages = ctx->cfg.rk;
    // faces: c0, c1, info, FP64 normal; cells: the arithmetic state; order 2: face-cell offsets
    // (FP64: face centres, partner centres and cell centres) and limited gradients
    // order 2: the side records (each read once), the record indices, the raw c0 state of boundary faces
    const double ninc = (double)ctx->n_inc, n2 = (double)ctx->prep.P.n_interior, nbnd = nf - n2;
    // a viscous stage's route (run_stage)
    const bool visc_patch = ctx->viscous && ctx->visc_patch &&
                            (ctx->resolved >= 0 ? ctx->resolved : ctx->strategy) != MST_STRATEGY_FACE;
    double flux_in = nf * (12 + 8 * D) + nc * r * NV;
    if (second) flux_in = nf * (12 + 8 * D + 8) + ninc * r * NV + nbnd * r * NV;
    // update: cell faces, stage state, volume, new state (+ FP32 shadow), Q^n on stages after the
    // first (mixed form: pre-combined stage states, Q^n only on RK3's middle stage), the CFL half-sums
    // on the last stage when the time step is reduced there
    const double qn_stages = mixed && !ctx->viscous ? std::max(stages - 2, 0.0) : stages - 1;
    double upd = ell + nc * (8 * NV + 8 + 8 * NV) + nc * 8 * NV * qn_stages / stages;
    if (mixed) upd += nc * 4 * NV;
    if (ctx->cfg.cfl > 0) upd += nc * 8 * D / stages;
    switch (kernel) {
        case MST_K_FLUX:
            *bytes = flux_in + nf * 8 * NV;
            break;
        case MST_K_GRAD:  // incidences: code, weight (not FP32 3D: folded into the normal), normal, offset,
                          // record out; cells: state, volume
            *bytes = 4.0 * ctx->slots * nc + ninc * (w_inc + 2 * r * D + r * NV) + nc * (r * NV + r);
            // viscous gradients out; the kinds of boundary faces
            if (visc_patch && second && !mixed) *bytes += nc * 8 * (D + 1) * D + nbnd * 8;
            break;
        case MST_K_UPDATE:
            *bytes = upd + nf * 8 * NV;
            break;
        case MST_K_CELL:  // flux inputs + update, no face-flux array; FP64 reads the stage state once
            *bytes = flux_in + upd - (mixed ? 0 : (second ? nbnd : nc) * 8 * NV);
            break;
        case MST_K_PATCH:  // as the cell kernel, with the patch face lists and local slots for the table
            // (a face's kind comes with its packed list entry when there is one)
            *bytes = flux_in + upd - (mixed ? 0 : (second ? nbnd : nc) * 8 * NV) - ell +
                     4.0 * (double)ctx->n_psolve + 2.0 * ctx->slots * nc - (ctx->pfi ? 4.0 * nf : 0.0);
            if (ctx->viscous) *bytes += nc * 8 * (D + 1) * D + n2 * 8;  // viscous gradients, eta of faces of two cells
            break;
        case MST_K_FUSED: {  // gradient inputs + per-face inputs + update, each once; no records
            // per incidence: code, weight, offset, and in 3D the normal (2D takes it from its face's)
            const double inc_geo = ctx->dim == 2 ? r + r * D : w_inc + 2 * r * D;
            const double grad_in = 4.0 * ctx->slots * nc + ninc * inc_geo + nc * (r * NV + r);
            const double flux_f = nf * ((ctx->pfi ? 0 : 4) + 8 * D) + 4.0 * (double)ctx->n_psolve + nbnd * 4;
            *bytes = grad_in + flux_f + upd - ell + 2.0 * ctx->slots * nc - (mixed ? 0 : nc * 8 * NV);
            break;
        }
        case MST_K_DT:
            *bytes = nc * (8 * NV + 8 + 8 * D);
            break;
        case MST_K_VISC: {
            const double nw = D + 1;
            const double grad = 4.0 * ctx->slots * nc + ninc * (8 + 8 * D) + nbnd * 8 + nc * (8 * NV + 8 + 8 * nw * D);
            const double face = nf * (8 + 4 + 8 * D + 2 * 8 * NV) + n2 * 8 + nc * (8 * NV + 8 * nw * D);
            // face route: the gradient kernel and the face kernel, averaged over the two launches
            *bytes = visc_patch ? grad : 0.5 * (grad + face);
            break;
        }
        case MST_K_LUSGS: {  // one iteration's sweeps, each array once per sweep, over their launches
            if (ctx->lu_start.size() < 2) return mst::fail(MST_E_ARG, "no LU-SGS iteration has run");
            std::vector<LuCount> count;
            try {
                count = lu_counts(ctx);
            } catch (const std::bad_alloc &) {
                return mst::fail(MST_E_ARG, "out of host memory");
            }
            // 2 K - 1 launches for K colours; 2 K - 2 where colour 0's sweeps of consecutive
            // iterations run fused (the iterations of a call before its last)
            const int K = (int)count.size();
            const bool bf = ctx->lu_inline && K >= 2;
            const double S = ctx->slots, v = 8 * NV;
            double total = 0;
            for (int k = 0; k < K; k++) {
                const LuCount &l = count[k];
                const double n = (double)l.n, inc = (double)l.inc, lo = (double)l.lo, hi = (double)l.hi;
                const double hinc = (double)l.inc_hi;
                const double rec = n * 4 + 4 * std::min(S * n, inc + n);  // positions, neighbour codes
                const bool last = k == K - 1;
                // forward: records, residual (or the face words to compute it from), normals, states of the cells and
                // their neighbours, lower neighbours' updates; update out, and radii and D, or the last colour's state
                if (k > 0 || !bf)
                    total += rec + n * (ctx->lu_inline ? 4 : v) + inc * 8 * D + v * (n + 2 * lo + hi) + v * n +
                             (last ? v * n : inc * 8 + n * 8);
                // backward (not the last colour): records, D, states and updates of the cells and their higher
                // neighbours with the normals and radii toward them; update and state out
                if (!last && (k > 0 || !bf)) total += rec + n * 8 + hinc * (8 * D + 8) + 2 * v * (n + hi) + 2 * v * n;
                // colour 0's backward and next forward sweep in one: the forward sweep's face words, the remaining
                // normals, radii, D and update out besides; no second read of a neighbour, one update stored
                if (k == 0 && bf)
                    total += rec + n * 8 + n * 4 + inc * 8 * D + hinc * 8 + 2 * v * (n + hi) + 2 * v * n + inc * 8 + n * 8;
            }
            *bytes = total / (bf ? 2 * K - 2 : 2 * K - 1);
            break;
        }
        default:
            return mst::fail(MST_E_ARG, "bad kernel id");
    }
    return MST_OK;
}

}  // extern "C"
