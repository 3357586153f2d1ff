// stage_fused.hpp -- launches of the fused strategy; stage_fused_{2d,3d}{64,32}.hip instantiate it.
#pragma once
#include "context.hpp"

namespace mstk {

// the fused kernel's packed halo geometry, gathered on the context's stream when the weights changed
static int ensure_halo_geo(mst_ctx *x) {
    if (!x->hg_dirty || !x->patch_ok || x->n_halo == 0) return MST_OK;
    const IncView<double> f64{x->inc_code, x->inc_w, x->inc_n, x->inc_dx, x->cvol, x->nc};
    const IncView<float> f32{x->mixed ? x->inc_code : nullptr, x->inc_w32, x->inc_n32, x->inc_dx32, x->ivol32, x->nc};
    HIPCHK(x->dim == 2 ? x->hg.fill<2>(x->slots, x->nc, x->n_halo, x->hcell, f64, f32, x->stream)
                       : x->hg.fill<3>(x->slots, x->nc, x->n_halo, x->hcell, f64, f32, x->stream));
    x->hg_dirty = false;
    return MST_OK;
}

// fused strategy (order 2): gradients, face states, fluxes, sums and update of a patch in one kernel
template <int DIM, typename T>
int run_fused_t(mst_ctx *x, int mode, int is, int in, const Stage &sg, int iout) {
    if (x->cfg.order < 2) return run_patch_t<DIM, T>(x, mode, is, in, sg, iout);
    if (!x->fused_ok) return mst::fail(MST_E_UNSUPPORTED, "fused strategy: a patch's face states exceed 64 KiB of LDS");
    int rc = ensure_halo_geo(x);
    if (rc) return rc;
    const GradArgs<T> ga = grad_args<T>(x, is, false);
    const FluxArgs<T> fa = flux_args<T>(x, is);
    const UpdArgs a = upd_args(x, mode, is, in, sg, iout);
    partials(x, mode, x->n_patch);
    PatchArgs pa;
    pa.start = x->pstart;
    pa.face = x->pface;
    pa.loc = x->ploc;
    pa.fi = x->pfi;
    HaloArgs ha;
    ha.start = x->hstart;
    ha.cell = x->hcell;
    ha.loc = x->hloc;
    x->hg.args<T>(ha);
    // the face states and fluxes (and in 2D the faces' normals), and afterwards the block reductions
    // (NV doubles per wave)
    const size_t shm = std::max(fused_lds_bytes(DIM, x->nv, x->max_pf, std::is_same<T, float>::value,
                                                fused_lds_normals<DIM>()),
                                sizeof(double) * x->nv * (2 * BLOCK / 64));
    const bool roe = x->cfg.scheme == MST_SCHEME_ROE;
    const int lim = x->cfg.limiter;
    // (the sweeps stand at mst_ctx::wide_patch)
    const bool wide = x->nblk_c <= (DIM == 2 && (x->slots == 3 || std::is_same<T, float>::value) ? 512 : 256);
#define MST_FUSED_L(SC, LM, MF)                                                                                         \
    if constexpr (has_sub_patches<DIM, T>()) if (x->patch_cells == SUB_PATCH)                                           \
        return launch_patch(x, MST_K_FUSED, k_fused<DIM, SC, LM, T, MF, SUB_PATCH, 2 * SUB_PATCH>, 2 * SUB_PATCH, shm,  \
                            ga, fa, a, pa, ha);                                                                         \
    return wide ? launch_patch(x, MST_K_FUSED, k_fused<DIM, SC, LM, T, MF, BLOCK, 2 * BLOCK>, 2 * BLOCK, shm, ga, fa, a, \
                               pa, ha)                                                                                  \
                : launch_patch(x, MST_K_FUSED, k_fused<DIM, SC, LM, T, MF>, BLOCK, shm, ga, fa, a, pa, ha);
#define MST_FUSED_S(SC, MF)                                                                   \
    if (lim == MST_LIM_NONE) { MST_FUSED_L(SC, MST_LIM_NONE, MF) }                            \
    if (lim == MST_LIM_MINMOD) { MST_FUSED_L(SC, MST_LIM_MINMOD, MF) }                        \
    MST_FUSED_L(SC, MST_LIM_VANLEER, MF)
#define MST_FUSED(MF)                          \
    if (roe) { MST_FUSED_S(MST_SCHEME_ROE, MF) } \
    MST_FUSED_S(MST_SCHEME_AUSM, MF)
    if (x->slots == 3) { MST_FUSED(3) }
    MST_FUSED(4)
#undef MST_FUSED
#undef MST_FUSED_S
#undef MST_FUSED_L
}

}  // namespace mstk
