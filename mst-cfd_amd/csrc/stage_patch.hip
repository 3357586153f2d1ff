// stage_patch.hip -- launches of the patch strategy.
#include "context.hpp"

namespace mstk {

// patch strategy: gradient + limiter (order 2), then the patch kernel (faces into LDS, sum, update)
template <int DIM, typename T>
int run_patch_t(mst_ctx *x, int mode, int is, int in, const Stage &sg, int iout) {
    if (!x->patch_ok) return mst::fail(MST_E_UNSUPPORTED, "no patch tables for this mesh");
    const FluxArgs<T> fa = flux_args<T>(x, is);
    const UpdArgs a = upd_args(x, mode, is, in, sg, iout);
    partials(x, mode, x->n_patch);
    PatchArgs pa;
    pa.start = x->pstart;
    pa.face = x->pface;
    pa.loc = x->ploc;
    pa.fi = x->pfi;
    const size_t shm = (size_t)x->max_pf * x->nv * sizeof(double);
    const bool second = x->cfg.order >= 2;
    const bool roe = x->cfg.scheme == MST_SCHEME_ROE, sub = x->patch_cells == SUB_PATCH;
    constexpr bool SUB = has_sub_patches<DIM, T>();
    if (x->viscous) {
        const ViscFace<DIM> vf{visc_args(x, is)};
#define MST_PATCH_V_N(MF, SECOND, PC, NT)                                                                                    \
    return roe ? launch_patch(x, MST_K_PATCH, k_patch<DIM, MST_SCHEME_ROE, SECOND, T, MF, true, PC, NT, ViscFace<DIM>>, NT, shm, \
                              fa, a, pa, vf)                                                                             \
               : launch_patch(x, MST_K_PATCH, k_patch<DIM, MST_SCHEME_AUSM, SECOND, T, MF, true, PC, NT, ViscFace<DIM>>, NT, \
                              shm, fa, a, pa, vf);
#define MST_PATCH_V(MF, SECOND)                      \
    if constexpr (SUB) if (sub) { MST_PATCH_V_N(MF, SECOND, SUB_PATCH, 2 * SUB_PATCH) } \
    if (x->wide_patch) { MST_PATCH_V_N(MF, SECOND, BLOCK, 2 * BLOCK) } \
    MST_PATCH_V_N(MF, SECOND, BLOCK, BLOCK)
        if (x->slots == 3) {
            if (second) { MST_PATCH_V(3, true) }
            MST_PATCH_V(3, false)
        }
        if (second) { MST_PATCH_V(4, true) }
        MST_PATCH_V(4, false)
#undef MST_PATCH_V_N
#undef MST_PATCH_V
    }
    if constexpr (std::is_same<T, float>::value) {
        if (second) {  // the mixed form stages its face states in LDS from the records (k_patch_rec)
            HaloArgs ha{};
            ha.start = x->hstart;
            ha.cell = x->hcell;
            ha.loc = x->hloc;
#define MST_PATCH_REC_N(MF, PC, NT)                                                                                  \
    return roe ? launch_patch(x, MST_K_PATCH, k_patch_rec<DIM, MST_SCHEME_ROE, MF, PC, NT>, NT, shm, fa, a, pa, ha)      \
               : launch_patch(x, MST_K_PATCH, k_patch_rec<DIM, MST_SCHEME_AUSM, MF, PC, NT>, NT, shm, fa, a, pa, ha);
#define MST_PATCH_REC(MF)                      \
    if constexpr (SUB) if (sub) { MST_PATCH_REC_N(MF, SUB_PATCH, 2 * SUB_PATCH) } \
    if (x->wide_patch) { MST_PATCH_REC_N(MF, BLOCK, 2 * BLOCK) } \
    MST_PATCH_REC_N(MF, BLOCK, BLOCK)
            if (x->slots == 3) { MST_PATCH_REC(3) }
            MST_PATCH_REC(4)
#undef MST_PATCH_REC
#undef MST_PATCH_REC_N
        }
    }
#define MST_PATCH_N(MF, SECOND, PC, NT)                                                                               \
    return roe ? launch_patch(x, MST_K_PATCH, k_patch<DIM, MST_SCHEME_ROE, SECOND, T, MF, true, PC, NT>, NT, shm, fa, a,  \
                              pa, NoExtra())                                                                      \
               : launch_patch(x, MST_K_PATCH, k_patch<DIM, MST_SCHEME_AUSM, SECOND, T, MF, true, PC, NT>, NT, shm, fa, a, \
                              pa, NoExtra());
#define MST_PATCH_W(MF, PC, NT)                      \
    if (second) { MST_PATCH_N(MF, true, PC, NT) }    \
    MST_PATCH_N(MF, false, PC, NT)
#define MST_PATCH(MF)                                         \
    if constexpr (SUB) if (sub) { MST_PATCH_W(MF, SUB_PATCH, 2 * SUB_PATCH) }    \
    if (x->wide_patch) { MST_PATCH_W(MF, BLOCK, 2 * BLOCK) }  \
    MST_PATCH_W(MF, BLOCK, BLOCK)
    if (x->slots == 3) { MST_PATCH(3) }
    MST_PATCH(4)
#undef MST_PATCH
#undef MST_PATCH_W
#undef MST_PATCH_N
}

template <int DIM>
int run_patch_residual_t(mst_ctx *x, int mode, int is) {
    const FluxArgs<double> fa = flux_args<double>(x, is);
    const UpdArgs a = upd_args(x, mode, is, -1, Stage{0, 0}, -1);
    partials(x, mode, x->n_patch);
    PatchArgs pa;
    pa.start = x->pstart;
    pa.face = x->pface;
    pa.loc = x->ploc;
    pa.fi = x->pfi;
    const size_t shm = (size_t)x->max_pf * x->nv * sizeof(double);
    const bool second = x->cfg.order >= 2;
    const bool roe = x->cfg.scheme == MST_SCHEME_ROE;
#define MST_PATCH_R_N(MF, SECOND, PC, NT)                                                                                  \
    return roe ? launch_patch(x, MST_K_PATCH, k_patch<DIM, MST_SCHEME_ROE, SECOND, double, MF, false, PC, NT>, NT, shm, fa, a, \
                              pa, NoExtra())                                                                           \
               : launch_patch(x, MST_K_PATCH, k_patch<DIM, MST_SCHEME_AUSM, SECOND, double, MF, false, PC, NT>, NT, shm, fa,   \
                              a, pa, NoExtra());
#define MST_PATCH_R_W(MF, PC, NT)                     \
    if (second) { MST_PATCH_R_N(MF, true, PC, NT) }   \
    MST_PATCH_R_N(MF, false, PC, NT)
#define MST_PATCH_R(MF)                                                                  \
    if (x->patch_cells == SUB_PATCH) { MST_PATCH_R_W(MF, SUB_PATCH, 2 * SUB_PATCH) }     \
    MST_PATCH_R_W(MF, BLOCK, BLOCK)
    if (x->slots == 3) { MST_PATCH_R(3) }
    MST_PATCH_R(4)
#undef MST_PATCH_R
#undef MST_PATCH_R_W
#undef MST_PATCH_R_N
}

template int run_patch_t<2, double>(mst_ctx *, int, int, int, const Stage &, int);
template int run_patch_t<3, double>(mst_ctx *, int, int, int, const Stage &, int);
template int run_patch_t<2, float>(mst_ctx *, int, int, int, const Stage &, int);
template int run_patch_t<3, float>(mst_ctx *, int, int, int, const Stage &, int);
template int run_patch_residual_t<2>(mst_ctx *, int, int);
template int run_patch_residual_t<3>(mst_ctx *, int, int);

}  // namespace mstk
