// context.hpp -- the device context behind include/mstcfd.h and what its launch files share: the launch itself
// (with per-dispatch timing) and the kernels' arguments.  solver.hip holds the C entry points and the
// drivers, stage_patch.hip and stage_fused*.hip the patch and fused strategies (files of their own because
// their many kernel variants compile side by side).
#pragma once
#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>

#include <algorithm>
#include <string>
#include <vector>

#include "kernels.hpp"
#include "mstcfd.h"
#include "prep.hpp"
#include "transfer.hpp"
#include "viscous.hpp"

using namespace mstk;

#define HIPCHK(expr)                                                                                     \
    do {                                                                                                 \
        hipError_t _e = (expr);                                                                          \
        if (_e != hipSuccess)                                                                            \
            return mst::fail(MST_E_HIP, std::string(#expr) + ": " + hipGetErrorString(_e));              \
    } while (0)

// blocks of BLOCK cells up to which patches are of SUB_PATCH cells, 2D and 3D (mst_ctx::patch_cells)
constexpr int64_t SUB_PATCH_MAX[2] = {128, 64};

// ====================================================================================== context
struct mst_ctx {
    mst_prep prep;
    mst_config cfg;
    Params<double> p64;
    Params<float> p32;
    bool mixed = false;
    int strategy = MST_STRATEGY_AUTO;
    int resolved = -1;  // strategy in use (AUTO: measured at the first stage after a configuration)
    hipStream_t stream = nullptr;
    int device = 0;
    int dim = 2, nv = 4, maxf = 3;
    int64_t nc = 0, nf = 0, nblk_c = 0, nblk_f = 0;
    // FP64 arrays (new order)
    int32_t *fc0 = nullptr, *fc1 = nullptr, *finfo = nullptr, *ell = nullptr;
    double *fn = nullptr, *fxf = nullptr, *pxf = nullptr, *feta = nullptr;
    double *cvol = nullptr, *cxc = nullptr, *cshalf = nullptr;
    double *Q[4] = {nullptr, nullptr, nullptr, nullptr};
    int iold = 0, inew = 1;
    double *G = nullptr, *rec = nullptr, *graw = nullptr, *phi = nullptr, *R = nullptr;
    int32_t *frec0 = nullptr, *frec1 = nullptr;  // incidence records of each face's c0 / c1 side
    // patch strategy: per patch of patch_cells cells its flux-carrying faces, per cell slot the local index
    int32_t *pstart = nullptr, *pface = nullptr;
    int16_t *ploc = nullptr;
    uint32_t *pfi = nullptr;  // pface with the faces' kinds and L/R masks packed in (null: 2^26 faces or more)
    int max_pf = 0;        // most faces of one patch (sizes the kernel's LDS)
    int64_t n_psolve = 0;  // Riemann problems per patch launch
    bool patch_ok = false;
    bool fused_ok = false;  // the fused kernel's LDS (states and staged normals) fits 64 KiB
    // fused strategy: each patch's halo cells (across its border faces) and their slots' local faces
    int32_t *hstart = nullptr, *hcell = nullptr;
    int16_t *hloc = nullptr;
    int64_t n_halo = 0;
    HaloGeo hg;  // the halo cells' incidence geometry in halo order, filled on the fused kernel's first use
    bool hg_dirty = true;  // hg does not hold the current incidence weights
    // mixed form: FP32 shadows of the states, FP32 geometry, offsets, face fluxes, limited gradients
    float *Q32[4] = {nullptr, nullptr, nullptr, nullptr};
    bool shadow_ok[4] = {false, false, false, false};
    float *rec32 = nullptr;  // FP32 reconstructed face states (order 2)
    // incidence layout of the gradient kernel (slot-major over the padded ELL slots)
    int slots = 3;
    int64_t n_inc = 0;  // non-empty incidences
    int32_t *inc_code = nullptr;
    double *inc_w = nullptr, *inc_n = nullptr, *inc_dx = nullptr;
    float *inc_w32 = nullptr, *inc_n32 = nullptr, *inc_dx32 = nullptr;
    float *ivol32 = nullptr;  // (float) 1/V, the FP32 gradient's volume input
    double *scal = nullptr;  // [0] dt, [1..5] l2 norms
    double *part = nullptr;  // per-block partials
    double *fin_mid = nullptr;  // first-level results of the two-level finish
    bool dt_valid = false;   // scal[0] holds the CFL time step of the current Old state
    double *pdt[2] = {nullptr, nullptr};  // per-block minima of the CFL time step: a step's last stage writes one
    int dt_from = -1;        // set while a step's stages take their time step from pdt[dt_from]
    int dt_to = 0;           // the array that dt-reducing launches write
    // Patch and fused kernels with 2 BLOCK lanes per patch (the halo's gradients beside the patch's, the faces in one
    // pass): where the time is one patch's and not the chip's.  Microseconds per SSP-RK2 step, BLOCK / 2 BLOCK
    // lanes, by patches: fused 2D triangles 23.6 / 20.4 (32), 31.0 / 28.7 (512), 40 / 46 (704); quadrilaterals FP64 31.4 /
    // 26.4 (224), 39.7 / 46.4 (308), 44.5 / 52.7 (512) and mixed 26.6 / 22.5 (224), 34.0 / 31.0 (512), so up to one
    // patch per CU in FP64 (run_fused_t); fused 3D 47.6 / 39.8 (188), 66 / 76 (324); first-order patch 2D 14.0 / 13.3
    // (176), 16.6 / 16.6 (313), 21.9 / 23.5 (704); patch 3D 36 / 32 (41), 57.0 / 54.4 (324), 80.3 / 80.9 (633).
    bool wide_patch = false;
    // Patches of SUB_PATCH cells where those of BLOCK cells would leave most of the chip idle: a stage's time is then
    // one patch's, and a patch of 64 cells is one wave of each phase's work on its compute unit instead of four (two in
    // a row on each SIMD).  One small patch per CU in 3D, two in 2D: beyond that their larger halo costs more.
    // Microseconds per step, wide patches / small ones, by blocks of BLOCK cells: fused 2D 20.3 / 16.4 (32), 20.5 /
    // 18.8 (95), 20.6 / 20.2 (133); first order 2D 11.4 / 9.9 (32), 11.8 / 11.7 (113), 12.0 / 13.2 (133); viscous 2D
    // 24.6 / 22.8 (32), 26.5 / 25.9 (113), 26.9 / 28.2 (133); patch 3D 31.2 / 29.2 (32), 31.6 / 29.8 (52), 32.4 /
    // 32.7 (80); first order 3D 17.0 / 15.8 (52), 17.1 / 17.7 (65); the mixed form in 3D 28.7 / 29.3 (24), so not there.
    // (A configuration of the other precision rebuilds the tables.)
    int patch_cells = BLOCK;  // BLOCK or SUB_PATCH
    int64_t n_patch = 0;
    int64_t dt_cnt[2] = {0, 0}, l2_cnt = 0;  // partials in pdt[i] and part, as their last writer left them
    int *bad = nullptr;
    Board *board = nullptr;  // pinned: the words the host waits for
    uint32_t board_seq = 0;
    int32_t *cnew = nullptr;  // device position of each file cell
    Transfer link;            // host states in file order
    bool viscous = false;     // mu or kappa > 0: the viscous kernels (viscous.hpp), patch or face route
    bool visc_patch = false;  // the mesh allows the patch route
    int g_of = -1;            // the state whose face fluxes G stands for but does not hold yet (ensure_fluxes), or -1
    double *gw = nullptr;     // viscous: per cell Green-Gauss gradients of (u, T), [nc][dim + 1][dim]
    // LU-SGS steady driver (built on first use): cell colours, the cells of each colour in ascending
    // order (colour k: lu_cells[lu_start[k] .. lu_start[k + 1])), face spectral radii, the update
    int32_t *lu_cells = nullptr, *lu_nb = nullptr, *lu_face = nullptr;
    uint32_t *lu_info = nullptr;
    std::vector<int64_t> lu_start;
    std::vector<int32_t> lu_colour;  // per cell (host copy)
    double *lu_n = nullptr, *lu_r = nullptr, *lu_D = nullptr, *lu_dQ = nullptr;
    int steady = MST_STEADY_EXPLICIT;
    double lu_cfl = 1e4, lu_omega = 1.0;
    bool lu_inline = false;  // the configuration lets the forward sweeps compute the residual (all but a
                             // call's last iteration do)
    bool timing = false;
    int timing_stride = 1;           // one launch in timing_stride of each kernel class carries events
    int64_t tick[MST_K_COUNT] = {};  // launches per kernel class since timing was enabled
    std::vector<std::pair<hipEvent_t, hipEvent_t>> ev[MST_K_COUNT];
    std::vector<hipEvent_t> pool;
};

namespace mstk {

inline hipEvent_t take_event(mst_ctx *x) {
    hipEvent_t e;
    if (!x->pool.empty()) {
        e = x->pool.back();
        x->pool.pop_back();
        return e;
    }
    if (hipEventCreate(&e) != hipSuccess) return nullptr;
    return e;
}

// A timed launch hands its two events to the dispatch itself (hipExtLaunchKernelGGL): they take the
// kernel's own start and end timestamps, with no marker packets between the kernels of a step, and
// the interval is the kernel alone.  Such a dispatch still costs about 3 us of throughput (12 us per
// step of four launches on the 2M-triangle vortex), so timing may sample one launch in n of each class.
// nt: lanes per block of BLOCK cells or faces.
template <typename K, typename... Args>
int launch_nt(mst_ctx *x, int kclass, K kernel, int64_t n, int nt, size_t shm, Args... args) {
    if (n <= 0) return MST_OK;
    const int64_t grid = (n + BLOCK - 1) / BLOCK;
    hipEvent_t e0 = nullptr, e1 = nullptr;
    if (x->timing && kclass >= 0 && x->tick[kclass]++ % x->timing_stride == 0) {
        e0 = take_event(x);
        e1 = take_event(x);
        if (!e0 || !e1) return mst::fail(MST_E_HIP, "hipEventCreate failed");
        hipExtLaunchKernelGGL(kernel, dim3((uint32_t)grid), dim3(nt), (uint32_t)shm, x->stream, e0, e1, 0, args...);
        HIPCHK(hipGetLastError());
        x->ev[kclass].push_back({e0, e1});
        return MST_OK;
    }
    hipLaunchKernelGGL(kernel, dim3((uint32_t)grid), dim3(nt), (uint32_t)shm, x->stream, args...);
    HIPCHK(hipGetLastError());
    return MST_OK;
}

// a kernel over the patches, nt lanes each
template <typename K, typename... Args>
int launch_patch(mst_ctx *x, int kclass, K kernel, int nt, size_t shm, Args... args) {
    return launch_nt(x, kclass, kernel, x->n_patch * BLOCK, nt, shm, args...);
}

template <typename K, typename... Args>
int launch(mst_ctx *x, int kclass, K kernel, int64_t nthreads, Args... args) {
    return launch_nt(x, kclass, kernel, nthreads, BLOCK, 0, args...);
}

template <typename T>
GradArgs<T> grad_args(const mst_ctx *x, int isrc, bool debug) {
    GradArgs<T> a;
    a.nc = x->nc;
    a.inc_code = x->inc_code;
    if constexpr (std::is_same<T, float>::value) {
        a.inc_w = x->inc_w32;
        a.inc_n = x->inc_n32;
        a.inc_dx = x->inc_dx32;
        a.Q = x->Q32[isrc];
        a.rec = x->rec32;
        a.vol = x->ivol32;
    } else {
        a.inc_w = x->inc_w;
        a.inc_n = x->inc_n;
        a.inc_dx = x->inc_dx;
        a.Q = x->Q[isrc];
        a.rec = x->rec;
        a.vol = x->cvol;
    }
    a.graw = debug ? x->graw : nullptr;
    a.phi = debug ? x->phi : nullptr;
    return a;
}

template <typename T>
FluxArgs<T> flux_args(const mst_ctx *x, int isrc) {
    FluxArgs<T> a;
    a.nf = x->nf;
    a.fc0 = x->fc0;
    a.fc1 = x->fc1;
    a.finfo = x->finfo;
    a.fn = x->fn;
    a.frec0 = x->frec0;
    a.frec1 = x->frec1;
    a.G = x->G;
    if constexpr (std::is_same<T, float>::value) {
        a.Q = x->Q32[isrc];
        a.rec = x->rec32;
        a.P = x->p32;
    } else {
        a.Q = x->Q[isrc];
        a.rec = x->rec;
        a.P = x->p64;
    }
    return a;
}

// the launch that follows writes n partials of what mode reduces
inline void partials(mst_ctx *x, int mode, int64_t n) {
    if (mode & UPD_DT) x->dt_cnt[x->dt_to] = n;
    if (mode & UPD_L2) x->l2_cnt = n;
}

inline UpdArgs upd_args(const mst_ctx *x, int mode, int is, int in, const Stage &sg, int iout) {
    UpdArgs a;
    a.nc = x->nc;
    a.ell = x->ell;
    a.G = x->G;
    a.Qs = is >= 0 ? x->Q[is] : nullptr;
    a.Qn = in >= 0 ? x->Q[in] : nullptr;
    a.vol = x->cvol;
    a.sh = x->cshalf;
    a.dt = x->scal;
    a.dt_part = x->dt_from >= 0 ? x->pdt[x->dt_from] : nullptr;
    a.dt_n = x->dt_from >= 0 ? (int)x->dt_cnt[x->dt_from] : 0;
    set_stage(a, sg);
    a.maxf = x->maxf;
    a.l2 = (mode & UPD_L2) != 0;
    a.dtred = (mode & UPD_DT) != 0;
    a.check = (mode & UPD_CHECK) != 0;
    a.gamma = x->cfg.gamma;
    a.cfl = x->cfg.cfl;
    a.Qout = iout >= 0 ? x->Q[iout] : nullptr;
    a.Qout32 = (iout >= 0 && x->mixed) ? x->Q32[iout] : nullptr;
    a.R = x->R;
    a.part_l2 = x->part;
    a.part_dt = x->pdt[x->dt_to];
    a.bad = x->bad;
    return a;
}

inline ViscArgs visc_args(const mst_ctx *x, int isrc) {
    ViscArgs a;
    a.nc = x->nc;
    a.nf = x->nf;
    a.inc_code = x->inc_code;
    a.ell = x->ell;
    a.finfo = x->finfo;
    a.inc_w = x->inc_w;
    a.inc_n = x->inc_n;
    a.vol = x->cvol;
    a.fc0 = x->fc0;
    a.fc1 = x->fc1;
    a.feta = x->feta;
    a.fn = x->fn;
    a.Q = x->Q[isrc];
    a.gw = x->gw;
    a.G = x->G;
    a.mu = x->cfg.mu;
    a.lam = x->cfg.lam;
    a.kappa = x->cfg.kappa;
    a.cv = x->cfg.cv;
    return a;
}

// whether kernels of dimension DIM and arithmetic T ever have patches of SUB_PATCH cells (patch_cells in solver.hip)
template <int DIM, typename T>
constexpr bool has_sub_patches() {
    return DIM == 2 || std::is_same<T, double>::value;
}

// one stage (mode includes UPD_STAGE) with the patch strategy (its gradient kernel has run) or the fused one;
// explicitly instantiated in their files
template <int DIM, typename T>
int run_patch_t(mst_ctx *x, int mode, int is, int in, const Stage &sg, int iout);
// (a viscous configuration: its viscous gradients have run too)
template <int DIM, typename T>
int run_fused_t(mst_ctx *x, int mode, int is, int in, const Stage &sg, int iout);
// the patch kernel's residual-only form (FP64): R of state is, and its L2 partials when mode has UPD_L2
template <int DIM>
int run_patch_residual_t(mst_ctx *x, int mode, int is);

}  // namespace mstk
