"""Algorithmic bytes of the LU-SGS sweeps and of the viscous kernels against a count from the mesh, the colours and the
route that the stages take."""
import numpy as np
import pytest

import mstcfd as M
from helpers import brick_grid, cons

pytestmark = pytest.mark.gpu

MIX2 = (M.BC_INLET, M.BC_OUTLET, M.BC_WALL, M.BC_SYMMETRY)
MESHES = {
    "tri": lambda: M.Mesh.gen_tri(31, 20, 0, 3, 0, 2, 0.15, 7, MIX2),
    "periodic": lambda: M.Mesh.gen_tri(9, 9, -1, 1, -1, 1, 0.15, 3, (M.BC_PERIODIC,) * 4),
    "brick": lambda: M.Mesh.from_raw(brick_grid(24, 20, h=0.05, jitter=0.1, seed=5, bc=M.BC_WALL)),
    "tet": lambda: M.Mesh.gen_tet(6, 5, 4, (0, 0, 0), (1, 0.8, 0.7), 0.15, 11, MIX2 + (M.BC_WALL,) * 2),
}


def state(m):
    rng = np.random.default_rng(3)
    n = m.n_cells
    return cons(rng.uniform(0.95, 1.05, n), rng.uniform(-0.1, 0.1, (n, m.dim)), rng.uniform(0.95, 1.05, n))


def incidences(m):
    """(cell, neighbour or -1) of every incidence"""
    raw = m.raw()
    c0, c1 = np.asarray(raw["c0"]), np.asarray(raw["c1"])
    part = raw.get("partner")
    out = []
    for f in range(len(c0)):
        if c1[f] >= 0:
            out += [(c0[f], c1[f]), (c1[f], c0[f])]
        else:
            per = part is not None and raw["ftype"][f] == M.BC_PERIODIC
            out.append((c0[f], c0[part[f]] if per else -1))
    return np.array(out)


@pytest.mark.parametrize("order", [1, 2])
@pytest.mark.parametrize("name", sorted(MESHES))
def test_lusgs_sweeps(name, order):
    m = MESHES[name]()
    Q = state(m)
    s = M.Solver(m, M.make_config(dim=m.dim, order=order, limiter=M.LIM_MINMOD if order == 2 else M.LIM_NONE, q_inlet=list(Q[0])))
    s.set_state(Q)
    s.set_steady_driver(M.STEADY_LUSGS, 0.5, 1.0)
    s.lusgs_step(3)
    col, K = s.lusgs_colours()
    got = s.algorithmic_bytes(M.K_LUSGS)
    s.close()
    inc = incidences(m)
    most = np.bincount(inc[:, 0]).max()
    slots = 3 if most <= 3 else (4 if most <= 4 else 8)
    inline = order == 1 and slots <= 4
    V, D8 = 8 * m.nv, 8 * m.dim
    total = 0
    for k in range(K):
        n = int((col == k).sum())
        mine = inc[col[inc[:, 0]] == k]
        near = mine[mine[:, 1] >= 0]
        up = near[col[near[:, 1]] > k]
        lo, hi = (len(np.unique(x[:, 1])) for x in (near[col[near[:, 1]] < k], up))
        rec = 4 * n + 4 * min(slots * n, len(mine) + n)  # positions, neighbour codes
        source = 4 * n if inline else V * n  # face words, or the residual
        back = 8 * n + 8 * len(up) + V * (2 * n + 2 * hi)  # D, radii, states and updates
        if inline and K >= 2 and k == 0:
            total += rec + source + back + D8 * len(mine) + 8 * len(mine) + 8 * n + 2 * V * n  # radii, D, state and update out
            continue
        total += rec + source + D8 * len(mine) + V * (n + lo + hi) + V * lo + V * n
        total += V * n if k == K - 1 else 8 * len(mine) + 8 * n
        if k < K - 1:
            total += rec + back + D8 * len(up) + 2 * V * n
    launches = 2 * K - 2 if inline and K >= 2 else 2 * K - 1
    print(f"{name} order {order}: {K} colours, {got:.0f} B per launch, counted {total / launches:.0f}", flush=True)
    assert got == pytest.approx(total / launches, rel=1e-12)


@pytest.mark.parametrize("order,prec", [(1, M.PREC_FP64), (2, M.PREC_FP64), (2, M.PREC_MIXED)])
@pytest.mark.parametrize("name", ["brick", "tet", "tri"])
def test_viscous_kernels(name, order, prec):
    m = MESHES[name]()
    Q = state(m)
    inc = incidences(m)
    n, nf, D, NV = m.n_cells, m.n_faces, m.dim, m.nv
    nb = int((inc[:, 1] < 0).sum())
    most = np.bincount(inc[:, 0]).max()
    slots = 3 if most <= 3 else (4 if most <= 4 else 8)
    gw = 8 * (D + 1) * D * n
    vgrad = 4 * slots * n + len(inc) * (8 + 8 * D) + 8 * nb + n * (8 * NV + 8) + gw
    vface = nf * (8 + 4 + 8 * D + 16 * NV) + 8 * (nf - nb) + 8 * NV * n + gw
    lim = M.LIM_MINMOD if order == 2 else M.LIM_NONE
    cfg = lambda mu: M.make_config(dim=m.dim, order=order, limiter=lim, rk=2, precision=prec, q_inlet=list(Q[0]), mu=mu,
                                   kappa=mu, cv=2.5)
    s = M.Solver(m, cfg(0.0))
    plain = {k: s.algorithmic_bytes(k) for k in (M.K_GRAD, M.K_PATCH)}
    s.set_config(cfg(0.03))
    for st in (M.STRATEGY_FACE, M.STRATEGY_CELL, M.STRATEGY_AUTO):
        s.strategy = st
        s.set_state(Q)
        s.set_dt(1e-4)
        s.timing_reset()
        s.timing(True)
        s.step(2)
        s.timing(False)
        patch = s.timing_get(M.K_PATCH)[0] > 0  # the route that ran
        assert patch == (name != "brick" and st != M.STRATEGY_FACE)
        fused = patch and order == 2 and prec == M.PREC_FP64  # one kernel for both gradients
        assert (s.timing_get(M.K_VISC)[0] == 0) == fused
        assert s.algorithmic_bytes(M.K_GRAD) == plain[M.K_GRAD] + (gw + 8 * nb if fused else 0)
        assert s.algorithmic_bytes(M.K_VISC) == (vgrad if patch else 0.5 * (vgrad + vface))
        if patch and prec == M.PREC_FP64:  # (the mixed form's stages read Q^n differently when they are viscous)
            assert s.algorithmic_bytes(M.K_PATCH) == plain[M.K_PATCH] + gw + 8 * (nf - nb)
    s.close()
