"""Meshes with patches of 64 cells against the face strategy (blocks of 256) bit for bit: states, residual norms (whose
partials are joined to those of 256 cells) and CFL time steps, at one cell pair, ragged last patches and blocks, and
either side of the sizes where the small patches end; both orders, schemes and precisions, and the implicit driver."""
import numpy as np
import pytest

import mstcfd as M
from helpers import cons

pytestmark = pytest.mark.gpu

MIX2 = (M.BC_INLET, M.BC_OUTLET, M.BC_WALL, M.BC_SYMMETRY)
BOX = MIX2 + (M.BC_WALL,) * 2
tri = lambda nx, ny: M.Mesh.gen_tri(nx, ny, 0, 4, 0, 2, 0.1, 7, MIX2)
tet = lambda n: M.Mesh.gen_tet(n, n, n, (0, 0, 0), (1, 1, 1), 0.1, 3, BOX)
MESHES = {
    "2": lambda: tri(1, 1), "66": lambda: tri(11, 3), "234": lambda: tri(13, 9), "322": lambda: tri(23, 7),
    "32768": lambda: tri(128, 128), "32770": lambda: tri(145, 113),
    "162 3D": lambda: tet(3), "13182 3D": lambda: tet(13), "16464 3D": lambda: tet(14),
}


@pytest.mark.parametrize("prec", [M.PREC_FP64, M.PREC_MIXED])
@pytest.mark.parametrize("name", sorted(MESHES))
def test_sub_patches_equal_face(name, prec):
    m = MESHES[name]()
    rng = np.random.default_rng(8)
    n = m.n_cells
    print(f"sub patches {name}: {n} cells, precision {prec}", flush=True)
    Q = cons(rng.uniform(0.95, 1.05, n), rng.uniform(-0.1, 0.1, (n, m.dim)), rng.uniform(0.95, 1.05, n))
    for scheme, order, lim in ((M.ROE, 1, M.LIM_NONE), (M.AUSM, 2, M.LIM_MINMOD)):
        out = []
        for st in (M.STRATEGY_FACE, M.STRATEGY_PATCH, M.STRATEGY_FUSED):
            s = M.Solver(m, M.make_config(dim=m.dim, scheme=scheme, order=order, limiter=lim, rk=2, cfl=0.2, precision=prec,
                                          q_inlet=list(Q[0])))
            s.strategy = st
            s.set_state(Q)
            s.step(1)
            r1 = s.residual_norms()
            s.step(3)
            got = [s.get_state(), r1, s.residual_norms(), np.array(s.compute_dt(0.2))]
            if prec == M.PREC_FP64:
                s.set_steady_driver(M.STEADY_LUSGS, 0.5, 1.0)
                s.lusgs_step(2)
                got += [s.get_state(), s.residual_norms()]
            out.append(got)
            s.close()
        for got in out:
            assert all(np.all(np.isfinite(g)) for g in got)
            assert all(np.array_equal(g, w) for g, w in zip(got, out[0])), (scheme, order)
