"""The patch kernels on both sides of the sizes where blocks of twice the lanes end (256 patches in 2D, 512 in 3D), and
with a last patch of two cells, against the face strategy bit for bit: inviscid and viscous, both orders and schemes."""
import numpy as np
import pytest

import mstcfd as M
from helpers import cons

pytestmark = pytest.mark.gpu

MIX2 = (M.BC_INLET, M.BC_OUTLET, M.BC_WALL, M.BC_SYMMETRY)
MESHES = {
    "256 patches": lambda: M.Mesh.gen_tri(256, 128, 0, 4, 0, 2, 0.1, 7, MIX2),
    "257 patches": lambda: M.Mesh.gen_tri(331, 99, 0, 4, 0, 2, 0.1, 7, MIX2),
    "462 patches 3D": lambda: M.Mesh.gen_tet(27, 27, 27, (0, 0, 0), (1, 1, 1), 0.1, 3, MIX2 + (M.BC_WALL,) * 2),
    "515 patches 3D": lambda: M.Mesh.gen_tet(28, 28, 28, (0, 0, 0), (1, 1, 1), 0.1, 3, MIX2 + (M.BC_WALL,) * 2),
}


@pytest.mark.parametrize("mu", [0.0, 0.02])
@pytest.mark.parametrize("name", sorted(MESHES))
def test_patch_equals_face(name, mu):
    m = MESHES[name]()
    rng = np.random.default_rng(5)
    n = m.n_cells
    print(f"patch sizes {name}: {n} cells, mu {mu}", flush=True)
    Q = cons(rng.uniform(0.95, 1.05, n), rng.uniform(-0.1, 0.1, (n, m.dim)), rng.uniform(0.95, 1.05, n))
    for scheme, order, lim in ((M.ROE, 1, M.LIM_NONE), (M.ROE, 2, M.LIM_VANLEER), (M.AUSM, 2, M.LIM_MINMOD)):
        out = []
        for st in (M.STRATEGY_FACE, M.STRATEGY_PATCH):
            s = M.Solver(m, M.make_config(dim=m.dim, scheme=scheme, order=order, limiter=lim, rk=2, cfl=0.2, mu=mu, kappa=mu,
                                          cv=2.5, q_inlet=list(Q[0])))
            s.strategy = st
            s.set_state(Q)
            s.step(2)
            out.append((s.get_state(), s.residual_norms()))
            s.close()
        assert np.all(np.isfinite(out[0][0]))
        assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])
