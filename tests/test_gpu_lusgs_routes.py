"""Several LU-SGS iterations in one call (the residual computed in the sweeps, colour 0's sweeps fused) equal the same
iterations one call each (the residual kernels) bit for bit, in a context and in a batch: Roe and AUSM cases, triangles,
quadrilaterals, tetrahedra, two and three colours, periodic faces (a mesh one cell pair wide too), a boundary of unknown
type, an inactive case, a changed configuration."""
import os

import numpy as np
import pytest

import mstcfd as M
from helpers import cons, periodic_in_x, quad_grid

pytestmark = pytest.mark.gpu

GOLDEN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "msh_2d-stair-un-5-tri.npz")


def unknown_side():
    raw = M.Mesh.gen_tri(30, 20, 0, 3, 0, 2, 0.15, 7, (M.BC_INLET, M.BC_OUTLET, M.BC_WALL, M.BC_SYMMETRY)).raw()
    raw["ftype"][raw["ftype"] == M.BC_SYMMETRY] = 36  # no Fluent type the solver knows: no convective flux
    return M.Mesh.from_raw(raw)


def stair():
    d = dict(np.load(GOLDEN))
    for k in ("dim", "n_cells", "n_int"):
        d[k] = int(d[k])
    return M.Mesh.from_raw(d)


GROUPS = {
    "tri": (lambda: M.Mesh.gen_tri(1, 1, 0, 1, 0, 1, 0.0, 1, (M.BC_INLET, M.BC_OUTLET, M.BC_WALL, M.BC_SYMMETRY)),
            lambda: M.Mesh.gen_tri(41, 25, 0, 4, 0, 2, 0.1, 7, (M.BC_INLET, M.BC_OUTLET, M.BC_WALL, M.BC_SYMMETRY)),
            lambda: M.Mesh.gen_tri(1, 9, 0, 1, 0, 9, 0.0, 3, (M.BC_PERIODIC,) * 2 + (M.BC_WALL,) * 2),
            unknown_side, stair,
            lambda: M.Mesh.gen_tri(24, 24, -1, 1, -1, 1, 0.15, 3, (M.BC_PERIODIC,) * 4)),
    "quad": (lambda: M.Mesh.from_raw(quad_grid(24, bc=M.BC_WALL, h=0.05, jitter=0.2, seed=4)),
             lambda: M.Mesh.gen_tri(13, 11, 0, 1, 0, 1, 0.1, 7, (M.BC_WALL,) * 4)),
    "tet": (lambda: M.Mesh.gen_tet(6, 5, 4, (0, 0, 0), (1, 0.8, 0.7), 0.15, 12,
                                   (M.BC_INLET, M.BC_OUTLET, M.BC_SYMMETRY, M.BC_WALL, M.BC_SYMMETRY, M.BC_SYMMETRY)),
            lambda: M.Mesh.from_raw(periodic_in_x(M.Mesh.gen_tet(6, 5, 4, (0, 0, 0), (1, 0.8, 0.7), 0.0, 13,
                                                                 (M.BC_WALL,) * 6).raw()))),
}


@pytest.mark.parametrize("n_iter", [2, 3, 5])
@pytest.mark.parametrize("name", sorted(GROUPS))
def test_iterations_together_equal_one_by_one(name, n_iter):
    meshes = [f() for f in GROUPS[name]]
    dim = meshes[0].dim
    qin = list(cons(np.array([1.2]), np.array([[0.6] + [0.1] * (dim - 1)]), np.array([1.1]))[0])
    schemes = [(M.AUSM, M.ROE)[i % 2] for i in range(len(meshes))]
    mk = lambda scheme, compat=0: M.make_config(dim=dim, scheme=scheme, order=1, q_inlet=qin, compat=compat, cfl=0.5)
    rng = np.random.default_rng(n_iter)
    states, want = [], []
    for m, scheme in zip(meshes, schemes):
        print(f"lusgs routes {name}: {m.n_cells} cells, scheme {scheme}, {n_iter} iterations", flush=True)
        n = m.n_cells
        q = cons(rng.uniform(0.9, 1.1, n), rng.uniform(-0.2, 0.2, (n, dim)), rng.uniform(0.9, 1.1, n))
        states.append(q)
        s = M.Solver(m, mk(scheme))
        s.set_steady_driver(M.STEADY_LUSGS, 0.5, 1.0)
        runs = []
        for compat in (0, M.COMPAT_BRANCH2_LR):  # the second configuration flips masks after the records were built
            s.set_config(mk(scheme, compat))
            for calls in ([1] * n_iter, [n_iter]):
                s.set_state(q)
                for k in calls:
                    s.lusgs_step(k)
                runs.append((s.get_state(), s.residual_norms()))
            assert np.all(np.isfinite(runs[-1][0]))
            assert np.array_equal(runs[-2][0], runs[-1][0]) and np.array_equal(runs[-2][1], runs[-1][1])
        want.append(runs[0])
        s.close()
    plain = [i for i, m in enumerate(meshes) if not np.any(m.raw()["ftype"] == M.BC_PERIODIC)]  # all a batch takes
    b = M.Batch([meshes[i] for i in plain], [mk(schemes[i]) for i in plain])
    for k, i in enumerate(plain):
        b.set_state(k, states[i])
    b.set_steady_driver(M.STEADY_LUSGS, 0.5, 1.0)
    act = np.ones(len(plain), np.uint8)
    act[-1] = len(plain) == 1
    b.set_active(act)
    b.lusgs_step(n_iter)
    for k, i in enumerate(plain):
        assert np.array_equal(b.get_state(k), want[i][0] if act[k] else states[i]), i
    b.close()
