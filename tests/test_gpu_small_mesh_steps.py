"""Patch kernels with two block sizes and the time step reduced between or inside the steps' kernels, at the patch
counts where the choice changes (256 | 257 and 512 | 513): the strategies agree bit for bit (the face strategy has
one block size), and steps in one call equal the same steps in one call each (whose time step takes the
other route)."""
import numpy as np
import pytest

import mstcfd as M

pytestmark = pytest.mark.gpu

BC2 = (M.BC_INLET, M.BC_OUTLET, M.BC_WALL, M.BC_SYMMETRY)
BC3 = BC2 + (M.BC_SYMMETRY, M.BC_WALL)


def tri(nx, ny):
    return M.Mesh.gen_tri(nx, ny, 0, 4, 0, 2, 0.1, 3, BC2)


MESHES = {  # name: (mesh, patches)
    "2d_1": (lambda: tri(3, 2), 1),
    "2d_256": (lambda: tri(256, 128), 256),
    "2d_257": (lambda: tri(32769, 1), 257),
    "2d_512": (lambda: tri(512, 128), 512),
    "2d_513": (lambda: tri(65537, 1), 513),
    "3d_256": (lambda: M.Mesh.gen_tet(32, 31, 11, jitter=0.1, seed=4, bc=BC3), 256),
    "3d_260": (lambda: M.Mesh.gen_tet(33, 24, 14, jitter=0.1, seed=4, bc=BC3), 260),
    "3d_514": (lambda: M.Mesh.gen_tet(32, 33, 21, jitter=0.1, seed=4, bc=BC3), 520),
}


@pytest.mark.parametrize("name", sorted(MESHES))
@pytest.mark.parametrize("order,prec", [(1, M.PREC_FP64), (2, M.PREC_FP64), (2, M.PREC_MIXED)])
def test_block_sizes_and_time_step_routes(name, order, prec):
    mk, patches = MESHES[name]
    m = mk()
    assert (m.n_cells + 255) // 256 == patches
    print(f"small mesh steps {name}: {m.n_cells} cells, order {order}, precision {prec}", flush=True)
    cc = m.cell_centres()
    Q = np.empty((m.n_cells, m.nv))
    Q[:, 0] = 1 + 0.1 * np.sin(3 * cc[:, 0])
    Q[:, 1:-1] = 0.2 * Q[:, :1]
    Q[:, -1] = 2.5 + 0.2 * np.cos(2 * cc[:, 1])
    qin = Q[0].tolist()
    s = M.Solver(m, M.make_config(scheme=M.ROE, order=order, limiter=M.LIM_VANLEER, rk=2, cfl=0.4, dim=m.dim, precision=prec,
                                  q_inlet=qin))
    ref = None
    for st in (M.STRATEGY_FACE, M.STRATEGY_PATCH, M.STRATEGY_FUSED):
        try:
            s.strategy = st
        except M.MstError:
            continue  # (fused 3D: a patch beyond 64 KiB)
        s.set_state(Q)
        s.step(4)
        out, norms = s.get_state(), s.residual_norms()
        s.set_state(Q)
        for _ in range(4):
            s.step(1)
        assert np.array_equal(s.get_state(), out) and np.array_equal(s.residual_norms(), norms)
        if ref is None:
            ref = out
        assert np.all(np.isfinite(out)) and np.array_equal(out, ref)
    s.close()
