"""States between host (file order) and device (curve order), at sizes around the chunks of the transfer:
one cell row, exactly one chunk and one record more, several chunks with an odd remainder, 2D and 3D."""
import numpy as np
import pytest

import mstcfd as M
from oracle import pyoracle as O

pytestmark = pytest.mark.gpu

MESHES = {
    "one": lambda: M.Mesh.gen_tri(1, 1, 0, 1, 0, 1, 0.0, 1),
    "chunk": lambda: M.Mesh.gen_tri(256, 128, 0, 2, 0, 1, 0.1, 2),       # 65,536 cells x 4 = 2^18 doubles
    "chunk+": lambda: M.Mesh.gen_tri(32769, 1, 0, 1, 0, 0.001, 0.1, 3),  # 65,538 cells
    "many": lambda: M.Mesh.gen_tri(401, 311, 0, 4, 0, 3, 0.1, 4),        # 249,422 cells: 4 chunks
    "tet": lambda: M.Mesh.gen_tet(23, 22, 21, jitter=0.1, seed=5),       # 63,756 cells x 5 (records across pairs)
}


@pytest.mark.parametrize("name", sorted(MESHES))
def test_state_round_trip_and_order(name):
    m = MESHES[name]()
    print(f"transfer {name}: {m.n_cells} cells", flush=True)
    rng = np.random.default_rng(7)
    cc = m.cell_centres()
    Q = np.empty((m.n_cells, m.nv))
    Q[:, 0] = 1 + 0.1 * np.sin(5 * cc[:, 0]) + 0.01 * rng.uniform(size=m.n_cells)
    Q[:, 1:-1] = 0.1 * Q[:, :1] * np.cos(3 * cc)
    Q[:, -1] = 2.5
    s = M.Solver(m, M.make_config(order=1, dim=m.dim))
    s.set_state(Q)
    assert np.array_equal(s.get_state(), Q)
    if m.n_cells > 2:  # every record in its own cell: the gradient of a varying field against the oracle's
        g, _ = s.gradient()
        gr = O.OracleMesh(m.raw()).gradient(O.make_config(order=1, dim=m.dim), Q)
        assert np.abs(g - gr.reshape(g.shape)).max() <= 1e-9 * np.abs(gr).max()
    s.close()


def test_batch_round_trip_with_growing_and_inactive_cases():
    rng = np.random.default_rng(8)
    ms = [M.Mesh.gen_tri(nx, 2, 0, 1, 0, 0.01, 0.1, 9) for nx in (1, 50, 17000, 3)]  # 68,000 cells: two chunks
    b = M.Batch(ms, [M.make_config(order=1, rk=2, cfl=0.5)] * len(ms))
    Qs = [np.column_stack([rng.uniform(1, 1.1, (m.n_cells, 3)) * [1, 0.1, 0.1], rng.uniform(2, 2.1, m.n_cells)]) for m in ms]
    b.set_active([True, False, True, True])
    for i, Q in enumerate(Qs):
        b.set_state(i, Q)
    for i, Q in enumerate(Qs):
        assert np.array_equal(b.get_state(i), Q)
    b.step(3)
    assert np.array_equal(b.get_state(1), Qs[1])
    assert all(not np.array_equal(b.get_state(i), Qs[i]) for i in (0, 2, 3))
    b.close()
