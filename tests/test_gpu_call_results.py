"""The few words a call waits for: the monitor's maxima against numpy (bit for bit: one subtraction and one division per
value), the time step of each call in order, the flag of a non-physical state raised once and cleared, norms and time
steps read back, and a warm start whose features do not fit a spare state buffer."""
import numpy as np
import pytest

import mstcfd as M
from helpers import cons

pytestmark = pytest.mark.gpu

MESHES = {  # one block, 257 partials and more (a second pass of the one finishing block), 3D
    "tri2": lambda: M.Mesh.gen_tri(1, 1, 0, 1, 0, 1, 0.0, 1, (M.BC_WALL,) * 4),
    "tri70k": lambda: M.Mesh.gen_tri(200, 175, 0, 2, 0, 2, 0.1, 5, (M.BC_WALL,) * 4),
    "tet": lambda: M.Mesh.gen_tet(7, 6, 5, (0, 0, 0), (1, 1, 1), 0.1, 3, (M.BC_WALL,) * 6),
}


def state(m, seed):
    rng = np.random.default_rng(seed)
    n = m.n_cells
    return cons(rng.uniform(0.9, 1.1, n), rng.uniform(0.05, 0.2, (n, m.dim)), rng.uniform(0.9, 1.1, n))


@pytest.mark.parametrize("name", sorted(MESHES))
def test_monitor_time_step_and_flag(name):
    m = MESHES[name]()
    print(f"call results {name}: {m.n_cells} cells", flush=True)
    Q = state(m, 2)
    cfg = M.make_config(dim=m.dim, scheme=M.ROE, order=1, cfl=0.4)
    s = M.Solver(m, cfg)
    s.set_state(Q)
    good = s.compute_dt(0.4)
    old = Q
    for dt in (0.5 * good, 0.25 * good, good):  # each call's own time step
        s.set_dt(dt)
        s.solve()
        mon = s.monitor_maxrel()
        s.update_new_to_old()
        new = s.get_state()
        assert np.array_equal(mon, np.maximum(0, np.abs(new - old) / old).max(0))
        one = M.Solver(m, cfg)
        one.set_state(old)
        one.set_dt(dt)
        one.solve()
        one.update_new_to_old()
        assert np.array_equal(one.get_state(), new)
        one.close()
        old = new
    for _ in range(2):
        s.set_state(Q)
        s.set_dt(1e6 * good)
        with pytest.raises(M.MstError):
            s.solve()
        s.set_state(Q)  # the flag is gone with the report
        s.set_dt(good)
        s.solve()
    assert s.compute_dt(0.4) == good
    s.step(2)
    assert np.all(np.isfinite(s.residual_norms()))
    s.close()


@pytest.mark.parametrize("n_cond", [1, 6, 8])
def test_warm_start_scratch(n_cond):
    m = MESHES["tri70k"]()
    print(f"warm start: {m.n_cells} cells, {n_cond} conditions", flush=True)
    net = M.MLP(2 + n_cond, 16, 2, 4, seed=3)
    cond = [0.5] + [0.1 * k for k in range(1, n_cond)]
    got = []
    for rounds in (1, 2):
        s = M.Solver(m, M.make_config(scheme=M.ROE, order=2, limiter=M.LIM_VANLEER, rk=2, cfl=0.3))
        s.set_state(state(m, 4))
        for _ in range(rounds):
            s.step(1)
            s.warm_start(net, cond)
        got.append(s.get_state())
        s.close()
    assert np.all(np.isfinite(got[0])) and np.array_equal(got[0], got[1])
    net.close()
