"""The monitor on large meshes: its maxima either side of the sizes where its partials and its finishing block change
form (2,048 blocks of 256 cells, 8,192), and its time, which is that of the pass over the states, as the allocation-free
monitor's, and not the finish's."""
import ctypes as C
import time

import numpy as np
import pytest
import torch

import mstcfd as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,nz", [(512, 512, 0), (641, 409, 0), (1024, 1024, 0), (1049, 1000, 0), (2000, 2000, 0),
                                      (45, 45, 44)])
def test_monitor_of_many_blocks(nx, ny, nz):
    m = M.Mesh.gen_tet(nx, ny, nz, (0, 0, 0), (1, 1, 1), 0.0, 7, (M.BC_WALL,) * 6) if nz else \
        M.Mesh.gen_tri(nx, ny, 0, 4, 0, 2, 0.0, 7, (M.BC_WALL,) * 4)
    n = m.n_cells
    print(f"monitor: {n} cells", flush=True)
    rng = np.random.default_rng(nx)
    Q = rng.uniform(1, 2, (n, m.nv))
    Q[:, -1] += 8
    s = M.Solver(m, M.make_config(dim=m.dim, order=1, q_inlet=list(Q[0])))
    s.strategy = M.STRATEGY_PATCH
    s.set_dt(1e-9)
    for at in (None, 0, n - 1, n // 2):
        q = Q.copy()
        if at is not None:
            q[at] *= 3
        s.set_state(q)
        s.solve()
        s.set_state(Q)  # Old is another state: the largest ratio is where it was changed
        new = s.get_new_state()
        assert np.array_equal(s.monitor_maxrel(), np.maximum(0, np.abs(new - Q) / Q).max(0)), at
    if n == 8_000_000:  # what bounds it: 512 MB of states
        a, b = (torch.from_numpy(x).cuda() for x in (new, Q))
        out = torch.zeros(4, dtype=torch.float64, device="cuda")
        f = M.lib().mst_monitor_maxrel_noalloc
        f.restype, f.argtypes = C.c_int, [C.c_void_p] * 2 + [C.c_int64, C.c_int, C.c_void_p, C.c_void_p]

        def plain():
            assert f(a.data_ptr(), b.data_ptr(), n, 4, out.data_ptr(), None) == 0
            torch.cuda.synchronize()

        t = {}
        for name, g in (("plain", plain), ("monitor", s.monitor_maxrel)):
            for _ in range(5):
                g()
            w = []
            for _ in range(40):
                t0 = time.perf_counter()
                g()
                w.append(time.perf_counter() - t0)
            t[name] = float(np.median(w)) * 1e6
        print(f"monitor {t['monitor']:.1f} us, allocation-free {t['plain']:.1f} us", flush=True)
        # the finish: one round of loads, 10 us with its launch; the plain one waits by a synchronisation
        assert t["monitor"] <= t["plain"] + 10
    s.close()
