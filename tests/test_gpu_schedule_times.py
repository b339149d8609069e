"""The schedule that a 3D solver picks by the box's size takes no longer than one set
by hand: boxes a few cells wide, where tiles and thread-per-cell launches idle most of
their lanes, and slabs, whose chunks along z are all start-up."""

import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():  # pragma: no cover
    pytest.skip("no GPU", allow_module_level=True)

from coffeegpu_amd import initial_data as ic  # noqa: E402
from coffeegpu_amd.gr import FieldSolverGREZ  # noqa: E402
from coffeegpu_amd.params import Grid, SimParams  # noqa: E402
from coffeegpu_amd.solver import FieldSolverEZ, SimData, SimEnvironment  # noqa: E402


# (variant, zchunk) set by hand; the picked schedule took 1.16 to 1.58 times as long
@pytest.mark.parametrize("gr,n,dtype,by_hand", [
    (False, (8, 8, 2000), np.float64, (3, 0)), (False, (4, 158, 158), np.float64, (3, 0)),
    (False, (254, 844, 7), np.float32, (2, 7)), (False, (212, 708, 10), np.float32, (2, 10)),
    (True, (73, 1468, 14), np.float32, (0, 7)), (True, (194, 644, 12), np.float32, (0, 6))])
def test_picked_schedule_is_no_slower(gr, n, dtype, by_hand):
    d = 1.0 / max(n)
    sp = SimParams(dt=0.1 * d, N=list(n), guard=[3, 3, 3], lower=[3.0, 3.0, 3.0] if gr else [0.0] * 3,
                   size=[v * d for v in n], nodes=[1, 1, 1], periodic_boundary=[not gr] * 3, pml=[0, 0, 0],
                   KOeps=0.1, use_edotb_damping=False, problem=0, KO_geometry=False, a=0.5)
    g = Grid.from_params(sp, dtype)
    U0 = 0.01 * np.random.default_rng(3).standard_normal((7,) + g.shape)
    U0[5] += 1.0
    U0 = ic.periodic_fill(U0, g, sp.periodic_boundary).astype(dtype)
    env = SimEnvironment(sp, dtype, "cuda:0")
    data = SimData(env)
    data.set_state(U0)
    solver = (FieldSolverGREZ if gr else FieldSolverEZ)(data, env)
    us = [1e30, 1e30]
    for _ in range(8):  # in turn; the least of each
        for k, sched in enumerate(((0, 0), by_hand)):
            solver.set_schedule(*sched)
            solver.evolve_fields(0.0)
            torch.cuda.synchronize()
            t = time.perf_counter()
            for _ in range(12):
                solver.evolve_fields(0.0)
            torch.cuda.synchronize()
            us[k] = min(us[k], (time.perf_counter() - t) / 12 * 1e6)
    solver.close()
    assert us[0] <= 1.1 * us[1], us
