"""The schedule the flat solver picks by grid size (thread-per-cell, 64 x 4, 64 x 8
or 128 x 8 tiles, one or several z chunks, tiles not in eights) against forced ones: bitwise the same
state, guards included.  Sizes on both sides of each line of the rule, with
remainders in every axis."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():  # pragma: no cover - CPU containers
    pytest.skip("no GPU", allow_module_level=True)

from coffeegpu_amd import initial_data as ic  # noqa: E402
from coffeegpu_amd.params import Grid, SimParams  # noqa: E402
from coffeegpu_amd.solver import FieldSolverEZ, SimData, SimEnvironment  # noqa: E402


@pytest.mark.parametrize("n", [(50, 51, 50), (52, 51, 50), (66, 67, 68), (67, 67, 68), (81, 83, 81),
                               (82, 83, 81), (127, 40, 70), (129, 190, 33), (256, 130, 9),
                               (192, 160, 64), (75, 77, 78), (92, 93, 94), (127, 126, 126),
                               (136, 136, 136)])
@pytest.mark.parametrize("problem", [0, 1])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_picked_schedule_is_bitwise_the_same(n, problem, dtype):
    box = [v / max(n) for v in n]
    sp = SimParams(dt=0.1 / max(n), N=list(n), guard=[3, 3, 3], lower=[-0.5 * b for b in box], size=box,
                   nodes=[1, 1, 1], periodic_boundary=[problem == 0] * 3, pml=[0, 0, 0], KOeps=0.1,
                   use_edotb_damping=False, problem=problem, radius=0.1, omega=0.5, b0=1.0,
                   KO_geometry=False)
    g = Grid.from_params(sp, dtype)
    rng = np.random.default_rng(3)
    U0 = 0.1 * rng.standard_normal((7,) + g.shape)
    U0[5] += 1.0
    U0 = ic.periodic_fill(U0, g, sp.periodic_boundary).astype(dtype)
    env = SimEnvironment(sp, dtype, "cuda:0")
    outs = []
    for variant, zchunk in ((0, 0), (1, 0), (2, 7)):
        data = SimData(env)
        data.set_state(U0)
        solver = FieldSolverEZ(data, env)
        solver.set_schedule(variant, zchunk)
        for s in range(2):
            solver.evolve_fields(s * sp.dt)
        outs.append(data.get_state())
        solver.close()
    assert np.isfinite(outs[0]).all()
    for o in outs[1:]:
        assert np.array_equal(o, outs[0])


# FP32 boxes that get 128 x 8 tiles (by the cost estimate 86 planes against 108 of 64 x
# 8, 50 against 62), and with a star on both sides of the line at 10 M cells, above
# which it gets them too (84 against 107)
@pytest.mark.parametrize("n,problem", [((254, 259, 131), 0), ((382, 350, 21), 0), ((250, 245, 163), 1),
                                       ((253, 245, 167), 1)])
def test_picked_schedule_of_large_boxes(n, problem):
    test_picked_schedule_is_bitwise_the_same(n, problem, np.float32)


# FP64 at the line by cells of tiles (148480 and 151040 of them, 49 of 64 columns and
# all filled), narrow boxes, FP32 at its line and slabs whose plane has 498 and 500
# tiles of 64 x 4
@pytest.mark.parametrize("n,problem,dtype", [
    ((49, 38, 58), 0, np.float64), ((49, 40, 59), 0, np.float64), ((64, 40, 58), 0, np.float64),
    ((64, 40, 59), 0, np.float64), ((8, 9, 500), 0, np.float64), ((4, 33, 200), 0, np.float64),
    ((66, 66, 68), 0, np.float32), ((65, 996, 8), 0, np.float32), ((65, 1000, 8), 0, np.float32),
    ((65, 1000, 8), 1, np.float32), ((254, 844, 7), 0, np.float32)])
def test_picked_schedule_of_narrow_boxes_and_slabs(n, problem, dtype):
    test_picked_schedule_is_bitwise_the_same(n, problem, dtype)
