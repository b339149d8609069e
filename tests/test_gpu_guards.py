"""Guard cells of the flat solver after a step: the periodic images stored by
the last stage (P) and Kreiss-Oliger (E, B), the fill kernel of boxes with a
frozen axis, and the frozen guards copied to the partner buffers.  Sizes from
the smallest periodic axis (n = guard: a cell then has images on both sides)
to partial tiles."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():  # pragma: no cover - CPU containers
    pytest.skip("no GPU", allow_module_level=True)

import oracle as O  # noqa: E402
from coffeegpu_amd import initial_data as ic  # noqa: E402
from coffeegpu_amd.params import Grid, SimParams  # noqa: E402
from coffeegpu_amd.solver import FieldSolverEZ, SimData, SimEnvironment  # noqa: E402

PERIODIC = [(True, True, True), (False, True, True), (True, False, False), (False, False, False)]


@pytest.mark.parametrize("n", [(3, 3, 3), (5, 4, 7), (70, 9, 11)])
@pytest.mark.parametrize("periodic", PERIODIC)
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_guard_cells_after_a_step(n, periodic, dtype):
    sp = SimParams(dt=0.1 / max(n), N=list(n), guard=[3, 3, 3], lower=[0.0] * 3, size=[1.0] * 3,
                   nodes=[1, 1, 1], periodic_boundary=list(periodic), pml=[0, 0, 0], KOeps=0.1,
                   use_edotb_damping=False, problem=0, KO_geometry=False)
    g = Grid.from_params(sp, dtype)
    rng = np.random.default_rng(5)
    U0 = 0.1 * rng.standard_normal((7,) + g.shape)
    U0[5] += 1.0
    U0 = ic.periodic_fill(U0, g, periodic).astype(dtype)
    env = SimEnvironment(sp, dtype, "cuda:0")
    outs = []
    for variant, zchunk in ((0, 0), (1, 0), (2, 2)):
        data = SimData(env)
        data.set_state(U0)
        solver = FieldSolverEZ(data, env)
        solver.set_schedule(variant, zchunk)
        for _ in range(2):
            solver.evolve_fields(0.0)
        outs.append(data.get_state())
        lanes = solver.mask_lanes
        solver.close()
    got = outs[0]
    # guards along a periodic axis hold the wrapped cells, exactly
    assert np.array_equal(got, ic.periodic_fill(got, g, periodic))
    for o in outs[1:]:
        assert np.array_equal(o, got)
    ref = O.FlatState(U0, dtype, None)
    O.flat_evolve(sp, ref, 2, mask_lanes=lanes)
    # the solver's parity tolerances, guards included
    assert O.rel_l2(got, ref.U) <= (1e-12 if dtype == np.float64 else 1e-5)
