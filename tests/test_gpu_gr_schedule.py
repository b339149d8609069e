"""The schedule the Kerr-Schild solver picks by grid size (point + stage sweep
below 100 000 cells, tiled with automatic z chunks above) against forced
ones: bitwise the same state, on both sides of the line and with partial
tiles and chunks."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():  # pragma: no cover - CPU containers
    pytest.skip("no GPU", allow_module_level=True)

from coffeegpu_amd.gr import FieldSolverGREZ  # noqa: E402
from coffeegpu_amd.solver import SimData, SimEnvironment  # noqa: E402
from tests.golden.cases_gr import case_gr  # noqa: E402


@pytest.mark.parametrize("n", [(46, 47, 46), (47, 47, 46), (70, 66, 40), (65, 130, 33)])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_picked_schedule_is_bitwise_the_same(n, dtype):
    d = 8.0 / max(n)
    sp, U0 = case_gr(dtype, a=0.7, n=n, lower=tuple(-0.5 * d * v for v in n),
                     size=tuple(d * v for v in n), pml=(3, 3, 3))
    env = SimEnvironment(sp, dtype, "cuda:0")
    outs = []
    for variant, zchunk in ((0, 0), (1, 0), (3, 7)):
        data = SimData(env)
        data.set_state(U0)
        solver = FieldSolverGREZ(data, env)
        solver.set_schedule(variant, zchunk)
        for _ in range(2):
            solver.evolve_fields(0.0)
        outs.append(data.get_state())
        solver.close()
    assert np.isfinite(outs[0]).all()
    for o in outs[1:]:
        assert np.array_equal(o, outs[0])
