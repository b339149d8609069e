"""A batch most of whose runs have stopped: its steps take as long, and its runs end in
the same state, whatever the order in which the caller lists the runs."""

import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():  # pragma: no cover
    pytest.skip("no GPU", allow_module_level=True)

from coffeegpu_amd.solver import SimData, SimEnvironment  # noqa: E402
from coffeegpu_amd.spherical import SphBatch  # noqa: E402
from tests.golden.cases_sph import case_sph  # noqa: E402

RUNS, ON = 96, 12  # runs, and how many of them go on


# the first shape fills the rounds of the default tile so that, listed evenly, its 12
# runs met few of the workgroups: 1061 us for 4 steps, 314 in either order now
@pytest.mark.parametrize("n,dtype", [((16, 512), np.float32), ((128, 64), np.float64)])
def test_order_of_the_runs_does_not_matter(n, dtype):
    sp, U0 = case_sph(dtype, n=n, omega=0.3, pml=2, dt=1e-4)
    env = SimEnvironment(sp, dtype, "cuda:0")
    batches, states = [], []
    for on in (range(0, RUNS, RUNS // ON), range(ON)):
        datas = [SimData(env) for _ in range(RUNS)]
        for d in datas:
            d.set_state(U0)
        b = SphBatch([env] * RUNS, datas, nsteps=[10 ** 9 if r in on else 2 for r in range(RUNS)])
        b.step(4)
        assert sum(b.status()[0]) == ON
        k = list(on)
        off = next(r for r in range(RUNS) if r not in on)
        states.append([datas[k[0]].get_state(), datas[k[-1]].get_state(), datas[off].get_state()])
        batches.append(b)
    for a, c in zip(*states):
        assert np.array_equal(a, c)
    us = [1e30, 1e30]
    for _ in range(8):  # in turn; the least of each
        for k, b in enumerate(batches):
            b.step(4)
            torch.cuda.synchronize()
            t = time.perf_counter()
            for _ in range(10):
                b.step(4)
            torch.cuda.synchronize()
            us[k] = min(us[k], (time.perf_counter() - t) / 10 * 1e6)
    for b in batches:
        b.close()
    assert max(us) <= 1.3 * min(us), us
