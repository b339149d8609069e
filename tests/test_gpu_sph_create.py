"""Tables of a batch are filled for all runs in one launch when it is made: runs of
several grids get what each of them gets alone."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():  # pragma: no cover
    pytest.skip("no GPU", allow_module_level=True)

import oracle as O  # noqa: E402
from coffeegpu_amd.solver import SimData, SimEnvironment  # noqa: E402
from coffeegpu_amd.spherical import SphBatch  # noqa: E402
from tests.golden.cases_sph import case_sph  # noqa: E402


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_runs_of_several_grids_get_their_own_tables(dtype):
    """Theta extents from the smallest to more than one launch row covers, each run
    with another star: each as a batch of its own."""
    cases = [case_sph(dtype, n=n, omega=w, pml=2)
             for n, w in (((16, 4), 0.3), ((12, 1100), 0.2), ((70, 33), 0.25), ((16, 256), 0.1))]

    def run(cs):
        envs = [SimEnvironment(sp, dtype, "cuda:0") for sp, _ in cs]
        datas = [SimData(e) for e in envs]
        for d, (_, U) in zip(datas, cs):
            d.set_state(U)
        b = SphBatch(envs, datas, nsteps=[0] * len(cs))
        b.step(2)
        out = [d.get_state() for d in datas]
        b.close()
        return out

    together = run(cases)
    for case, got in zip(cases, together):
        assert np.array_equal(run([case])[0], got)
        if dtype == np.float64:
            ref = O.SphState(case[1], dtype)
            O.sph_evolve(case[0], ref, 2)
            assert O.rel_l2(got, ref.U) <= 1e-12
