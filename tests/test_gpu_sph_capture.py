"""Calls of a spherical batch recorded in a graph of the caller's: every replay
takes the recorded number of steps on from whatever ran before it (replays of odd
and even length, direct calls, the batch's own graphs), bitwise as direct calls of
the same lengths do, with a twist pulse (its boundary takes the time of the step)
and past the step at which a run stops; recording alone advances nothing."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():  # pragma: no cover
    pytest.skip("no GPU", allow_module_level=True)

from coffeegpu_amd.solver import SimData, SimEnvironment  # noqa: E402
from coffeegpu_amd.spherical import SphBatch  # noqa: E402
from tests.golden.cases_sph import case_sph  # noqa: E402


def make(dtype, tile):
    sp, U0 = case_sph(dtype, n=(65, 21), omega=0.3, dw0=0.2, pml=2)
    rng = np.random.default_rng(4)
    U0 = (U0 + 1e-3 * rng.standard_normal(U0.shape)).astype(dtype)
    env = SimEnvironment(sp, dtype, "cuda:0")
    datas = [SimData(env) for _ in range(3)]
    for d in datas:
        d.set_state(U0)
    b = SphBatch([env] * 3, datas, nsteps=[0, 9, 14])
    b.set_tile(tile)
    return b, datas


def record(b, k):
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        b.step(k)
    return g


@pytest.mark.parametrize("tile", [0, 10])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_replays_go_on_from_the_state_before_them(dtype, tile):
    b, datas = make(dtype, tile)
    ref, rdatas = make(dtype, tile)
    g1, g3 = record(b, 1), record(b, 3)
    assert b.status() == ref.status()  # recording ran nothing

    def same():
        torch.cuda.synchronize()
        assert b.status() == ref.status()
        for d, r in zip(datas, rdatas):
            assert np.array_equal(d.get_state(), r.get_state())

    # (steps, how): r = replay of the recorded call, d = a direct call, g = a direct call
    # through the batch's own graphs
    for k, how in ((1, "d"), (1, "r"), (1, "r"), (3, "r"), (2, "d"), (3, "r"), (1, "r"), (1, "g"),
                   (1, "r"), (3, "g"), (3, "r"), (1, "r"), (1, "d")):
        if how == "r":
            (g1 if k == 1 else g3).replay()
        else:
            b.use_graph(how == "g")
            b.step(k)
        ref.step(k)
        same()
    assert ref.status()[0] == [1, 0, 0] and ref.status()[2] == [22, 9, 14]
    b.close()
    ref.close()


@pytest.mark.parametrize("warm", [0, 1, 4])
def test_recording_a_batch_that_replays_its_own_graphs(warm):
    b, datas = make(np.float64, 0)
    ref, rdatas = make(np.float64, 0)
    b.use_graph(True)
    if warm:
        b.step(warm)
        ref.step(warm)
    g = record(b, 3)
    torch.cuda.synchronize()
    assert b.status() == ref.status()
    for _ in range(3):
        g.replay()
        ref.step(3)
        b.step(1)
        ref.step(1)
        torch.cuda.synchronize()
        assert b.status() == ref.status()
        for d, r in zip(datas, rdatas):
            assert np.array_equal(d.get_state(), r.get_state())
    b.close()
    ref.close()
