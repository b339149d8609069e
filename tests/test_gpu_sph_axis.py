"""Axis rows and clocks of the spherical batch: the copies stored by the tile
kernels, the axis launch of the march kernels, the preparation once per call
and the two alternating clocks of a run.  From the smallest theta extent (the
rows next to both axes overlap) to partial tiles; steps taken in calls of odd
and even length, replayed and direct; one run retiring on the way; a caller
that changes the state between calls."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():  # pragma: no cover
    pytest.skip("no GPU", allow_module_level=True)

import oracle as O  # noqa: E402
from coffeegpu_amd.solver import SimData, SimEnvironment  # noqa: E402
from coffeegpu_amd.spherical import SphBatch, tile_shapes  # noqa: E402
from tests.golden.cases_sph import case_sph  # noqa: E402

CALLS = (1, 2, 3)


@pytest.mark.parametrize("n", [(8, 4), (65, 5), (70, 33)])
@pytest.mark.parametrize("tile", [0, 5, 10])
@pytest.mark.parametrize("graph", [False, True])
def test_axis_rows_and_clocks(n, tile, graph):
    dtype = np.float64
    sp, U0 = case_sph(dtype, n=n, omega=0.3, dw0=0.2, pml=2)
    rng = np.random.default_rng(4)
    U0 = U0 + 1e-3 * rng.standard_normal(U0.shape)
    env = SimEnvironment(sp, dtype, "cuda:0")
    datas = [SimData(env) for _ in range(2)]
    for d in datas:
        d.set_state(U0)
    stop = 4
    b = SphBatch([env, env], datas, nsteps=[0, stop])
    assert tile < len(tile_shapes())
    b.set_tile(tile)
    b.use_graph(graph)
    ref = [O.SphState(U0, dtype), O.SphState(U0, dtype)]
    done = 0
    for k in CALLS:
        b.step(k)
        left = min(k, max(0, stop - done))
        O.sph_evolve(sp, ref[0], k, time=done * sp.dt)
        if left:
            O.sph_evolve(sp, ref[1], left, time=done * sp.dt)
        done += k
        active, t, steps = b.status()
        assert steps == [done, min(done, stop)] and active == [1, int(done < stop)]
        for d, r in zip(datas, ref):
            # the solver's FP64 parity tolerance, guard rows included
            assert O.rel_l2(d.get_state(), r.U) <= 1e-12
        # the caller writes its own arrays between calls: the axis boundary is
        # applied to them again at the start of the next one
        if not (done >= stop):
            for d, r in zip(datas, ref):
                U = r.U * 1.25
                d.set_state(U)
                for q in range(7):
                    r.U[q][...] = U[q]
    b.close()


# total cells on both sides of the lines (FP32 800 k, FP64 100 k), extents off every
# tile shape, runs that stop together and runs that do not (either order of the
# work list)
@pytest.mark.parametrize("dtype,n", [(np.float32, (799, 500)), (np.float32, (801, 501)),
                                     (np.float64, (333, 150)), (np.float64, (335, 151))])
@pytest.mark.parametrize("stops", [(0, 0), (1, 3)])
def test_default_tile_is_bitwise_the_first(dtype, n, stops):
    sp, U0 = case_sph(dtype, n=n, omega=0.3, dw0=0.2, pml=2)
    env = SimEnvironment(sp, dtype, "cuda:0")
    outs = []
    for tile in (None, 0, 11):
        datas = [SimData(env) for _ in range(2)]
        for d in datas:
            d.set_state(U0)
        b = SphBatch([env, env], datas, nsteps=list(stops))
        if tile is not None:
            b.set_tile(tile)
        b.step(2)
        outs.append([d.get_state() for d in datas])
        b.close()
    for o in outs[1:]:
        for x, y in zip(o, outs[0]):
            assert np.array_equal(x, y)
