"""The z-marching tiled kernels of the 3D solvers on the small parity boxes, where
the default schedule is one thread per cell (flat) or the point sweep (Kerr-Schild):
state, currents, divergences and energy accounting against the CPU oracle and, bitwise,
against the other schedule.  Production boxes run these kernels."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():  # pragma: no cover
    pytest.skip("no GPU", allow_module_level=True)

import oracle as O  # noqa: E402
from coffeegpu_amd.gr import FieldSolverGREZ  # noqa: E402
from coffeegpu_amd.params import Grid  # noqa: E402
from coffeegpu_amd.solver import FieldSolverEZ, SimData, SimEnvironment  # noqa: E402
from tests.golden.cases import CASES  # noqa: E402
from tests.golden.cases_gr import GR_CASES, case_gr  # noqa: E402

ACC = ("dU_KO", "dU_Epar", "dU_EgtB", "dU_KO_cum", "dU_Epar_cum", "dU_EgtB_cum")


def run(cls, sp, U0, dtype, nsteps, sched, diag=False, bbg=None):
    env = SimEnvironment(sp, dtype, "cuda:0")
    data = SimData(env)
    data.set_state(U0)
    solver = cls(data, env)
    solver.set_schedule(*sched)
    if bbg is not None:
        for n in range(3):
            solver.Bbg.data(n).set(bbg[n])
    if diag:
        solver.set_diagnostics(True)
    t = np.dtype(dtype).type(0.0)
    for _ in range(nsteps):
        solver.evolve_fields(float(t))
        t = np.dtype(dtype).type(t + np.dtype(dtype).type(sp.dt))
    torch.cuda.synchronize()
    out = {"U": data.get_state().copy()}
    if diag:
        out["J"] = np.stack([data.B0.data(n).sync_to_host() for n in range(3)])
        out["divE"], out["divB"] = data.divE.sync_to_host().copy(), data.divB.sync_to_host().copy()
        if cls is FieldSolverEZ:
            out.update({k: getattr(data, k).sync_to_host().copy() for k in ACC})
    lanes = getattr(solver, "mask_lanes", 1)
    solver.close()
    return out, lanes


# default tile in chunks of 3 planes, 64 x 4, 64 x 8, 64 x 16 (FP64 64 x 8), 256 x 4 (FP64 128 x 4)
TILES = ((0, 3), (2, 0), (3, 5), (4, 0), (6, 4))


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("name", list(CASES))
def test_flat_diagnostics_of_the_tiled_kernels(name, dtype):
    sp, U0 = CASES[name](dtype)
    bbg = O.flat_bbg(sp, dtype) if any(sp.pml) else None
    want, _ = run(FieldSolverEZ, sp, U0, dtype, 3, (1, 0), True, bbg)
    plain, _ = run(FieldSolverEZ, sp, U0, dtype, 3, (2, 0), False, bbg)
    assert np.array_equal(plain["U"], want["U"])
    for sched in TILES:
        got, _ = run(FieldSolverEZ, sp, U0, dtype, 3, sched, True, bbg)
        for k, v in want.items():
            assert np.array_equal(got[k], v), (sched, k)


@pytest.mark.parametrize("name", list(CASES))
@pytest.mark.parametrize("sched", [(0, 3), (2, 0)])
def test_flat_tiled_kernels_match_the_oracle(name, sched):
    """FP64, the quantities, cases and tolerances of the default schedule's tests: the
    state of every case, the accounting of the noise and pulsar ones (1e-10 of the largest
    value), current and divergences of the noise one."""
    dtype = np.float64
    sp, U0 = CASES[name](dtype)
    bbg = O.flat_bbg(sp, dtype) if any(sp.pml) else None
    shape, it = U0.shape[1:], Grid.from_params(sp, dtype).interior()

    def oracle(nsteps, lanes, diag):
        ref = O.FlatState(U0, dtype, bbg)
        O.flat_evolve(sp, ref, nsteps, mask_lanes=lanes, diag=diag)
        return ref.U

    got, lanes = run(FieldSolverEZ, sp, U0, dtype, 3, sched, True, bbg)
    acc = {k: np.zeros(shape) for k in ACC}
    assert O.rel_l2(got["U"], oracle(3, lanes, acc)) <= 1e-12
    if name in ("noise", "pulsar"):
        for k, ref in acc.items():
            assert np.abs(got[k][it] - ref[it]).max() <= 1e-10 * max(np.abs(ref[it]).max(), 1e-300), k
    if name == "noise":
        got, lanes = run(FieldSolverEZ, sp, U0, dtype, 1, sched, True, bbg)
        diag = {"J": [np.zeros(shape) for _ in range(3)], "divE": np.zeros(shape), "divB": np.zeros(shape)}
        oracle(1, lanes, diag)
        for n in range(3):
            assert O.rel_l2(got["J"][n][it], diag["J"][n][it]) <= 1e-12
        for k in ("divE", "divB"):
            assert O.rel_l2(got[k][it], diag[k][it]) <= 1e-12


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("name", list(GR_CASES))
def test_gr_tiled_kernels(name, dtype):
    """Halo three planes ahead (FP32 default), one ahead (variant 3), from the table
    (variant 2): state and diagnostics of the point sweep, bitwise."""
    sp, U0 = case_gr(dtype, **GR_CASES[name])
    want, _ = run(FieldSolverGREZ, sp, U0, dtype, 3, (1, 0), True)
    for sched in ((0, 5), (0, 24), (3, 0), (2, 7)):
        for diag in (True, False):
            got, _ = run(FieldSolverGREZ, sp, U0, dtype, 3, sched, diag)
            for k, v in got.items():
                assert np.array_equal(v, want[k]), (sched, k)


@pytest.mark.parametrize("name", list(GR_CASES))
def test_gr_tiled_kernels_match_the_oracle(name):
    sp, U0 = case_gr(np.float64, **GR_CASES[name])
    it = Grid.from_params(sp, np.float64).interior()
    got, _ = run(FieldSolverGREZ, sp, U0, np.float64, 10, (0, 5))
    st = O.GrState(U0)
    O.gr_evolve(sp, st, 10)
    assert O.rel_l2(got["U"], st.U) <= 1e-12
    got, _ = run(FieldSolverGREZ, sp, U0, np.float64, 1, (0, 5), True)
    shape = U0.shape[1:]
    d = {"J": np.zeros((3,) + shape), "divB": np.zeros(shape), "divE": np.zeros(shape)}
    O.gr_evolve(sp, O.GrState(U0), 1, diag=d)
    for k in ("divB", "divE", "J"):
        ref, val = (v[(slice(None),) + it] if k == "J" else v[it] for v in (d[k], got[k]))
        assert np.abs(val - ref).max() <= 1e-10 * max(np.abs(ref).max(), 1e-30), k
