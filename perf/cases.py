"""Timed workloads of the framework through its public entry points.

Each case is one kind of work at one size: time steps of the three field
solvers (flat 3D, Kerr-Schild 3D, log-spherical 2D alone and batched) and the
learned warm start's network (one layer, one training iteration, one
prediction).  `listed` holds the sizes the project's own configurations,
tests and benchmark use, from the smallest to the largest; `draw` gives others
of the same ranges.  `exact` evaluates the same work in FP64 with plain torch.
"""

import ctypes
import math

import numpy as np
import torch

from coffeegpu_amd import _lib
from coffeegpu_amd.gr import FieldSolverGREZ
from coffeegpu_amd.params import SimParams
from coffeegpu_amd.solver import FieldSolverEZ, SimData, SimEnvironment
from coffeegpu_amd.spherical import FieldSolverEZSpherical, SphBatch
from coffeegpu_amd.surrogate import UNet, layer_specs, pad16

DEV = "cuda:0"
SWEEP_GRIDS = ((512, 256), (1024, 512), (2048, 1024))


# ---- the cases -------------------------------------------------------------


def listed():
    return [
        # the smallest box of the parity tests: launches and latency count
        dict(name="flat_wave_32_f32", kind="flat", problem=0, nx=32, ny=32, nz=32, f64=False),
        # an FP64 production box whose axes are no multiples of anything
        dict(name="flat_alfven_ragged_f64", kind="flat", problem=0, nx=150, ny=123, nz=101, f64=True),
        # rotating multipole star in an absorbing box (frozen guards)
        dict(name="flat_pulsar_f32", kind="flat", problem=1, nx=160, ny=128, nz=120, f64=False),
        # the headline benchmark
        dict(name="flat_alfven_512_f32", kind="flat", problem=0, nx=512, ny=512, nz=512, f64=False),
        # Kerr-Schild Wald problem in FP64 on a ragged box, and the benchmark's size
        dict(name="gr_wald_ragged_f64", kind="gr", nx=92, ny=74, nz=61, f64=True, spin=0.5),
        dict(name="gr_wald_384_f32", kind="gr", nx=384, ny=384, nz=384, f64=False, spin=0.9),
        # one spherical run stepped alone, as a reference driver does
        dict(name="sph_single_f64", kind="sph1", nr=256, nth=128, f64=True),
        # the warm start's relaxation: many small runs, luminosity sampled between chunks of steps
        dict(name="sph_relax_64x128x64_f32", kind="relax", runs=64, nr=128, nth=64, steps=20),
        # the batched sweep over the benchmark's three grids, tile autotuned, graph replay
        dict(name="sph_sweep_48_f32", kind="sweep", runs=48, scale=1.0),
        # one convolution layer: forward, weight and bias gradient, input gradient
        dict(name="unet_layer_128", kind="layer", n=8, h=64, w=128, cin=128, cout=128),
        # one training iteration of the warm start (forward, loss, backward, Adam)
        dict(name="unet_train_8x64x128", kind="train", n=8, h=64, w=128, levels=4, base=32),
        # prediction for a batch of held-out runs
        dict(name="unet_predict_16x128x256", kind="predict", n=16, h=128, w=256, levels=4, base=32),
    ]


def draw(rng):
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    def box(lo, hi):
        n = log_int(lo, hi)
        return [max(lo, min(hi, int(round(n * rng.uniform(0.8, 1.25))))) for _ in range(3)]

    kind = rng.choice(["flat", "flat", "flat", "gr", "sph1", "relax", "sweep", "layer", "layer",
                       "train", "predict"])
    if kind == "flat":
        n = box(24, 256)
        return dict(kind=kind, problem=rng.choice([0, 0, 1]), nx=n[0], ny=n[1], nz=n[2],
                    f64=rng.random() < 0.4)
    if kind == "gr":
        n = box(32, 192)
        return dict(kind=kind, nx=n[0], ny=n[1], nz=n[2], f64=rng.random() < 0.4,
                    spin=round(rng.uniform(0.0, 0.95), 3))
    if kind == "sph1":
        return dict(kind=kind, nr=log_int(64, 1024), nth=log_int(32, 512), f64=rng.random() < 0.5)
    if kind == "relax":
        return dict(kind=kind, runs=log_int(4, 128), nr=8 * log_int(8, 32), nth=8 * log_int(4, 16),
                    steps=rng.randint(5, 20))
    if kind == "sweep":
        return dict(kind=kind, runs=log_int(4, 48), scale=round(rng.uniform(0.25, 1.0), 3))
    if kind == "layer":
        return dict(kind=kind, n=rng.randint(1, 16), h=log_int(8, 128), w=log_int(8, 160),
                    cin=rng.choice([16, 32, 64, 96, 128, 256]),
                    cout=rng.choice([16, 32, 64, 96, 128, 256]))
    return dict(kind=kind, n=rng.randint(1, 16), h=8 * log_int(4, 16), w=8 * log_int(4, 32),
                levels=rng.choice([3, 4]), base=32)


def work(case):
    """Bytes: state in and out once per step (network: inputs, weights and
    results once); flops: the arithmetic of the scheme per cell and step."""
    kind = case["kind"]
    if kind in ("flat", "gr"):
        cells = case["nx"] * case["ny"] * case["nz"]
        return {"bytes": 14 * (8 if case["f64"] else 4) * cells,
                "flops": (1250 if kind == "flat" else 3000) * cells}
    if kind == "sph1":
        cells = case["nr"] * case["nth"]
        return {"bytes": 14 * (8 if case["f64"] else 4) * cells, "flops": 1700 * cells}
    if kind == "relax":
        cells = case["runs"] * case["nr"] * case["nth"]
        return {"bytes": 14 * 4 * cells * case["steps"], "flops": 1700 * cells * case["steps"]}
    if kind == "sweep":
        cells = sum(a * b for a, b in _sweep_grids(case))
        return {"bytes": 14 * 4 * cells, "flops": 1700 * cells}
    pix = case["n"] * case["h"] * case["w"]
    if kind == "layer":
        ci, co = case["cin"], case["cout"]
        return {"bytes": 2 * pix * (2 * ci + 2 * co) + 9 * ci * co * (2 * 2 + 4),
                "flops": 3 * 2 * 9 * ci * co * pix}
    flops = nw = 0
    for name, ci, co, _ in layer_specs(case["levels"], case["base"], 7, 6):
        level = 0 if name == "head" else int(name[3])
        flops += 2 * 9 * ci * co * (pix >> (2 * level))
        nw += 9 * ci * co + co
    if kind == "predict":
        return {"bytes": pix * (2 * 16 + 4 * 16) + 4 * nw, "flops": flops}
    return {"bytes": pix * (2 * 16 + 4 * 6 + 4 * 16) + 4 * nw * 7, "flops": 3 * flops}


# ---- parameters and inputs ---------------------------------------------------


def _np_type(case):
    return np.float64 if case.get("f64") else np.float32


def _flat_params(case):
    n = [case["nx"], case["ny"], case["nz"]]
    if case["problem"] == 0:
        return SimParams(dt=0.4 / max(n), N=n, guard=[3, 3, 3], lower=[0.0] * 3, size=[1.0] * 3,
                         nodes=[1, 1, 1], periodic_boundary=[True] * 3, pml=[0, 0, 0],
                         divB_clean=True, ch2=1.0, tau=2.0, KOeps=0.1, use_edotb_damping=False,
                         problem=0, KO_geometry=False)
    d = 4.0 / n[0]
    size = [d * v for v in n]
    return SimParams(dt=0.32 * d, N=n, guard=[3, 3, 3], lower=[-0.5 * s - 0.5 * d for s in size],
                     size=size, nodes=[1, 1, 1], periodic_boundary=[False] * 3,
                     pml=[max(3, v // 10) for v in n], pmllen=max(2, n[0] // 16), sigpml=0.5,
                     divB_clean=True, ch2=1.0, tau=2.0, KOeps=0.2, use_edotb_damping=False,
                     problem=1, radius=0.55, omega=0.3, b0=1.0, p1=0.1, p2=0.0, p3=1.0, q11=0.05,
                     q12=0.02, q13=0.01, q22=-0.03, q23=0.02, q_offset_x=0.05, q_offset_z=0.02,
                     KO_geometry=False)


def _gr_params(case):
    n = [case["nx"], case["ny"], case["nz"]]
    d = 40.0 / max(n)
    size = [d * v for v in n]
    return SimParams(dt=0.3 * d, N=n, guard=[3, 3, 3], lower=[-0.5 * s for s in size], size=size,
                     nodes=[1, 1, 1], periodic_boundary=[False] * 3, pml=[max(3, v // 12) for v in n],
                     pmllen=1, sigpml=10.0, divB_clean=True, ch2=1.0, tau=2.0, KOeps=0.1,
                     use_edotb_damping=False, problem=0, a=case["spin"])


def _sph_params(nr, nth, rlc, ko_geometry):
    r_out, r_abs, x0 = 60.0, 48.0, -0.1
    size_x = math.log(r_out) - x0
    dx, dth = size_x / nr, math.pi / nth
    pml = int(math.ceil((math.log(r_out) - math.log(r_abs)) / dx))
    return SimParams(dt=0.4 * min(dx, dth), N=[nr, nth, 1], guard=[3, 4, 0], lower=[x0, 0.0, 0.0],
                     size=[size_x, math.pi, 0.0], nodes=[1, 1, 1],
                     periodic_boundary=[False] * 3, pml=[pml, 0, 0], pmllen=10, sigpml=1.0,
                     divB_clean=True, ch2=1.0, tau=2.0, KOeps=0.1, KO_geometry=ko_geometry,
                     use_edotb_damping=False, problem=0, radius=1.0, omega=1.0 / rlc, b0=1.0)


def _sweep_grids(case):
    s = case["scale"]
    return [tuple(max(16, int(v * s)) for v in SWEEP_GRIDS[(7 * r + 1) % 3])
            for r in range(case["runs"])]


def _rng(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(1000003 + seed)
    return g


def _axes(sp):
    """Node positions per axis (guards included), shaped for (z, y, x) arrays, FP64."""
    out = []
    for a in range(3):
        d = sp.size[a] / sp.N[a]
        i = torch.arange(sp.N[a] + 2 * sp.guard[a], dtype=torch.float64, device=DEV)
        p = sp.lower[a] + d * (i - sp.guard[a])
        shape = [1, 1, 1]
        shape[2 - a] = p.numel()
        out.append(p.view(shape))
    return out


def _alfven_state(sp, seed, dt):
    """Two counter-propagating Alfven packets on B = z in the unit box, with
    the small cleaning potential a run carries after its first steps."""
    u = np.random.default_rng(seed).uniform(size=5)
    x, y, z = _axes(sp)

    def gauss(zc):
        d = z - zc
        d = (d + 0.5) - torch.floor(d + 0.5) - 0.5
        return torch.exp(-d * d / 0.02)

    b1 = (0.1 + 0.4 * u[0]) * gauss(0.25) * torch.sin(2 * math.pi * (x + u[2]))
    b2 = (0.1 + 0.4 * u[1]) * gauss(0.75) * torch.sin(2 * math.pi * (y + u[3]))
    shape = [t.numel() for t in (z, y, x)]
    zero = torch.zeros((1, 1, 1), dtype=torch.float64, device=DEV)
    p = 1e-3 * torch.sin(2 * math.pi * (x + 2 * z + u[4])) * torch.cos(2 * math.pi * y)
    comp = (b1, b2, zero, b2, b1, zero + 1.0, p)
    return [torch.broadcast_to(c, shape).to(dt).contiguous() for c in comp]


def _multipole(sp, x, y, z, phase, tiny):
    """Rotating dipole + offset quadrupole field."""
    c, s = math.cos(phase), math.sin(phase)
    p = (sp.p1 * c - sp.p2 * s, sp.p1 * s + sp.p2 * c, sp.p3)
    q11 = sp.q11 * c * c - 2 * sp.q12 * c * s + sp.q22 * s * s
    q12 = sp.q12 * math.cos(2 * phase) + (sp.q11 - sp.q22) * c * s
    q22 = sp.q22 * c * c + sp.q11 * s * s + 2 * sp.q12 * c * s
    q13, q23, q33 = sp.q13 * c - sp.q23 * s, sp.q23 * c + sp.q13 * s, -sp.q11 - sp.q22
    r2 = x * x + y * y + z * z
    den = r2 * torch.sqrt(r2) + tiny
    pr = p[0] * x + p[1] * y + p[2] * z
    x1 = x - (sp.q_offset_x * c - sp.q_offset_y * s)
    y1 = y - (sp.q_offset_x * s + sp.q_offset_y * c)
    z1 = z - sp.q_offset_z
    R2 = x1 * x1 + y1 * y1 + z1 * z1
    R7 = R2 ** 3 * torch.sqrt(R2) + tiny
    xqx = (q11 * x1 * x1 + 2 * q12 * x1 * y1 + q22 * y1 * y1 + 2 * (q13 * x1 + q23 * y1) * z1
           + q33 * z1 * z1)
    rows = ((q11, q12, q13), (q12, q22, q23), (q13, q23, q33))
    out = []
    for n in range(3):
        a = rows[n]
        dip = (3.0 * (x, y, z)[n] * pr / (r2 + tiny) - p[n]) / den
        quad = (-2.0 * (a[0] * x1 + a[1] * y1 + a[2] * z1) * R2 + 5.0 * (x1, y1, z1)[n] * xqx) / R7
        out.append(sp.b0 * (dip + quad))
    return out


def _pulsar_state(sp, seed, dt, tiny):
    x, y, z = _axes(sp)
    b = _multipole(sp, x, y, z, 0.0, tiny)
    g = _rng(seed)
    zero = torch.zeros_like(b[0])
    r2 = x * x + y * y + z * z
    noise = [1e-3 * torch.randn(zero.shape, dtype=torch.float64, device=DEV, generator=g)
             * torch.exp(-r2) for _ in range(6)]
    comp = [noise[0], noise[1], noise[2], b[0] + noise[3], b[1] + noise[4], b[2] + noise[5], zero]
    return [c.to(dt).contiguous() for c in comp]


def _cks(a, x, y, z):
    """Cartesian Kerr-Schild: r, s = 2H, s/(1+s), l (M = 1)."""
    tiny = 1e-11
    w = x * x + y * y + z * z - a * a
    r = torch.sqrt((w + torch.sqrt(torch.clamp(w * w + 4 * (a * z) ** 2, min=tiny))) / 2)
    q = r ** 4 + (a * z) ** 2
    A = torch.clamp(a * a + r * r, min=tiny)
    s = 2 * r ** 3 / torch.clamp(q, min=tiny)
    bu = 2 * r ** 3 / torch.clamp(q + 2 * r ** 3, min=tiny)
    lz = torch.where(r > 0, z / torch.where(r > 0, r, torch.ones_like(r)), torch.zeros_like(r))
    return r, s, bu, ((r * x + a * y) / A, (r * y - a * x) / A, lz)


def _wald_state(sp, seed, dt):
    x, y, z = _axes(sp)
    _, s, _, _ = _cks(sp.a, x, y, z)
    bz = 1.0 / torch.sqrt(1.0 + s)
    del s
    g = _rng(seed)
    out = []
    for n in range(7):
        v = torch.zeros(bz.shape, dtype=dt, device=DEV)
        if 3 <= n < 6:
            v += 1e-3 * torch.randn(bz.shape, dtype=dt, device=DEV, generator=g)
        if n == 5:
            v += bz.to(dt)
        out.append(v)
    return out


def _magnetosphere(sp, seed, dt):
    """A rotating magnetosphere some way into its relaxation, in upper
    components of (ln r, theta): aligned dipole of seeded strength, E
    corotating inside the light cylinder (E.B = 0), swept-back B_phi."""
    x, y, _ = _axes(sp)
    r, sn = torch.exp(x), torch.sin(y)
    b0 = sp.b0 * (1.0 + 0.01 * float(np.random.default_rng(seed).uniform()))
    w = sp.omega / torch.sqrt(1.0 + (sp.omega * r) ** 2)
    bx = b0 * 2.0 * torch.cos(y) / r ** 4
    by = b0 * sn / r ** 4
    comp = (w * r * sn * by, -w * r * sn * bx, 0.0 * bx, bx, by, -0.5 * w * sn * r * bx, 0.0 * bx)
    shape = (1, y.numel(), x.numel())
    return [torch.broadcast_to(c, shape).to(dt) for c in comp]


def _fill(data, state):
    for arr, src in zip(data.state_arrays(), state):
        arr.dev.copy_(src)


def _pool(datas):
    """Moves the state arrays of runs of one grid into one allocation, each
    array at a 256-byte boundary; returns it as (run, field, scalars)."""
    first = datas[0].P.dev
    per = (first.numel() * first.element_size() + 255) // 256 * 256 // first.element_size()
    pool = torch.zeros((len(datas), 7, per), dtype=first.dtype, device=DEV)
    for r, d in enumerate(datas):
        for c, arr in enumerate(d.state_arrays()):
            arr.dev = pool[r, c, :first.numel()].view(first.shape)
    return pool


def _sph_runs(case, seed):
    """(parameters, state seed) of every run of a batch."""
    rng = np.random.default_rng(seed)
    if case["kind"] == "sph1":
        grids = [(case["nr"], case["nth"])]
    elif case["kind"] == "relax":
        grids = [(case["nr"], case["nth"])] * case["runs"]
    else:
        grids = _sweep_grids(case)
    return [(_sph_params(nr, nth, float(rng.uniform(3.0, 20.0)), case["kind"] != "relax"),
             int(rng.integers(1 << 30))) for nr, nth in grids]


def _groups(runs):
    """Indices of the runs of each grid."""
    groups = {}
    for i, (sp, _) in enumerate(runs):
        groups.setdefault((sp.N[0], sp.N[1]), []).append(i)
    return list(groups.values())


def _net_params(case, seed):
    """Seeded weights W[ky, kx, ci, co] and biases of every layer."""
    rng = np.random.default_rng(seed)
    out = {}
    for name, ci, co, _ in layer_specs(case["levels"], case["base"], 7, 6):
        w = rng.standard_normal((3, 3, ci, co)) * math.sqrt(2.0 / (9 * ci))
        out[name] = (w.astype(np.float32), (0.05 * rng.standard_normal(co)).astype(np.float32))
    return out


def _net_input(case, seed):
    """BF16 images: 6 field channels falling off along the radial axis, one
    constant R_LC channel, zero padding; and FP32 targets."""
    g = _rng(seed)
    n, h, w = case["n"], case["h"], case["w"]
    fall = torch.exp(-torch.linspace(0.0, 2.0, w, device=DEV)).view(1, 1, w, 1)
    x = torch.zeros((n, h, w, pad16(7)), dtype=torch.bfloat16, device=DEV)
    f = torch.randn((n, h, w, 6), device=DEV, generator=g)
    x[..., :6] = (fall * f).bfloat16()
    x[..., 6] = (0.15 + 0.85 * torch.rand((n, 1, 1), device=DEV, generator=g)).bfloat16()
    t = fall * (0.5 * f.roll(1, 3) + 0.5 * torch.randn((n, h, w, 6), device=DEV, generator=g))
    return x, t.contiguous()


def _layer_input(case, seed):
    g = _rng(seed)
    n, h, w, ci, co = (case[k] for k in ("n", "h", "w", "cin", "cout"))

    def bf(*shape):
        return torch.randn(shape, device=DEV, generator=g).bfloat16()

    x = torch.relu(bf(n, h, w, ci))
    wt = bf(9, co, ci) * math.sqrt(2.0 / (9 * ci))
    bias = 0.05 * torch.randn(co, device=DEV, generator=g)
    dz = bf(n, h, w, co) * 0.01
    return x, wt, bias, dz


# ---- prepare and run ---------------------------------------------------------


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("flat", "gr"):
        sp = _flat_params(case) if kind == "flat" else _gr_params(case)
        env = SimEnvironment(sp, _np_type(case), DEV)
        data = SimData(env)
        dt = data.P.dev.dtype
        if kind == "gr":
            _fill(data, _wald_state(sp, seed, dt))
            solver = FieldSolverGREZ(data, env)
        else:
            _fill(data, _alfven_state(sp, seed, dt) if sp.problem == 0
                  else _pulsar_state(sp, seed, dt, _tiny(case)))
            solver = FieldSolverEZ(data, env)
        return dict(kind=kind, data=data, solver=solver, t=0.0, dt=sp.dt)
    if kind in ("sph1", "relax", "sweep"):
        runs = _sph_runs(case, seed)
        envs = [SimEnvironment(sp, _np_type(case), DEV) for sp, _ in runs]
        datas = [SimData(env) for env in envs]
        pools = [] if kind == "sph1" else [_pool([datas[i] for i in m]) for m in _groups(runs)]
        for data, (sp, s) in zip(datas, runs):
            _fill(data, _magnetosphere(sp, s, data.P.dev.dtype))
        if kind == "sph1":
            return dict(kind=kind, data=datas[0], solver=FieldSolverEZSpherical(datas[0], envs[0]),
                        t=0.0, dt=runs[0][0].dt)
        batch = SphBatch(envs, datas, nsteps=[0] * len(envs))
        if kind == "sweep":
            batch.autotune(trials=3)
        batch.use_graph(True)
        return dict(kind=kind, pools=pools, batch=batch, steps=case.get("steps", 1),
                    radii=[1.5 / sp.omega for sp, _ in runs])
    if kind == "layer":
        x, w, b, dz = _layer_input(case, seed)
        n, h, wd, ci, co = (case[k] for k in ("n", "h", "w", "cin", "cout"))
        pix = n * h * wd
        nsplit = max(1, min(256, pix // 512))
        return dict(kind=kind, shape=(n, h, wd, ci, co), x=x, w=w, wt=w.transpose(1, 2).contiguous(),
                    b=b, dz=dz, nsplit=nsplit,
                    y=torch.empty((n, h, wd, co), dtype=torch.bfloat16, device=DEV),
                    dx=torch.empty((n, h, wd, ci), dtype=torch.bfloat16, device=DEV),
                    part=torch.empty(nsplit * 9 * ci * co, device=DEV),
                    dw=torch.empty((9, co, ci), device=DEV), db=torch.empty(co, device=DEV))
    net = UNet(case["levels"], case["base"], 7, 6, device=DEV)
    net.set_params(_net_params(case, seed))
    x, t = _net_input(case, seed)
    return dict(kind=kind, net=net, x=x.view(torch.int16).view(-1), target=t.view(-1),
                shape=(case["n"], case["h"], case["w"]))


def run(state):
    kind = state["kind"]
    if kind in ("flat", "gr", "sph1"):
        state["solver"].evolve_fields(state["t"])
        state["t"] += state["dt"]
        return [a.dev for a in state["data"].state_arrays()]
    if kind in ("relax", "sweep"):
        state["batch"].step(state["steps"])
        if kind == "relax":
            return state["pools"] + [state["batch"].luminosity(state["radii"])]
        return state["pools"]
    if kind == "layer":
        L = _lib.load()
        s = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
        n, h, w, ci, co = state["shape"]
        p = {k: v.data_ptr() for k, v in state.items() if isinstance(v, torch.Tensor)}
        _lib.check(L.coffee_unet_conv3x3(p["x"], p["w"], p["b"], p["y"], None, n, h, w, ci, co, 0, 1, s))
        _lib.check(L.coffee_unet_conv3x3_wgrad(p["x"], p["dz"], p["part"], state["nsplit"], p["dw"],
                                               p["db"], n, h, w, ci, co, s))
        _lib.check(L.coffee_unet_conv3x3(p["dz"], p["wt"], None, p["dx"], None, n, h, w, co, ci, 1, 0, s))
        return [state["y"], state["dw"], state["db"], state["dx"]]
    net, (n, h, w) = state["net"], state["shape"]
    out = net.forward(state["x"], n, h, w)
    if kind == "predict":
        return out.view(n, h, w, -1)[..., :6]
    loss, dout = net.loss_and_grad(out, state["target"], n, h, w)
    net.backward(dout)
    net.adam_step(lr=1e-3)
    return {"out": out.view(n, h, w, -1)[..., :6], "loss": loss,
            "layers": [[P[k] for k in ("gw", "gb", "w")] for P in net.params.values()]}


# ---- the same work in FP64 with plain torch ----------------------------------

LSRK_A = (0.0, -0.4178904745, -1.192151694643, -1.697784692471, -1.514183444257)
LSRK_B = (0.1496590219993, 0.3792103129999, 0.8229550293869, 0.6994504559488, 0.1530572479681)
LSRK_C = (0.0, 0.1496590219993, 0.3704009573644, 0.6222557631345, 0.9582821306784)


def _tiny(case):
    return 1e-11 if case.get("f64") else 1e-7


def _cross(a, b):
    return [a[1] * b[2] - a[2] * b[1], a[2] * b[0] - a[0] * b[2], a[0] * b[1] - a[1] * b[0]]


def _dot(a, b):
    return a[0] * b[0] + a[1] * b[1] + a[2] * b[2]


class _Box:
    """Interior views and stencils of guarded arrays whose last dimensions are
    (z,) y, x."""

    def __init__(self, sp, nax):
        self.n, self.g, self.nax = sp.N, sp.guard, nax
        self.delta = [sp.size[a] / sp.N[a] for a in range(nax)]

    def at(self, f, ax=0, d=0):
        idx = [slice(None)] * f.dim()
        for a in range(self.nax):
            o = self.g[a] + (d if a == ax else 0)
            if f.shape[f.dim() - 1 - a] > 1:
                idx[f.dim() - 1 - a] = slice(o, o + self.n[a])
        return f[tuple(idx)]

    def diff(self, f, ax):
        at = lambda d: self.at(f, ax, d)  # noqa: E731
        return (8.0 * (at(1) - at(-1)) + (at(-2) - at(2))) / (12.0 * self.delta[ax])

    def delta6(self, f, ax):
        at = lambda d: self.at(f, ax, d)  # noqa: E731
        return (at(-3) + at(3)) - 6.0 * (at(-2) + at(2)) + 15.0 * (at(-1) + at(1)) - 20.0 * at(0)

    def curl(self, v):
        d = self.diff
        return [d(v[2], 1) - d(v[1], 2), d(v[0], 2) - d(v[2], 0), d(v[1], 0) - d(v[0], 1)]

    def put(self, U, new, periodic):
        for f, v in zip(U, new):
            self.at(f).copy_(v)
            for a in range(self.nax):
                if periodic[a]:
                    dim, g, n = f.dim() - 1 - a, self.g[a], self.n[a]
                    f.narrow(dim, 0, g).copy_(f.narrow(dim, n, g))
                    f.narrow(dim, n + g, g).copy_(f.narrow(dim, g, g))


def _project(D, B, lower, tiny):
    """Remove D.B, then cap D at B (metric norms)."""
    Bd = lower(B)
    B2 = torch.clamp(_dot(B, Bd), min=tiny)
    f = _dot(D, Bd) / B2
    D = [d - f * b for d, b in zip(D, B)]
    D2 = torch.clamp(_dot(D, lower(D)), min=tiny)
    s = torch.where(D2 > B2, torch.sqrt(B2 / D2), torch.ones_like(B2))
    return [s * d for d in D]


def _relax_to(U, Un, sig, tiny, background=None):
    """Absorbing layer: E, B toward their step-start values (B about a
    background) with the integrated damping factors."""
    on = sig > tiny
    sig = torch.where(on, sig, torch.ones_like(sig))
    e, f = torch.exp(-sig), -torch.expm1(-sig) / sig
    out = []
    for c in range(6):
        bg = background[c - 3] if background is not None and c >= 3 else 0.0
        out.append(torch.where(on, bg + e * (Un[c] - bg) + f * (U[c] - Un[c]), U[c]))
    return out + [U[6]]


def _lsrk_step(U, box, rhs, after, ko, periodic, t, dt):
    """One LSRK(5,4) step with the pointwise operations `after` each stage and
    the Kreiss-Oliger pass `ko`.  U: full arrays, changed in place."""
    Un = [box.at(f).clone() for f in U]
    dU = [torch.zeros_like(v) for v in Un]
    for s in range(5):
        k = rhs(U)
        dU = [LSRK_A[s] * a + b for a, b in zip(dU, k)]
        new = [box.at(f) + LSRK_B[s] * a for f, a in zip(U, dU)]
        new = after(new, t + LSRK_C[s] * dt, Un if s == 4 else None)
        box.put(U, new, periodic)
    box.put(U, after(ko(U), t + dt, None), periodic)


def _flat_exact(case, seed):
    sp, tiny = _flat_params(case), _tiny(case)
    dt_in = torch.float64 if case["f64"] else torch.float32
    U = (_alfven_state(sp, seed, dt_in) if sp.problem == 0 else _pulsar_state(sp, seed, dt_in, tiny))
    U = [u.double() for u in U]
    box = _Box(sp, 3)
    x, y, z = [box.at(p) for p in _axes(sp)]
    # the cleaning mask is taken at positions shifted by the vector lane of the
    # reference's CPU build (8 doubles or 16 floats per vector)
    lanes = 8 if case["f64"] else 16
    lane = (torch.arange(sp.N[0], device=DEV) % lanes).double().view(1, 1, -1)
    d = box.delta
    r = torch.sqrt(x * x + (y + lane * d[1]) ** 2 + (z + lane * d[2]) ** 2)
    mask = 0.5 * (1.0 - torch.tanh((r - 3.0) * 2.0))
    del r

    def rhs(U):
        E, B, P = U[:3], U[3:6], U[6]
        rotE, rotB = box.curl(E), box.curl(B)
        divE = sum(box.diff(E[a], a) for a in range(3))
        divB = sum(box.diff(B[a], a) for a in range(3))
        e, b, p = [box.at(f) for f in E], [box.at(f) for f in B], box.at(P)
        B2 = torch.clamp(_dot(b, b), min=tiny)
        Jp = _dot(b, rotB) - _dot(e, rotE)
        exb = _cross(e, b)
        out = [sp.dt * (rotB[a] - (divE * exb[a] + Jp * b[a]) / B2) for a in range(3)]
        out += [-sp.dt * (rotE[a] + mask * box.diff(P, a)) for a in range(3)]
        return out + [-p / sp.tau - sp.dt * sp.ch2 * divB]

    star = sp.problem == 1
    if star:
        r2 = torch.clamp(x * x + y * y + z * z, min=tiny)
        r = torch.sqrt(r2)
        blend = lambda r0, w: 0.5 * (1.0 - torch.tanh((r - r0) / w))  # noqa: E731
        s_b = blend(sp.radius - 4.0 * d[0], 0.5 * d[0])
        s_perp, s_par = blend(sp.radius, 0.25 * d[0]), blend(sp.radius, 0.5 * d[0])
        bg = [box.at(v) for v in _multipole(sp, *_axes(sp), 0.0, tiny)]
        sig = torch.zeros_like(r)
        for a, p in enumerate((x, y, z)):
            lo, hi = sp.lower[a] + sp.pml[a] * d[a], sp.lower[a] + sp.size[a] - sp.pml[a] * d[a]
            depth = torch.clamp(p - hi, min=0.0) + torch.clamp(lo - p, min=0.0)
            sig = sig + sp.sigpml * (depth / (sp.pmllen * d[a])) ** 3

    def rotate(U, t):
        bn = _multipole(sp, x, y, z, sp.omega * t, tiny)
        b = [s_b * n + (1.0 - s_b) * v for n, v in zip(bn, U[3:6])]
        near = r < 1.5 * sp.radius
        b = [torch.where(near, n, v) for n, v in zip(b, U[3:6])]
        vx, vy = -sp.omega * y, sp.omega * x
        en = [-vy * b[2], vx * b[2], vy * b[0] - vx * b[1]]
        pos = (x, y, z)
        en_r, e_r = _dot(en, pos) / r2, _dot(U[:3], pos) / r2
        e = [s_perp * en_r * p + (1.0 - s_perp) * e_r * p + s_par * (n - en_r * p)
             + (1.0 - s_par) * (v - e_r * p) for p, n, v in zip(pos, en, U[:3])]
        core = r < 0.5 * sp.radius
        e = [torch.where(core, n, torch.where(near, q, v)) for n, q, v in zip(en, e, U[:3])]
        b = [torch.where(core, n, q) for n, q in zip(bn, b)]
        return e + b + [U[6]]

    def after(U, t, Un):
        U = _project(U[:3], U[3:6], lambda v: v, tiny) + list(U[3:])
        if star:
            U = rotate(U, t)
            if Un is not None:
                U = _relax_to(U, Un, sig, tiny, bg)
        return U

    def ko(U):
        return [box.at(f) + sp.KOeps / 64.0 * sum(box.delta6(f, a) for a in range(3))
                for f in U[:6]] + [box.at(U[6])]

    _lsrk_step(U, box, rhs, after, ko, sp.periodic_boundary, 0.0, sp.dt)
    return U


def _gr_exact(case, seed):
    sp, tiny = _gr_params(case), _tiny(case)
    U = [u.double() for u in _wald_state(sp, seed, torch.float64 if case["f64"] else torch.float32)]
    box = _Box(sp, 3)
    x, y, z = _axes(sp)
    r, s, bu, l = _cks(sp.a, x, y, z)
    sg = torch.sqrt(1.0 + s)
    ri, si, bui, sgi = (box.at(v) for v in (r, s, bu, sg))
    li = [box.at(v) for v in l]
    weight = 0.5 * (1.0 - torch.tanh(ri - 5.0))
    del r

    def lower(v):
        f = si * _dot(li, v)
        return [v[a] + f * li[a] for a in range(3)]

    def rhs(U):
        D, B, P = U[:3], U[3:6], U[6]
        lD, lB = s * _dot(l, D), s * _dot(l, B)
        cB, cD = _cross(l, B), _cross(l, D)
        E = [(D[a] + lD * l[a]) / sg + sg * bu * cB[a] for a in range(3)]
        H = [(B[a] + lB * l[a]) / sg - sg * bu * cD[a] for a in range(3)]
        del lD, lB, cB, cD
        rotE = [v / sgi for v in box.curl(E)]
        rotH = [v / sgi for v in box.curl(H)]
        ei = [box.at(v) for v in E]
        del H
        divD = sum(box.diff(sg * D[a], a) for a in range(3)) / sgi
        divB = sum(box.diff(sg * B[a], a) for a in range(3)) / sgi
        Di, Bi, p = [box.at(v) for v in D], [box.at(v) for v in B], box.at(P)
        Bd, Dd = lower(Bi), lower(Di)
        B2 = torch.clamp(_dot(Bi, Bd), min=tiny)
        Jp = _dot(Bd, rotH) - _dot(Dd, rotE)
        exb = _cross(ei, Bd)
        gP = [box.diff(P, a) for a in range(3)]
        lP = bui * _dot(li, gP)
        out = [sp.dt * (rotH[a] - (divD * exb[a] / sgi + Jp * Bi[a]) / B2) for a in range(3)]
        out += [sp.dt * (-rotE[a] + weight * (-(gP[a] - lP * li[a]) / sgi + bui * li[a] * divB))
                for a in range(3)]
        return out + [sp.dt * (-divB / sgi + lP) - p / sgi / sp.tau]

    xi, yi, zi = (box.at(v) for v in (x, y, z))
    sig = torch.zeros_like(ri)
    d = box.delta
    for a, pos in enumerate((xi, yi, zi)):
        lo, hi = sp.lower[a] + sp.pml[a] * d[a], sp.lower[a] + sp.size[a] - sp.pml[a] * d[a]
        depth = torch.clamp(pos - hi, min=0.0) + torch.clamp(lo - pos, min=0.0)
        sig = sig + sp.sigpml * (depth / (sp.pmllen * d[0])) ** 3
    r_h = 1.0 + math.sqrt(1.0 - sp.a * sp.a)
    sig_in = sp.sigpml * sp.dt * (torch.clamp(0.7 * r_h - ri, min=0.0) / (0.2 * r_h)) ** 3

    def after(U, t, Un):
        U = _project(U[:3], U[3:6], lower, tiny) + list(U[3:])
        if Un is not None:
            U = _relax_to(_relax_to(U, Un, sig, tiny), Un, sig_in, tiny)
            U = [torch.where(ri < 0.01 * r_h, torch.zeros_like(v), v) for v in U[:6]] + [U[6]]
        return U

    def ko(U):
        return [box.at(f) + sp.KOeps / 64.0 * sum(box.delta6(f, a) for a in range(3)) for f in U]

    _lsrk_step(U, box, rhs, after, ko, sp.periodic_boundary, 0.0, sp.dt)
    return U


def _sph_evolve(params, U, steps, tiny):
    """Runs of one grid together: U holds 7 tensors (run, theta, r)."""
    sp = params[0]
    box = _Box(sp, 2)
    x, y, _ = _axes(sp)
    r, sn = torch.exp(x), torch.sin(y)
    sqg = r ** 3 * torch.abs(sn)
    gm = torch.clamp(box.at(sqg), min=tiny)
    low = [r * r, r * r, (r * sn) ** 2]
    low_i = [torch.broadcast_to(box.at(v), gm.shape) for v in low]
    ri, th = box.at(r), box.at(y)
    omega = torch.tensor([p.omega for p in params], dtype=torch.float64, device=DEV).view(-1, 1, 1)
    d = box.delta

    def lower(v):
        return [low_i[a] * v[a] for a in range(3)]

    def curl(v):
        w = [low[a] * v[a] for a in range(3)]
        return [box.diff(w[2], 1) / gm, -box.diff(w[2], 0) / gm,
                (box.diff(w[1], 0) - box.diff(w[0], 1)) / gm]

    def rhs(U):
        E, B, P = U[:3], U[3:6], U[6]
        rotE, rotB = curl(E), curl(B)
        div = lambda v: (box.diff(sqg * v[0], 0) + box.diff(sqg * v[1], 1)) / gm  # noqa: E731
        e, b, p = [box.at(v) for v in E], [box.at(v) for v in B], box.at(P)
        el, bl = lower(e), lower(b)
        B2 = torch.clamp(_dot(b, bl), min=tiny)
        Jp = _dot(bl, rotB) - _dot(el, rotE)
        exb = _cross(el, bl)
        a = div(E) / gm
        out = [sp.dt * (rotB[c] - (a * exb[c] + Jp * b[c]) / B2) for c in range(3)]
        gP = [box.diff(P, 0) / (ri * ri), box.diff(P, 1) / (ri * ri), 0.0]
        out += [-sp.dt * (rotE[c] + gP[c]) for c in range(3)]
        return out + [-sp.dt * sp.ch2 * div(B) - p / sp.tau]

    # rotating conductor: r < R + dx (all of it inside R, the surface row partly)
    surf = torch.abs(ri - sp.radius) < 0.5 * d[0]
    inside = (ri < sp.radius - tiny) & ~surf
    bxn, byn = 2.0 * sp.b0 * torch.cos(th) / ri ** 3, sp.b0 * torch.sin(th) / ri ** 3
    v3 = omega * ri * torch.sin(th)
    star = [(inside, v3 * byn / ri), (surf | inside, -v3 * bxn / ri), (surf | inside, None),
            (surf | inside, bxn / ri), (inside, byn / ri), (inside, None)]
    xh = sp.lower[0] + sp.size[0] - sp.pml[0] * d[0]
    sig = sp.sigpml * (torch.clamp(ri - math.exp(xh), min=0.0) / sp.pmllen) ** 3

    def after(U, t, Un):
        U = _project(U[:3], U[3:6], lower, tiny) + list(U[3:])
        U = [torch.where(m, torch.zeros_like(u) if v is None else torch.broadcast_to(v, u.shape), u)
             for (m, v), u in zip(star, U[:6])] + [U[6]]
        return _relax_to(U, Un, torch.broadcast_to(sig, U[0].shape), tiny) if Un is not None else U

    def axis(U):
        g0, n0 = box.g[0], box.n[0]
        for j, dr in ((box.g[1], 1), (box.g[1] + box.n[1], -1)):
            V = [u.narrow(2, g0, n0) for u in U]
            for c in range(7):
                V[c][:, j] = V[c][:, j + dr] if c in (0, 3, 6) else 0.0
                for k in (1, 2, 3):
                    if c < 6:
                        V[c][:, j - dr * k] = V[c][:, j + dr * k] * (1.0 if c in (0, 3) else -1.0)

    class WithAxis(_Box):
        def put(self, U, new, periodic):
            super().put(U, new, periodic)
            axis(U)

    axbox = WithAxis(sp, 2)
    w = sqg if sp.KO_geometry else torch.ones_like(sqg)
    iw = 1.0 / gm if sp.KO_geometry else torch.ones_like(gm)

    def ko(U):
        return [box.at(f) + sp.KOeps / 64.0 * iw * (box.delta6(w * f, 0) + box.delta6(w * f, 1))
                for f in U]

    axis(U)
    for n in range(steps):
        _lsrk_step(U, axbox, rhs, after, ko, [False] * 3, n * sp.dt, sp.dt)


def _luminosity(sp, U, b, radius):
    g0, g1, n0, n1 = sp.guard[0], sp.guard[1], sp.N[0], sp.N[1]
    dx, dy = sp.size[0] / n0, sp.size[1] / n1
    f = (math.log(radius) - sp.lower[0]) / dx + g0
    i0 = min(max(int(math.floor(f)), g0), g0 + n0 - 2)
    w = min(max(f - i0, 0.0), 1.0)
    sn = torch.sin(dy * torch.arange(n1, dtype=torch.float64, device=DEV))
    tot = 0.0
    for i, wi in ((i0, 1.0 - w), (i0 + 1, w)):
        r = math.exp(sp.lower[0] + dx * (i - g0))
        v = [U[c][b, g1:g1 + n1, i] for c in (1, 2, 4, 5)]
        flux = r * v[0] * r * sn * v[3] - r * sn * v[1] * r * v[2]
        tot += wi * r * r * float((flux * sn).sum())
    return 2.0 * math.pi * tot * dy


def _sph_exact(case, seed):
    runs = _sph_runs(case, seed)
    dt_in = torch.float64 if case.get("f64") else torch.float32
    pools, lum = [], np.zeros(len(runs))
    for members in _groups(runs):
        states = [_magnetosphere(runs[i][0], runs[i][1], dt_in) for i in members]
        U = [torch.cat([s[c] for s in states]).double() for c in range(7)]
        _sph_evolve([runs[i][0] for i in members], U, case.get("steps", 1), _tiny(case))
        if case["kind"] == "sph1":
            return U
        if case["kind"] == "relax":
            for b, i in enumerate(members):
                lum[i] = _luminosity(runs[i][0], U, b, 1.5 / runs[i][0].omega)
        cells = U[0][0].numel()
        pool = torch.zeros((len(members), 7, (cells + 63) // 64 * 64), dtype=torch.float64, device=DEV)
        for c in range(7):
            pool[:, c, :cells] = U[c].reshape(len(members), cells)
        pools.append(pool)
    return pools + [lum] if case["kind"] == "relax" else pools


def _conv(x, w, b):
    """3x3 convolution, zero padding: x (n, h, w, ci), w (9, co, ci)."""
    n, h, wd, ci = x.shape
    xp = torch.nn.functional.pad(x, (0, 0, 1, 1, 1, 1))
    out = None
    for k in range(9):
        t = xp[:, k // 3:k // 3 + h, k % 3:k % 3 + wd].reshape(-1, ci) @ w[k].t()
        out = t if out is None else out + t
    out = out.view(n, h, wd, -1)
    return out if b is None else out + b


def _layer_exact(case, seed):
    x, w, b, dz = (v.double() for v in _layer_input(case, seed))
    x.requires_grad_(True)
    w.requires_grad_(True)
    z = _conv(x, w, b)
    z.backward(dz)
    return [torch.relu(z.detach()), w.grad, dz.sum(dim=(0, 1, 2)), x.grad]


def _net_exact(case, seed):
    W = {}
    for name, (w, b) in _net_params(case, seed).items():
        w = torch.from_numpy(w.astype(np.float64)).to(DEV).reshape(9, w.shape[2], w.shape[3])
        W[name] = (w.transpose(1, 2).contiguous().requires_grad_(True),
                   torch.from_numpy(b.astype(np.float64)).to(DEV).requires_grad_(True))
    x, target = _net_input(case, seed)
    h = x[..., :7].double()
    relu, skips = torch.relu, []
    for l in range(case["levels"]):
        if l:
            n, hh, ww, c = h.shape
            h = h.view(n, hh // 2, 2, ww // 2, 2, c).mean(dim=(2, 4))
        h = relu(_conv(relu(_conv(h, *W[f"enc{l}a"])), *W[f"enc{l}b"]))
        skips.append(h)
    for l in range(case["levels"] - 2, -1, -1):
        h = h.repeat_interleave(2, 1).repeat_interleave(2, 2)
        h = torch.cat([relu(_conv(h, *W[f"dec{l}up"])), skips[l]], dim=3)
        h = relu(_conv(relu(_conv(h, *W[f"dec{l}a"])), *W[f"dec{l}b"]))
    out = _conv(h, *W["head"])
    if case["kind"] == "predict":
        return out.detach()
    loss = ((out - target.double()) ** 2).mean()
    loss.backward()
    layers = []
    for name, ci, co, _ in layer_specs(case["levels"], case["base"], 7, 6):
        w, b = W[name]

        def pad(v):
            full = torch.zeros((9, pad16(co), pad16(ci)) if v.dim() == 3 else (pad16(co),),
                               dtype=torch.float64, device=DEV)
            if v.dim() == 3:
                full[:, :co, :ci] = v
            else:
                full[:co] = v
            return full

        step = lambda p: p.detach() - 1e-3 * p.grad / (p.grad.abs() + 1e-8)  # noqa: E731
        layers.append([pad(w.grad), pad(b.grad), pad(step(w))])
    return {"out": out.detach(), "loss": float(loss.detach()), "layers": layers}


def exact(case, seed):
    kind = case["kind"]
    if kind == "flat":
        return _flat_exact(case, seed)
    if kind == "gr":
        return _gr_exact(case, seed)
    if kind in ("sph1", "relax", "sweep"):
        return _sph_exact(case, seed)
    if kind == "layer":
        return _layer_exact(case, seed)
    with torch.enable_grad():
        return _net_exact(case, seed)
