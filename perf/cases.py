"""Performance cases: the work a user of this framework has it do, through its public entry points.

A case is a dict of plain values; ``prepare`` builds what a program has in hand before the call, ``run`` is one pass,
``work`` the bytes and operations a pass cannot do without, and ``exact`` the same outputs from plain torch in 64
bits.  The kinds:

* ``loop``     a program's own time loop over ``create_lb_function`` kernels (bench.py, lbmpy's tests): one EVEN / ODD
               pair of an in-place pattern, or two pull steps.
* ``step``     ``LatticeBoltzmannStep.run`` on the scenarios (cavity, duct, obstacles, periodic box): a number of time
               steps, then density and velocity on the host, as every lbmpy script does between two looks at its flow.
* ``ensemble`` ``BatchedSweep.run`` on many small channels, each with its own size, force and viscosity.
* ``closure``  the sweep with the learned closure in place of the shear rate.
* ``train``    ``ClosureModel.train``: one epoch of the closure's training on minibatches.
* ``analyse``  what a program asks of a field between time steps: conserved sums, the check for NaN, density and
               velocity.
"""
import math

import numpy as np
import torch

# the directions of D3Q27 in lbmpy's 'walberla' order; D3Q19 is its first 19, D2Q9 its plane z = 0
C27 = ((0, 0, 0), (0, 1, 0), (0, -1, 0), (-1, 0, 0), (1, 0, 0), (0, 0, 1), (0, 0, -1), (-1, 1, 0), (1, 1, 0),
       (-1, -1, 0), (1, -1, 0), (0, 1, 1), (0, -1, 1), (-1, 0, 1), (1, 0, 1), (0, 1, -1), (0, -1, -1), (-1, 0, -1),
       (1, 0, -1), (1, 1, 1), (-1, 1, 1), (1, -1, 1), (-1, -1, 1), (1, 1, -1), (-1, 1, -1), (1, -1, -1), (-1, -1, -1))
DIRECTIONS = {"D2Q9": tuple(c[:2] for c in C27 if c[2] == 0), "D3Q19": C27[:19], "D3Q27": C27}
ITEM = {"float64": 8, "float32": 4, "float16": 2}
# rough operations of one cell's collision, for the operation floor
CELL_FLOPS = {("D2Q9", "srt"): 150, ("D2Q9", "trt"): 180, ("D3Q19", "srt"): 300, ("D3Q19", "trt"): 350,
              ("D3Q19", "mrt"): 450, ("D3Q27", "srt"): 450, ("D3Q27", "cumulant"): 700}


def listed():
    return [
        # the headline: the Taylor-Green vortex of bench.py, in FP32 and (ragged, no power of two) in FP16 storage
        dict(name="loop_cumulant_f32_256", kind="loop", stencil="D3Q27", method="cumulant", pattern="aa",
             dtype="float32", nx=256, ny=256, nz=256, walls=False, force=0.0, omega=1.98),
        dict(name="loop_cumulant_f16_250x200x180", kind="loop", stencil="D3Q27", method="cumulant", pattern="aa",
             dtype="float16", nx=250, ny=200, nz=180, walls=False, force=0.0, omega=1.95),
        # double precision (lbmpy's default type) on an odd box
        dict(name="loop_cumulant_f64_131x117x101", kind="loop", stencil="D3Q27", method="cumulant", pattern="aa",
             dtype="float64", nx=131, ny=117, nz=101, walls=False, force=0.0, omega=1.9),
        # the MRT channel of bench.py, the largest domain: walls, a body force, two arrays
        dict(name="loop_channel_mrt_f32_512x256x256", kind="loop", stencil="D3Q19", method="mrt", pattern="pull",
             dtype="float32", nx=512, ny=256, nz=256, walls=True, force=1e-6, omega=1.8),
        # the smallest calls: lbmpy's 2-D cavity in double precision, where launches and latency count
        dict(name="step_cavity_d2q9_f64_40x80", kind="step", scenario="cavity", stencil="D2Q9", method="srt",
             pattern="pull", dtype="float64", nx=40, ny=80, nz=1, steps=100, force=0.0, omega=1.8),
        # the force-driven duct of lbmpy's quick tests, at its size
        dict(name="step_duct_srt_f64_64x32x32", kind="step", scenario="duct", stencil="D3Q19", method="srt",
             pattern="pull", dtype="float64", nx=64, ny=32, nz=32, steps=100, force=1e-6, omega=1.7),
        # a medium cavity in place, in FP32
        dict(name="step_cavity_trt_f32_96", kind="step", scenario="cavity", stencil="D3Q19", method="trt",
             pattern="aa", dtype="float32", nx=96, ny=96, nz=96, steps=50, force=0.0, omega=1.8),
        # flow through a box of spheres (index-list walls inside the domain), sizes no multiple of a wavefront
        dict(name="step_spheres_trt_f32_150x90x75", kind="step", scenario="spheres", stencil="D3Q19", method="trt",
             pattern="pull", dtype="float32", nx=150, ny=90, nz=75, steps=40, force=1e-6, omega=1.6),
        # the ensemble of bench.py: channels of 32..96 cells a side
        dict(name="ensemble_48_trt_f32", kind="ensemble", members=48, low=32, high=96, sizes=2024, steps=10,
             dtype="float32"),
        # the learned closure's coarse run, and its training
        dict(name="closure_cumulant_f32_128", kind="closure", dtype="float32", nx=128, ny=128, nz=128, omega=1.99),
        dict(name="train_closure_1m", kind="train", samples=1 << 20, batch=65536),
        # looking at a field between time steps
        dict(name="analyse_trt_f32_192x160x144", kind="analyse", stencil="D3Q19", dtype="float32", nx=192, ny=160,
             nz=144, omega=1.8),
    ]


def _spread(rng, lo, hi):
    """A whole number of lo..hi, spread over its logarithm; every third or so rounded to 16."""
    v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    return max(lo, v // 16 * 16) if rng.random() < 0.33 and v >= 32 else v


def draw(rng):
    kind = rng.choice(["loop", "loop", "loop", "step", "step", "step", "ensemble", "closure", "train", "analyse"])
    if kind == "loop":
        stencil, method = rng.choice([("D3Q27", "cumulant"), ("D3Q27", "cumulant"), ("D3Q19", "srt"),
                                      ("D3Q19", "trt"), ("D3Q19", "mrt"), ("D3Q27", "srt")])
        walls = method != "cumulant" and rng.random() < 0.5
        pattern = rng.choice(["aa", "aa", "pull"] if walls else ["aa", "aa", "pull", "esotwist"])
        dtype = rng.choice(["float32", "float32", "float64", "float16"])
        force = 0.0 if method == "cumulant" or dtype == "float16" else rng.choice([0.0, 1e-6])
        c = dict(kind=kind, stencil=stencil, method=method, pattern=pattern, dtype=dtype, nx=_spread(rng, 24, 600),
                 ny=_spread(rng, 24, 300), nz=_spread(rng, 24, 300), walls=walls, force=force,
                 omega=round(rng.uniform(1.5, 1.98), 4))
        while _sweep_bytes(c) > 10.1e9:
            c["nz"] = max(1, c["nz"] // 2)
        return c
    if kind == "step":
        scenario = rng.choice(["cavity", "duct", "spheres", "periodic", "cavity2d"])
        c = dict(kind=kind, scenario=scenario, stencil="D3Q19", method=rng.choice(["srt", "trt"]),
                 pattern=rng.choice(["pull", "aa"]), dtype=rng.choice(["float64", "float32"]),
                 nx=_spread(rng, 16, 180), ny=_spread(rng, 16, 140), nz=_spread(rng, 16, 140),
                 steps=2 * _spread(rng, 5, 60), force=0.0, omega=round(rng.uniform(1.5, 1.9), 4))
        if scenario == "cavity2d":
            c.update(scenario="cavity", stencil="D2Q9", nz=1, nx=_spread(rng, 16, 1200), ny=_spread(rng, 16, 1200))
        elif scenario == "duct":
            c["force"] = 1e-6
        elif scenario == "spheres":
            c.update(force=1e-6, pattern="pull", nx=max(40, c["nx"]), ny=max(40, c["ny"]), nz=max(40, c["nz"]))
        elif scenario == "periodic":
            c.update(stencil="D3Q27", method="cumulant")
        return c
    if kind == "ensemble":
        return dict(kind=kind, members=rng.randint(8, 56), low=rng.choice([16, 24, 32]), high=rng.choice([64, 80, 96]),
                    sizes=rng.randrange(1 << 20), steps=2 * rng.randint(2, 8), dtype=rng.choice(["float32", "float64"]))
    if kind == "closure":
        return dict(kind=kind, dtype="float32", nx=64 * rng.randint(1, 3), ny=_spread(rng, 32, 192),
                    nz=_spread(rng, 32, 192), omega=round(rng.uniform(1.9, 1.99), 4))
    if kind == "train":
        return dict(kind=kind, samples=_spread(rng, 1 << 16, 1 << 21), batch=rng.choice([16384, 65536, 131072]))
    return dict(kind=kind, stencil=rng.choice(["D3Q19", "D3Q27"]), dtype=rng.choice(["float32", "float64", "float16"]),
                nx=_spread(rng, 32, 256), ny=_spread(rng, 32, 200), nz=_spread(rng, 32, 200), omega=1.8)


# ---------------------------------------------------------------------- the least work
def _cells(c):
    return c["nx"] * c["ny"] * c["nz"]


def _q(stencil):
    return len(DIRECTIONS[stencil])


def _sweep_bytes(c, steps=2):
    return 2 * _q(c["stencil"]) * ITEM[c["dtype"]] * _cells(c) * steps


def work(case):
    kind = case["kind"]
    if kind == "loop":                 # two calls: each reads and writes every population once
        return {"bytes": _sweep_bytes(case), "flops": 2 * _cells(case) * CELL_FLOPS[case["stencil"], case["method"]]}
    if kind == "step":                 # one call: populations in and out once, density and velocity (FP64) out
        d = len(DIRECTIONS[case["stencil"]][0])
        return {"bytes": _sweep_bytes(case, 1) + 8 * (1 + d) * _cells(case),
                "flops": case["steps"] * _cells(case) * CELL_FLOPS[case["stencil"], case["method"]]}
    if kind == "ensemble":             # one call, too
        n = sum(x * y * z for (x, y, z), _, _ in _members(case))
        return {"bytes": 2 * 19 * ITEM[case["dtype"]] * n, "flops": case["steps"] * n * CELL_FLOPS["D3Q19", "trt"]}
    if kind == "closure":
        n = _cells(case)
        return {"bytes": 2 * 2 * 27 * 4 * n, "flops": 2 * n * (CELL_FLOPS["D3Q27", "cumulant"] + 2 * (10 * 32 + 32 * 32 + 32))}
    if kind == "train":                # every sample's features and target once; forward, backward, weight gradients
        return {"bytes": 44 * case["samples"], "flops": case["samples"] * 6 * (10 * 32 + 32 * 32 + 32)}
    n = _cells(case)                   # analyse: three questions, each reads the field; density and velocity out
    q = _q(case["stencil"])
    return {"bytes": 3 * q * ITEM[case["dtype"]] * n + 16 * n, "flops": 6 * q * n}


# ---------------------------------------------------------------------- initial states
def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _flow(shape, seed, amplitude=0.03):
    """A smooth periodic flow of a few random waves: (density, velocity (D, [z,] y, x)) in 64 bits."""
    g = np.random.default_rng(seed)
    dim = len(shape)
    rev = shape[::-1]
    u = torch.zeros((dim,) + tuple(rev), dtype=torch.float64, device=_device())
    rho = torch.ones(tuple(rev), dtype=torch.float64, device=_device())
    for _ in range(3):
        k = g.integers(1, 3, size=dim)
        ph = g.uniform(0, 2 * np.pi, size=dim)
        a = g.normal(size=dim)
        waves = []
        for ax in range(dim):                      # axis ax is tensor axis dim - 1 - ax
            t = (torch.arange(shape[ax], dtype=torch.float64, device=_device()) + 0.5) * (2 * np.pi * int(k[ax]) / shape[ax])
            view = [1] * dim
            view[dim - 1 - ax] = shape[ax]
            waves.append((t + float(ph[ax])).view(view))
        s = torch.sin(sum(waves[1:], waves[0]))
        for ax in range(dim):
            u[ax] += amplitude / 3 * float(a[ax]) * s
        rho += 0.05 * amplitude * float(g.normal()) * s
    return rho, u


def _weights(stencil):
    table = {"D2Q9": (4 / 9, 1 / 9, 1 / 36), "D3Q19": (1 / 3, 1 / 18, 1 / 36), "D3Q27": (8 / 27, 2 / 27, 1 / 54, 1 / 216)}[stencil]
    return [table[sum(abs(v) for v in c)] for c in DIRECTIONS[stencil]]


def _inverse(stencil):
    d = DIRECTIONS[stencil]
    return [d.index(tuple(-v for v in c)) for c in d]


def _equilibrium(stencil, method, rho, u):
    """Zero-centred equilibrium populations (Q, ...): the cumulant method's product form, or the second-order one
    (incompressible), which on D3Q19 has the moments x^2 y^2 of the continuous Maxwellian."""
    out = torch.empty((_q(stencil),) + tuple(rho.shape), dtype=torch.float64, device=rho.device)
    w = _weights(stencil)
    uu = (u * u).sum(0)
    for i, c in enumerate(DIRECTIONS[stencil]):
        if method == "cumulant":
            f = rho
            for a, e in enumerate(c):
                f = f * ((2 / 3 - u[a] * u[a]) if e == 0 else 0.5 * (1 / 3 + u[a] * u[a] + e * u[a]))
            out[i] = f - w[i]
        else:
            cu = sum(e * u[a] for a, e in enumerate(c))
            out[i] = w[i] * ((rho - 1) + 3 * cu + 4.5 * cu * cu - 1.5 * uu)
            if stencil == "D3Q19":
                along = sum(u[a] * u[a] for a, e in enumerate(c) if e) if any(c) else 0.0
                out[i] += (uu - along) * (1 / 6, -1 / 12, 1 / 24)[sum(abs(e) for e in c)]
    return out


def _initial(case, seed):
    """The populations at the start (Q, [z,] y, x) in the storage type, direction by direction."""
    shape = (case["nx"], case["ny"], case["nz"])
    rho, u = _flow(shape, seed)
    f = _equilibrium(case["stencil"], case["method"], rho, u)
    dtype = getattr(torch, case["dtype"])
    return f.to(dtype)


def _laid_out(f, stencil, pattern, back=False):
    """Populations in the slots where an even step of an in-place pattern leaves them (back: the reverse)."""
    if pattern == "pull":
        return f
    out = torch.empty_like(f)
    inv = _inverse(stencil)
    for i, c in enumerate(DIRECTIONS[stencil]):
        shift = [max(v, 0) if pattern == "esotwist" else 0 for v in c]
        dims = [f.dim() - 1 - a for a in range(len(c))]
        if back:
            out[i] = torch.roll(f[inv[i]], [-s for s in shift], [d - 1 for d in dims])
        else:
            out[inv[i]] = torch.roll(f[i], shift, [d - 1 for d in dims])
    return out


def _method_kwargs(case):
    from lbmpy_amd import LBStencil, Method, ForceModel
    m = {"cumulant": Method.CUMULANT, "srt": Method.SRT, "trt": Method.TRT, "mrt": Method.MRT}[case["method"]]
    kw = dict(stencil=LBStencil(case["stencil"]), method=m, relaxation_rate=case["omega"])
    if case["method"] == "cumulant":
        kw["compressible"] = True
    if case.get("force"):
        kw.update(force=(case["force"], 0.0, 0.0)[:len(DIRECTIONS[case["stencil"]][0])], force_model=ForceModel.GUO)
    return kw


def _compute(dtype):
    return "float64" if dtype == "float64" else "float32"


# ---------------------------------------------------------------------- preparing and running
def prepare(case, seed):
    return {"loop": _prepare_loop, "closure": _prepare_loop, "step": _prepare_step, "ensemble": _prepare_ensemble,
            "train": _prepare_train, "analyse": _prepare_analyse}[case["kind"]](case, seed)


def run(state):
    return state["run"](state)


def _as_loop(case):
    """A closure case as the loop it runs in."""
    if case["kind"] == "closure":
        return dict(case, stencil="D3Q27", method="cumulant", pattern="aa", walls=False, force=0.0)
    return case


def _prepare_loop(case, seed):
    from lbmpy_amd import LBMConfig, CreateKernelConfig, Target, Timestep, create_lb_function
    from lbmpy_amd.sweep import create_pdf_array
    c = _as_loop(case)
    config = CreateKernelConfig(target=Target.GPU, data_type=c["dtype"], compute_type=_compute(c["dtype"]),
                                ghost_layers=0)
    kw = dict(_method_kwargs(c), streaming_pattern=c["pattern"])
    if c["pattern"] == "pull":
        kernels = [create_lb_function(lbm_config=LBMConfig(**kw), config=config)]
    else:
        kernels = [create_lb_function(lbm_config=LBMConfig(**kw, timestep=t), config=config)
                   for t in (Timestep.ODD, Timestep.EVEN)]
    model = _closure_model(seed) if case["kind"] == "closure" else None
    for k in kernels:
        k.set_faces(["periodic", "noslip" if c["walls"] else "periodic", "periodic"])
        if model is not None:
            k.set_closure(model)
    size = (c["nx"], c["ny"], c["nz"])
    src = create_pdf_array(size, _q(c["stencil"]), ghost_layers=0, dtype=c["dtype"])
    src.permute(3, 2, 1, 0).copy_(_laid_out(_initial(c, seed), c["stencil"], c["pattern"]))
    dst = torch.zeros_like(src) if c["pattern"] == "pull" else None
    return dict(run=_run_loop, kernels=kernels, src=src, dst=dst, model=model)


def _run_loop(s):
    if s["dst"] is not None:
        k = s["kernels"][0]
        k(src=s["src"], dst=s["dst"])
        k(src=s["dst"], dst=s["src"])
    else:
        for k in s["kernels"]:
            k(src=s["src"])
    return {"pdf": s["src"]}


def _sphere_mask(case):
    """Cells (x, y, z; midpoints) inside one of a few spheres, the same for every seed."""
    n = np.array([case["nx"], case["ny"], case["nz"]], dtype=float)
    g = np.random.default_rng(7)
    centres = [n * g.uniform(0.3, 0.7, 3) for _ in range(4)]
    radius = 0.12 * n.min()

    def mask(x, y, z):
        m = np.zeros(np.broadcast(x, y, z).shape, dtype=bool)
        for p in centres:
            m |= (x - p[0]) ** 2 + (y - p[1]) ** 2 + (z - p[2]) ** 2 < radius ** 2
        return m
    return mask


def _prepare_step(case, seed):
    from lbmpy_amd import (LBMConfig, CreateKernelConfig, Target, create_channel, create_fully_periodic_flow,
                           create_lid_driven_cavity)
    from lbmpy_amd.boundaries import NoSlip
    dim = len(DIRECTIONS[case["stencil"]][0])
    size = (case["nx"], case["ny"], case["nz"])[:dim]
    kw = dict(_method_kwargs(case), streaming_pattern=case["pattern"])
    config = CreateKernelConfig(target=Target.GPU, data_type=case["dtype"], compute_type=_compute(case["dtype"]))
    _, u = _flow(size, seed, 0.01 if case["scenario"] != "periodic" else 0.03)
    u = u.permute(*range(dim, 0, -1), 0).cpu().numpy()
    if case["scenario"] == "cavity":
        step = create_lid_driven_cavity(domain_size=size, lid_velocity=0.01, lbm_config=LBMConfig(**kw), config=config)
    elif case["scenario"] == "periodic":
        step = create_fully_periodic_flow(u, lbm_config=LBMConfig(**kw), config=config)
    else:
        force = kw.pop("force")[0]
        step = create_channel(domain_size=size, force=force, duct=True, config=config, **kw)
        if case["scenario"] == "spheres":
            step.boundary_handling.set_boundary(NoSlip("obstacle"), mask_callback=_sphere_mask(case))
    step.velocity[...][...] = u
    step.set_pdf_fields_from_macroscopic_values()
    return dict(run=_run_step, step=step, steps=case["steps"], dim=dim)


def _run_step(s):
    s["step"].run(s["steps"])
    inner = (slice(1, -1),) * s["dim"]
    return {"pdf": s["step"].pdf_array[inner], "density": s["step"].density[...], "velocity": s["step"].velocity[...]}


def _members(case):
    """((nx, ny, nz), force, omega) of each channel of an ensemble, from the case alone."""
    g = np.random.default_rng(case["sizes"])
    sizes = np.arange(case["low"], case["high"] + 1, 8)
    return [(tuple(int(v) for v in g.choice(sizes, 3)), float(np.exp(g.uniform(np.log(1e-7), np.log(1e-5)))),
             float(g.uniform(1.5, 1.95))) for _ in range(case["members"])]


def _member_case(case, shape, force, omega):
    return dict(stencil="D3Q19", method="trt", dtype=case["dtype"], nx=shape[0], ny=shape[1], nz=shape[2], walls=True,
                force=force, omega=omega, pattern="pull")


def _prepare_ensemble(case, seed):
    from lbmpy_amd import LBMConfig, CreateKernelConfig, Target, create_lb_function
    from lbmpy_amd.batch import BatchedSweep
    from lbmpy_amd.sweep import create_pdf_array
    config = CreateKernelConfig(target=Target.GPU, data_type=case["dtype"], ghost_layers=0)
    kernels, src, dst = [], [], []
    for n, (shape, force, omega) in enumerate(_members(case)):
        c = _member_case(case, shape, force, omega)
        k = create_lb_function(lbm_config=LBMConfig(**_method_kwargs(c)), config=config)
        k.set_faces(["periodic", "noslip", "periodic"])
        a = create_pdf_array(shape, 19, ghost_layers=0, dtype=case["dtype"])
        a.permute(3, 2, 1, 0).copy_(_initial(c, seed + 1000 * n))
        kernels.append(k)
        src.append(a)
        dst.append(torch.zeros_like(a))
    return dict(run=_run_ensemble, batch=BatchedSweep(kernels, src, dst), steps=case["steps"])


def _run_ensemble(s):
    s["batch"].run(s["steps"])
    return s["batch"].current_arrays()


def _closure_model(seed):
    from lbmpy_amd.closure import ClosureModel
    model = ClosureModel(seed=seed, nu_scale=2e-3)
    model.in_scale = np.array([1e3] * 8 + [1e6, 1e9], dtype=np.float32)
    model.pack()
    return model


def _samples(case, seed):
    """Features and targets as the coarse flows give them: second moments of the size of a strain rate, and an eddy
    viscosity that grows with it."""
    g = torch.Generator(device="cpu").manual_seed(seed)
    pi = (1e-3 * torch.randn(case["samples"], 6, generator=g)).to(_device())
    rho = (1 + 1e-2 * torch.randn(case["samples"], generator=g)).to(_device())
    return pi, rho


def _prepare_train(case, seed):
    model = _closure_model(seed)
    pi, rho = _samples(case, seed)
    x = model.features(pi, rho)
    y = 200.0 * x[:, 6].abs() + 20.0 * x[:, 3].abs()
    model.set_normalisation(x)
    model.set_output_bias(y)
    return dict(run=_run_train, model=model, x=x, y=y, batch=case["batch"])


def _run_train(s):
    m = s["model"]
    loss = m.train(s["x"], s["y"], epochs=1, batch=s["batch"], lr=1e-3)
    return {"loss": loss, "weights": m.master, "m": m.m, "v": m.v}


def _prepare_analyse(case, seed):
    from lbmpy_amd import (LBMConfig, CreateKernelConfig, Target, create_lb_function,
                           compile_macroscopic_values_getter)
    from lbmpy_amd.sweep import create_field_array, create_pdf_array
    c = dict(case, method="srt")
    config = CreateKernelConfig(target=Target.GPU, data_type=c["dtype"], compute_type=_compute(c["dtype"]),
                                ghost_layers=0)
    k = create_lb_function(lbm_config=LBMConfig(**_method_kwargs(c)), config=config)
    k.set_faces(["periodic"] * 3)
    size = (c["nx"], c["ny"], c["nz"])
    pdf = create_pdf_array(size, _q(c["stencil"]), ghost_layers=0, dtype=c["dtype"])
    pdf.permute(3, 2, 1, 0).copy_(_initial(c, seed))
    getter = compile_macroscopic_values_getter(k.method, ["density", "velocity"], ghost_layers=0)
    kind = "float64" if c["dtype"] == "float64" else "float32"
    return dict(run=_run_analyse, kernel=k, getter=getter, pdf=pdf, density=create_field_array(size, 1, 0, kind),
                velocity=create_field_array(size, 3, 0, kind))


def _run_analyse(s):
    sums = s["kernel"].conserved(s["pdf"])
    bad = s["kernel"].nonfinite_count(s["pdf"])
    s["getter"](s["pdf"], density=s["density"], velocity=s["velocity"])
    return {"sums": sums, "nonfinite": bad, "density": s["density"], "velocity": s["velocity"]}


# ---------------------------------------------------------------------- the same in 64 bits, from plain torch
def _moments(f, stencil):
    d = DIRECTIONS[stencil]
    j = [sum((f[i] if c[a] > 0 else -f[i]) for i, c in enumerate(d) if c[a]) for a in range(len(d[0]))]
    return f.sum(0), j


def _collide_moment(f, case, omega):
    """SRT, TRT (magic number 3/16) and MRT (shear moments at omega, the others at 1), incompressible, with Guo's
    force along x."""
    stencil, method, force = case["stencil"], case["method"], case.get("force", 0.0)
    d, w, inv = DIRECTIONS[stencil], _weights(stencil), _inverse(stencil)
    drho, j = _moments(f, stencil)
    u = torch.stack(j)
    u[0] += 0.5 * force
    delta = _equilibrium(stencil, method, drho + 1, u) - f
    term = [w[i] * force * (3 * (c[0] - u[0]) + 9 * sum(c[a] * u[a] for a in range(len(c))) * c[0])
            for i, c in enumerate(d)]
    if method == "mrt":
        # the projector on the shear moments: (9/2) w_i c_i c_i : (traceless part of sum_j c_j c_j x_j)
        def shear(x):
            p = [[sum(c[a] * c[b] * x[i] for i, c in enumerate(d) if c[a] * c[b]) for b in range(3)] for a in range(3)]
            t = (p[0][0] + p[1][1] + p[2][2]) / 3
            return [4.5 * w[i] * sum(c[a] * c[b] * (p[a][b] - (t if a == b else 0)) for a in range(3) for b in range(3))
                    if any(c) else torch.zeros_like(x[0]) for i, c in enumerate(d)]
        sd = shear(delta)
        out = f + delta
        for i in range(len(d)):
            out[i] += (omega - 1) * sd[i]
        if force:
            sf = shear(term)
            for i in range(len(d)):
                out[i] += 0.5 * term[i] + 0.5 * (1 - omega) * sf[i]
        return out
    odd = omega if method == "srt" else (4 - 2 * omega) / (4 * (3 / 16) * omega + 2 - omega)
    out = f.clone()
    for i in range(len(d)):
        k = inv[i]
        out[i] += 0.5 * omega * (delta[i] + delta[k]) + 0.5 * odd * (delta[i] - delta[k])
        if force:
            out[i] += 0.5 * (1 - omega / 2) * (term[i] + term[k]) + 0.5 * (1 - odd / 2) * (term[i] - term[k])
    return out


def _collide_cumulant(f, omega, model=None):
    """The D3Q27 cumulant collision (no force) with the second-order cumulants' deviators relaxed at omega and all
    else at 1: populations of the Gaussian with the relaxed covariance, by its moments up to order 2 per axis."""
    d = DIRECTIONS["D3Q27"]
    w = _weights("D3Q27")
    drho, j = _moments(f, "D3Q27")
    rho = 1 + drho
    u = [x / rho for x in j]
    full = f + torch.tensor(w, dtype=f.dtype, device=f.device).view([27] + [1] * (f.dim() - 1))
    s = {}
    for a in range(3):
        for b in range(a, 3):
            s[a, b] = sum(c[a] * c[b] * full[i] for i, c in enumerate(d) if c[a] * c[b]) / rho - u[a] * u[b]
    if model is not None:
        omega = _closure_rate(s, rho, omega, model)
    t = (s[0, 0] + s[1, 1] + s[2, 2]) / 3
    for a in range(3):
        for b in range(a, 3):
            s[a, b] = (1 - omega) * (s[a, b] - t) + 1 / 3 if a == b else (1 - omega) * s[a, b]
    xx, yy, zz, xy, xz, yz = s[0, 0], s[1, 1], s[2, 2], s[0, 1], s[0, 2], s[1, 2]
    one, none = torch.ones_like(rho), torch.zeros_like(rho)
    m = [[[none] * 3 for _ in range(3)] for _ in range(3)]       # central moments over rho
    m[0][0][0] = one
    m[2][0][0], m[0][2][0], m[0][0][2], m[1][1][0], m[1][0][1], m[0][1][1] = xx, yy, zz, xy, xz, yz
    m[2][2][0], m[2][0][2], m[0][2][2] = xx * yy + 2 * xy * xy, xx * zz + 2 * xz * xz, yy * zz + 2 * yz * yz
    m[2][1][1], m[1][2][1], m[1][1][2] = xx * yz + 2 * xy * xz, yy * xz + 2 * xy * yz, zz * xy + 2 * xz * yz
    m[2][2][2] = xx * yy * zz + 2 * (xx * yz * yz + yy * xz * xz + zz * xy * xy) + 8 * xy * xz * yz
    for axis in range(3):                                         # about u -> about 0, then values at c = -1, 0, 1
        for p in range(3):
            for q in range(3):
                def at(e):
                    return [(e, p, q), (p, e, q), (p, q, e)][axis]
                k0, k1, k2 = (m[at(e)[0]][at(e)[1]][at(e)[2]] for e in range(3))
                m1 = k1 + u[axis] * k0
                m2 = k2 + 2 * u[axis] * k1 + u[axis] * u[axis] * k0
                for e, v in enumerate(((m2 - m1) / 2, k0 - m2, (m2 + m1) / 2)):
                    m[at(e)[0]][at(e)[1]][at(e)[2]] = v
    out = torch.empty_like(f)
    for i, c in enumerate(d):
        out[i] = rho * m[c[0] + 1][c[1] + 1][c[2] + 1] - w[i]
    return out


def _network(x, p):
    """The closure's network on normalised features, from its parameters in 64 bits."""
    h = torch.tanh(x @ p["w1"].T + p["b1"])
    h = torch.tanh(h @ p["w2"].T + p["b2"])
    return h @ p["w3"] + p["b3"]


def _features(pi, rho):
    q = pi / rho[:, None]
    xx, yy, zz, xy, xz, yz = q.unbind(1)
    qq = xx * xx + yy * yy + zz * zz + 2 * (xy * xy + xz * xz + yz * yz)
    t3 = xx ** 3 + yy ** 3 + zz ** 3 + 3 * (xy * xy * (xx + yy) + xz * xz * (xx + zz) + yz * yz * (yy + zz)) \
        + 6 * xy * xz * yz
    return torch.cat([q, torch.sqrt(2 * qq)[:, None], (xx + yy + zz)[:, None], qq[:, None], t3[:, None]], dim=1)


def _split(master):
    """The master parameters as the network's matrices."""
    return {"w1": master[:512].view(32, 16)[:, :10], "w2": master[512:1536].view(32, 32), "w3": master[1536:1568],
            "b1": master[1568:1600], "b2": master[1600:1632], "b3": master[1632]}


def _closure_rate(s, rho, omega, model):
    pi = torch.stack([rho * (s[k] - (1 / 3 if k[0] == k[1] else 0)) for k in
                      ((0, 0), (1, 1), (2, 2), (0, 1), (0, 2), (1, 2))]).reshape(6, -1).T
    x = _features(pi, rho.reshape(-1)) * model["scale"]
    nu = 2e-3 * torch.nn.functional.softplus(_network(x, _split(model["master"])))
    return (1 / torch.clamp(1 / omega + 3 * nu, min=0.500003)).view(rho.shape)


def _closure_master(seed):
    """The seeded network's parameters (Glorot uniform, no biases)."""
    g = np.random.default_rng(seed)
    m = np.zeros(1633, dtype=np.float32)
    w1 = g.uniform(-1, 1, (32, 16)) * math.sqrt(6 / 42)
    w1[:, 10:] = 0
    m[:512] = w1.ravel()
    m[512:1536] = (g.uniform(-1, 1, (32, 32)) * math.sqrt(6 / 64)).ravel()
    m[1536:1568] = g.uniform(-1, 1, 32) * math.sqrt(6 / 33)
    return torch.from_numpy(m).to(_device())


def _collide(f, case, omega, model=None):
    """In place, slab by slab."""
    for z in range(0, f.shape[1], 16):
        part = f[:, z:z + 16]
        f[:, z:z + 16] = _collide_cumulant(part, omega, model) if case["method"] == "cumulant" else \
            _collide_moment(part, case, omega)


def _stream(f, case, flags=None, lid=0.0):
    """Pull: every population from its neighbour; from a wall cell (flags > 0, one ghost layer around the domain) the
    cell's own opposite one comes back, with the lid's momentum where the wall is the lid (2)."""
    d, w, inv = DIRECTIONS[case["stencil"]], _weights(case["stencil"]), _inverse(case["stencil"])
    dim = len(d[0])
    axes = list(range(dim - 1, -1, -1))
    out = torch.empty_like(f)
    for i, c in enumerate(d):
        out[i] = torch.roll(f[i], list(c), axes)
        if flags is not None and any(c):
            own = flags[tuple(slice(1, -1) for _ in range(dim))]
            nb = flags[tuple(slice(1 - c[dim - 1 - t], flags.shape[t] - 1 - c[dim - 1 - t]) for t in range(dim))]
            hit = (nb > 0) & (own == 0)
            out[i] = torch.where(hit, f[inv[i]], out[i])
            if lid and c[0]:       # the link's direction is -c: f - 6 w (-c . u)
                out[i] = torch.where(hit & (nb == 2), out[i] + 6 * w[i] * c[0] * lid, out[i])
    return out


def _wall_flags(case):
    """Flags with one ghost layer, ([z,] y, x): 0 fluid, 1 resting wall, 2 lid.  Ghost cells of periodic axes hold what
    the cells at the other side hold."""
    dim = len(DIRECTIONS[case["stencil"]][0])
    size = (case["nx"], case["ny"], case["nz"])[:dim]
    f = np.zeros([n + 2 for n in size], dtype=np.int8)
    if case["scenario"] == "periodic":
        return None
    if case["scenario"] == "cavity":
        f[:, -1] = 2
        f[:, 0] = 1
        f[0] = f[-1] = 1
        if dim == 3:
            f[:, :, 0] = f[:, :, -1] = 1
    else:
        if case["scenario"] == "spheres":
            x = np.meshgrid(*[np.arange(n) + 0.5 for n in size], indexing="ij")
            f[1:-1, 1:-1, 1:-1][_sphere_mask(case)(*x)] = 1
        f[0], f[-1] = f[-2].copy(), f[1].copy()
        f[:, 0] = f[:, -1] = 1
        f[:, :, 0] = f[:, :, -1] = 1
    return torch.from_numpy(np.ascontiguousarray(f.T)).to(_device())


def exact(case, seed):
    kind = case["kind"]
    if kind in ("loop", "closure"):
        c = _as_loop(case)
        f = _initial(c, seed).double()
        flags = None
        if c["walls"]:
            flags = torch.zeros(tuple(n + 2 for n in f.shape[1:]), dtype=torch.int8, device=f.device)
            flags[:, 0] = flags[:, -1] = 1
        model = None
        if kind == "closure":
            scale = torch.tensor([1e3] * 8 + [1e6, 1e9], dtype=torch.float64, device=f.device)
            model = {"master": _closure_master(seed).double(), "scale": scale}
        for _ in range(2):
            f = _stream(f, c, flags)
            _collide(f, c, c["omega"], model)
        return {"pdf": _laid_out(f, c["stencil"], c["pattern"]).permute(3, 2, 1, 0)}
    if kind == "ensemble":
        out = []
        for n, (shape, force, omega) in enumerate(_members(case)):
            c = _member_case(case, shape, force, omega)
            f = _initial(c, seed + 1000 * n).double()
            flags = torch.zeros(tuple(n + 2 for n in f.shape[1:]), dtype=torch.int8, device=f.device)
            flags[:, 0] = flags[:, -1] = 1
            for _ in range(case["steps"]):
                f = _stream(f, c, flags)
                _collide(f, c, omega)
            out.append(f.permute(3, 2, 1, 0))
        return out
    if kind == "step":
        return _exact_step(case, seed)
    if kind == "train":
        return _exact_train(case, seed)
    f = _initial(dict(case, method="srt"), seed).double()
    drho, j = _moments(f, case["stencil"])
    sums = torch.stack([drho.sum() + drho.numel()] + [v.sum() for v in j])
    return {"sums": sums, "nonfinite": 0, "density": (1 + drho).permute(2, 1, 0),
            "velocity": torch.stack(j).permute(3, 2, 1, 0)}


def _exact_step(case, seed):
    dim = len(DIRECTIONS[case["stencil"]][0])
    size = (case["nx"], case["ny"], case["nz"])[:dim]
    force = case["force"]
    _, u = _flow(size, seed, 0.01 if case["scenario"] != "periodic" else 0.03)
    rho = torch.ones(u.shape[1:], dtype=torch.float64, device=u.device)
    shifted = u.clone()
    shifted[0] -= 0.5 * force
    f = _equilibrium(case["stencil"], case["method"], rho, shifted).to(getattr(torch, case["dtype"])).double()
    flags = _wall_flags(case)
    lid = 0.01 if case["scenario"] == "cavity" else 0.0
    flat = f.dim() == 3
    for _ in range(case["steps"]):
        f = _stream(f, case, flags, lid)
        if flat:
            f = _collide_moment(f, case, case["omega"])
        else:
            _collide(f, case, case["omega"])
    drho, j = _moments(f, case["stencil"])
    j = torch.stack(j)
    j[0] += 0.5 * force
    if case["method"] == "cumulant":
        j = j / (1 + drho)
    back = tuple(range(dim - 1, -1, -1))
    return {"pdf": _laid_out(f, case["stencil"], case["pattern"]).permute(*range(dim, -1, -1)),
            "density": (1 + drho).permute(*back), "velocity": j.permute(*range(dim, -1, -1))}


def _exact_train(case, seed):
    pi, rho = _samples(case, seed)
    x = _features(pi.double(), rho.double())
    y = 200.0 * x[:, 6].abs() + 20.0 * x[:, 3].abs()
    x = (x - x.mean(0)) / x.std(0)
    p = _closure_master(seed).double()
    p[1632] = math.log(math.expm1(float(y.mean())))
    mask = torch.ones_like(p)
    mask[:512].view(32, 16)[:, 10:] = 0
    m, v = torch.zeros_like(p), torch.zeros_like(p)
    order = torch.randperm(len(x), generator=torch.Generator(device=x.device).manual_seed(0), device=x.device)
    losses, t = [], 0
    for s in range(0, len(x), case["batch"]):
        idx = order[s:s + case["batch"]]
        q = p.clone().requires_grad_(True)
        loss = ((torch.nn.functional.softplus(_network(x[idx], _split(q))) - y[idx]) ** 2).mean()
        loss.backward()
        g = q.grad * mask
        t += 1
        m = 0.9 * m + 0.1 * g
        v = 0.999 * v + 0.001 * g * g
        p = p - 1e-3 * (m / (1 - 0.9 ** t)) / (torch.sqrt(v / (1 - 0.999 ** t)) + 1e-8)
        losses.append(float(loss))
    return {"loss": [sum(losses) / len(losses)], "weights": p, "m": m, "v": v}
