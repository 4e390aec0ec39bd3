"""Performance cases of the ARTSS solver hot path: what a user's program has
the library do, through its public entry points.

A case's `kind` names the work:

  advect         Domain.sl_advect of one scalar (every transported field of
                 every solver, each step)
  diffuse        Domain.diffuse: the implicit Jacobi or colored Gauss-Seidel
                 loop to its tolerance, laminar or with an eddy viscosity
  explicit       the one-pass operators of a step in a row: smagorinsky,
                 divergence, projection, buoyancy_force, add_source
  vcycle         Multigrid.pressure: the reference's two V-cycles of a step,
                 and the residual norm after them
  step           Solver.step: a whole time step ("tg": NSSolver, periodic
                 Taylor-Green; "plume": NSTempTurbSolver with obstacles);
                 accelerated = the GCR solve to a residual target
  ensemble       Ensemble.step: uneven plume members advanced together
  unet_forward   UNet.forward of the learned warm start
  unet_train     UNet.gradients and UNet.adam_step: one training step

Sizes are those of artss_amd/configs, of bench.py and of
artss_amd/scenarios.py, odd and ragged boxes as in the tests, and the small
boxes of the smoke test.  Fields are float64 (x fastest, one ghost layer),
the network's volumes float32.
"""
import math
import os

import numpy as np
import torch

import artss_amd
from artss_amd import scenarios

H = scenarios.H        # cell size of the plume boxes [m]
T_AMBIENT = 293.15
KAPPA, DT = 4.2e-5, 0.005  # the plume configurations' constants
CS, BETA, G = 0.2, 3.34e-3, -9.81
TG_NU, TG_DT = 0.01, 0.001             # the Taylor-Green configuration's
DIFF_TOL, DIFF_MAX = 1e-7, 100
TARGET = 1e-8                          # pressure residual target per step
CHANNELS = ((2, 16, 0), (16, 16, 0), (16, 32, 1), (32, 64, 2), (64, 64, 3), (64, 64, 2), (64, 32, 1), (32, 16, 0),
            (16, 1, 0))                # (c_in, c_out, level) of the network's layers


# ---------------------------------------------------------------- the cases
def listed():
    return [
        # the smallest call: one operator on the smoke test's box, all latency
        {"name": "advect_16x16x16", "kind": "advect", "nx": 16, "ny": 16, "nz": 16, "obstacles": 0},
        # one operator on an ordinary ragged box with obstacles
        {"name": "advect_150x70x93", "kind": "advect", "nx": 150, "ny": 70, "nz": 93, "obstacles": 2},
        # the turbulent diffusion of one field at the benchmark size
        {"name": "diffuse_cgs_256x128x128", "kind": "diffuse", "nx": 256, "ny": 128, "nz": 128, "obstacles": 1,
         "method": "ColoredGaussSeidel", "turbulent": True},
        # the laminar diffusion with the other method, odd sides
        {"name": "diffuse_jacobi_97x61x45", "kind": "diffuse", "nx": 97, "ny": 61, "nz": 45, "obstacles": 1,
         "method": "Jacobi", "turbulent": False},
        # turbulence, divergence, projection and buoyancy on an ordinary room
        {"name": "explicit_200x100x50", "kind": "explicit", "nx": 200, "ny": 100, "nz": 50, "obstacles": 2},
        # the reference's pressure call on a room of the ensemble range
        {"name": "vcycle_160x96x64", "kind": "vcycle", "nx": 160, "ny": 96, "nz": 64, "obstacles": 2, "levels": 4},
        # artss_amd/configs/taylor_green_64.xml as it stands (the default path)
        {"name": "step_tg_64", "kind": "step", "flow": "tg", "nx": 64, "ny": 64, "nz": 64, "obstacles": 0, "levels": 4,
         "accelerated": False},
        # the plume at 128^3 on the default path (the reference's schedule)
        {"name": "step_plume_128", "kind": "step", "flow": "plume", "nx": 128, "ny": 128, "nz": 128, "obstacles": 1,
         "levels": 5, "accelerated": False},
        # bench.py's workload and settings: the accelerated plume step
        {"name": "step_plume_gcr_256x128x128", "kind": "step", "flow": "plume", "nx": 256, "ny": 128, "nz": 128,
         "obstacles": 1, "levels": 5, "accelerated": True},
        # bench.py's ensemble distribution, eight members on eight host threads
        {"name": "ensemble_8", "kind": "ensemble", "members": 8, "boxes": 2026, "max_nx": 160, "max_ny": 96,
         "max_nz": 64},
        # the learned start's forward pass at the benchmark size
        {"name": "unet_forward_256x128x128", "kind": "unet_forward", "nx": 256, "ny": 128, "nz": 128},
        # one training step of the network on a room of the ensemble range
        {"name": "unet_train_128x64x64", "kind": "unet_train", "nx": 128, "ny": 64, "nz": 64},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _box(rng, lo, hi, most, q=1):
    """three sides in [lo, hi] (multiples of q), at most `most` cells"""
    while True:
        n = [max(lo, _log_int(rng, lo, hi) // q * q) for _ in range(3)]
        if n[0] * n[1] * n[2] <= most:
            return {"nx": n[0], "ny": n[1], "nz": n[2]}


def draw(rng):
    kind = rng.choice(["advect", "diffuse", "explicit", "vcycle", "step", "step", "ensemble", "unet_forward",
                       "unet_train"])
    most = 256 * 128 * 128
    if kind == "advect" or kind == "explicit":
        return dict(_box(rng, 12, 256, most), kind=kind, obstacles=rng.randint(0, 3))
    if kind == "diffuse":
        return dict(_box(rng, 16, 256, most), kind=kind, obstacles=rng.randint(0, 3),
                    method=rng.choice(["ColoredGaussSeidel", "Jacobi"]), turbulent=rng.random() < 0.6)
    if kind == "vcycle":
        n = _box(rng, 16, 256, most)
        return dict(n, kind=kind, obstacles=rng.randint(0, 2), levels=_levels(n))
    if kind == "step":
        accelerated = rng.random() < 0.5
        if accelerated:
            n = _box(rng, 32, 256, most, 8)
            return dict(n, kind=kind, flow="plume", obstacles=rng.randint(0, 2), levels=_levels(n), accelerated=True)
        flow = rng.choice(["tg", "plume"])
        n = _box(rng, 32, 128, 128 ** 3)
        return dict(n, kind=kind, flow=flow, obstacles=0 if flow == "tg" else rng.randint(0, 2), levels=_levels(n),
                    accelerated=False)
    if kind == "ensemble":
        return {"kind": kind, "members": rng.randint(2, 8), "boxes": rng.randint(1, 9999),
                "max_nx": 8 * rng.randint(8, 20), "max_ny": 8 * rng.randint(8, 12), "max_nz": 8 * rng.randint(4, 8)}
    most_net = 256 * 128 * 128 if kind == "unet_forward" else 128 * 64 * 64
    return dict(_box(rng, 16, 256 if kind == "unet_forward" else 128, most_net, 8), kind=kind)


def _levels(n):
    """multigrid levels as the configurations choose them: the coarsest level
    keeps a few cells along the shortest side"""
    return max(2, min(5, int(math.log2(min(n["nx"], n["ny"], n["nz"]))) - 2))


# ---------------------------------------------------------------- inputs
def _obstacle_boxes(case):
    """inclusive cell ranges (x1, x2, y1, y2, z1, z2; inner cells count from
    1) of the case's obstacles: boxes on the floor, clear of the side walls
    and of each other, on multiples of four cells where the box is large"""
    n = (case["nx"], case["ny"], case["nz"])
    out = []
    for o in range(case.get("obstacles", 0)):
        q = 4 if min(n) >= 32 else 1
        x1 = max(q, (2 + 4 * o) * n[0] // 16 // q * q)
        z1 = max(q, 10 * n[2] // 16 // q * q)
        wx, wy, wz = (max(q, n[a] // d // q * q) for a, d in ((0, 8), (1, 3), (2, 6)))
        out.append((x1 + 1, x1 + wx, 1, wy, z1 + 1, z1 + wz))
    return out


def _plume_text(case, peak_kw=50.0, source=None):
    n = (case["nx"], case["ny"], case["nz"])
    boxes = [((b[0] - 1) * H, b[1] * H, (b[2] - 1) * H, b[3] * H, (b[4] - 1) * H, b[5] * H)
             for b in _obstacle_boxes(case)]
    return scenarios.plume_xml(n, peak_kw, source, boxes, levels=case.get("levels", 1))


def _tg_text(case):
    with open(os.path.join(artss_amd.CONFIG_DIR, "taylor_green_64.xml")) as fh:
        text = fh.read()
    for a in ("x", "y", "z"):
        text = text.replace("<n%s> 64 </n%s>" % (a, a), "<n%s> %d </n%s>" % (a, case["n" + a], a))
    return text.replace("<n_level> 4 </n_level>", "<n_level> %d </n_level>" % case["levels"])


def _coords(case):
    """cell centres per axis in units of the box side, (z, y, x) broadcastable"""
    out = []
    for a, n in enumerate((case["nz"], case["ny"], case["nx"])):
        c = (torch.arange(n + 2, dtype=torch.float64, device="cuda") - 0.5) / n
        out.append(c.reshape([-1 if d == a else 1 for d in range(3)]))
    return out


def _smooth(case, gen, modes=3, whole=1):
    """a smooth field of unit size: a few products of cosines; whole = 2
    gives whole periods per side (periodic boxes)"""
    z, y, x = _coords(case)
    f = 0.0
    for _ in range(modes):
        k = torch.randint(1, 4, (3,), generator=gen, device="cuda").tolist()
        ph = (2 * math.pi * torch.rand(3, generator=gen, device="cuda", dtype=torch.float64)).tolist()
        f = f + (torch.cos(math.pi * whole * k[0] * x + ph[0]) * torch.cos(math.pi * whole * k[1] * y + ph[1]) *
                 torch.cos(math.pi * whole * k[2] * z + ph[2]))
    return f / math.sqrt(modes)


def _inputs(case, seed):
    """the fields a step has in hand (z, y, x, with ghosts): velocity up to
    about one cell per step, a heated column, pressure of the plume's scale"""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(int(seed))

    def rough(scale):
        shape = (case["nz"] + 2, case["ny"] + 2, case["nx"] + 2)
        return scale * torch.randn(shape, generator=gen, device="cuda", dtype=torch.float64)

    f = {}
    speed = 0.6 * H / DT
    for c in "uvw":
        f[c] = speed * _smooth(case, gen) + rough(0.01 * speed)
    z, y, x = _coords(case)
    cx, cz = (0.3 + 0.4 * torch.rand(2, generator=gen, device="cuda", dtype=torch.float64)).tolist()
    f["T"] = T_AMBIENT + 40.0 * torch.exp(-((x - cx) ** 2 + (z - cz) ** 2) / 0.03 - y) + rough(0.05)
    f["p"] = 1e-3 * _smooth(case, gen) + rough(1e-6)
    f["rhs"] = _smooth(case, gen) + rough(0.05)
    f["nu_t"] = 1e-4 * (1.0 + _smooth(case, gen) ** 2)
    return f


def _tg_inputs(case, seed):
    """velocity of a periodic box: the Taylor-Green field and a seeded
    smooth disturbance"""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(int(seed))
    z, y, x = (2 * math.pi * c for c in _coords(case))
    f = {"u": torch.sin(x) * torch.cos(y) * torch.cos(z), "v": -torch.cos(x) * torch.sin(y) * torch.cos(z)}
    f["w"] = torch.zeros_like(f["u"])
    return {c: (f[c] + 0.1 * _smooth(case, gen, whole=2)).contiguous() for c in "uvw"}


def _plume_start(case_n, seed):
    """a developing plume: velocity from a stream function that vanishes at
    the walls (no divergence to speak of) and a warm column over the source"""
    nx, ny, nz = case_n
    rng = np.random.default_rng(int(seed))
    x, y, z = ((np.arange(n + 2) - 0.5) / n for n in (nx, ny, nz))
    amp, shift = 0.25 * rng.uniform(0.8, 1.2), rng.uniform(-0.05, 0.05)
    sx, sy, sz = np.sin(math.pi * x), np.sin(math.pi * y), np.sin(math.pi * z)
    cx, cy = np.cos(math.pi * x), np.cos(math.pi * y)
    # psi = amp sx^2 sy^2 sz^2 / pi (per metre of the box's height)
    u = 2 * amp * (sz ** 2)[:, None, None] * (sy * cy)[None, :, None] * (sx ** 2)[None, None, :]
    v = -2 * amp * ny / nx * (sz ** 2)[:, None, None] * (sy ** 2)[None, :, None] * (sx * cx)[None, None, :]
    T = T_AMBIENT + 20.0 * (np.exp(-((z - 0.5 - shift) / 0.12) ** 2)[:, None, None] *
                            np.exp(-y / 0.4)[None, :, None] *
                            np.exp(-((x - 0.5 + shift) / 0.1) ** 2)[None, None, :])
    return u, v, T


class _Memory:
    """a device array of the library as an argument of torch.as_tensor; the
    tensor keeps this object and so the array's owner"""

    def __init__(self, owner, shape, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": shape, "typestr": typestr, "data": (owner.ptr.value, False),
                                         "version": 3, "strides": None}


def _field_view(field):
    return torch.as_tensor(_Memory(field, (field.n,), "<f8"), device="cuda")


def _buffer_view(buf):
    return torch.as_tensor(_Memory(buf, buf.shape, "<f4"), device="cuda")


def _set_fields(solver, fields):
    """an initial state: the field and its copies of the step before"""
    for name, host in fields.items():
        for copy in (name, name + "0", name + "_tmp"):
            solver.set_field(copy, host)


def _accelerate(solver, sweeps=True):
    """bench.py's settings of the accelerated path"""
    solver.set_mg_schedule(2, 4096)
    solver.set_pressure_mode(True, TARGET, 500)
    solver.set_pressure_method(2, 5)
    solver.set_coarse_tolerance(-1.0)
    if sweeps:
        solver.set_mixed_sweeps(1, 1, 0.9)
        solver.set_coarse_solve(True)
        solver.set_mixed_tail(3)
    solver.set_warm_start(1)


class _Arrays:
    """torch tensors handed to the library's operators as device fields"""

    def __init__(self, dom, tensors):
        self.t = {k: v.contiguous() for k, v in tensors.items()}
        self.f = {k: artss_amd.DeviceField.view(dom, v.data_ptr(), v.numel()) for k, v in self.t.items()}


def _net_params(seed):
    """a trained network's scale of weights: He-distributed, small biases"""
    rng = np.random.default_rng(int(seed))
    flat = []
    for ci, co, _ in CHANNELS:
        flat.append(rng.standard_normal(27 * ci * co) * math.sqrt(2.0 / (27 * ci)))
        flat.append(0.05 * rng.standard_normal(co))
    return np.concatenate(flat).astype(np.float32)


def _net_volumes(case, seed):
    """input (residual and increment, unit scale) and target, (z, y, x, c)"""
    rng = np.random.default_rng(int(seed) + 1)
    n = (case["nz"], case["ny"], case["nx"])
    x = np.empty(n + (2,), np.float32)
    x[..., 0] = rng.standard_normal(n, dtype=np.float32)
    c = [np.cos(2 * math.pi * np.arange(m) / m + rng.uniform(0, 6)).astype(np.float32) for m in n]
    x[..., 1] = c[0][:, None, None] + c[1][None, :, None] * c[2][None, None, :]
    t = 0.5 * x[..., :1] + 0.2 * rng.standard_normal(n + (1,), dtype=np.float32)
    return x, t


# ---------------------------------------------------------------- prepare and run
def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case}
    if kind in ("advect", "diffuse", "explicit", "vcycle"):
        dom = artss_amd.Domain(_plume_text(case))
        f = _inputs(case, seed)
        empty = lambda: torch.zeros_like(f["u"])  # noqa: E731
        if kind == "advect":
            f.update(out=empty())
        elif kind == "diffuse":
            f.update(b=f["T"], out=f["T"].clone(), start=f["T"].clone())
            f["in"] = f["T"].clone()
        elif kind == "explicit":
            f.update(ev=empty(), div=empty(), ou=empty(), ov=empty(), ow=empty(), force=empty(),
                     Ta=torch.full_like(f["u"], T_AMBIENT))
        else:
            f.update(start=f["p"].clone())
        s.update(dom=dom, a=_Arrays(dom, f))
        if kind == "vcycle":
            s["mg"] = dom.multigrid()
    elif kind == "step" and case["flow"] == "tg":
        s["solver"] = solver = artss_amd.Solver(_tg_text(case))
        fields = {c: v.cpu().numpy() for c, v in _tg_inputs(case, seed).items()}
        _set_fields(solver, {c: v.reshape(-1) for c, v in fields.items()})
        s.update(n=1, dt=TG_DT, out={c: _field_view(solver.device_field(c)) for c in "uvwp"})
    elif kind == "step":
        rng = np.random.default_rng(int(seed))
        X, Z = case["nx"] * H, case["nz"] * H
        source = (X * rng.uniform(0.55, 0.6), Z * rng.uniform(0.3, 0.4))
        s["solver"] = solver = artss_amd.Solver(_plume_text(case, rng.uniform(40.0, 60.0), source))
        if case["accelerated"]:
            _accelerate(solver)
        u, v, T = _plume_start((case["nx"], case["ny"], case["nz"]), seed)
        _set_fields(solver, {"u": u.reshape(-1), "v": v.reshape(-1), "T": T.reshape(-1)})
        s.update(n=1, dt=DT, out={c: _field_view(solver.device_field(c)) for c in ("u", "v", "w", "p", "T")})
        for _ in range(4):  # a run under way: set-up and the steps from the start are behind it
            run(s)
    elif kind == "ensemble":
        texts = scenarios.ensemble_members(case["members"], seed=case["boxes"], nx=(64, case["max_nx"]),
                                           ny=(64, case["max_ny"]), nz=(32, case["max_nz"]))
        s["members"] = members = [artss_amd.Solver(t) for t in texts]
        for i, m in enumerate(members):
            _accelerate(m, sweeps=False)
            u, v, T = _plume_start(m.domain.info(0)["n"], 100 * int(seed) + i)
            _set_fields(m, {"u": u.reshape(-1), "v": v.reshape(-1), "T": T.reshape(-1)})
            for n in range(2, 6):  # set-up and the first steps, one member after the other
                m.step(n * DT)
        s["ensemble"] = artss_amd.Ensemble(members, threads=8)
        s.update(n=5, out=[{c: _field_view(m.device_field(c)) for c in ("u", "v", "w", "p", "T")} for m in members])
    else:
        dom = artss_amd.Domain(os.path.join(artss_amd.CONFIG_DIR, "taylor_green_64.xml"))
        net = artss_amd.UNet(dom, seed=1)
        net.set_params(_net_params(seed))
        x, t = _net_volumes(case, seed)
        s.update(dom=dom, net=net, x=artss_amd.Buffer(dom, x))
        if kind == "unet_forward":
            s["y"] = artss_amd.Buffer(dom, np.zeros_like(t))
            s["out"] = _buffer_view(s["y"])
        else:
            s["target"] = artss_amd.Buffer(dom, t)
    torch.cuda.synchronize()  # the inputs are complete before the library's own stream reads them
    return s


def run(s):
    kind = s["case"]["kind"]
    if kind == "advect":
        d, f = s["dom"], s["a"].f
        d.sl_advect(f["out"], f["T"], f["u"], f["v"], f["w"], artss_amd.T)
        return s["a"].t["out"]
    if kind == "diffuse":
        d, f, t = s["dom"], s["a"].f, s["a"].t
        # the loop iterates from the advected field and leaves its last two
        # iterates in out and in; torch's copy is waited for, since the
        # library runs on its own stream
        t["in"].copy_(t["start"])
        torch.cuda.current_stream().synchronize()
        it, _ = d.diffuse(s["case"]["method"], f["out"], f["in"], f["b"], KAPPA,
                          f["nu_t"] if s["case"]["turbulent"] else None, artss_amd.T, DIFF_MAX, DIFF_TOL, 1.0)
        return {"out": t["out"], "in": t["in"], "iterations": it}
    if kind == "explicit":
        d, f, t = s["dom"], s["a"].f, s["a"].t
        d.smagorinsky(f["ev"], f["u"], f["v"], f["w"], CS)
        d.divergence(f["div"], f["u"], f["v"], f["w"])
        d.projection(f["ou"], f["ov"], f["ow"], f["u"], f["v"], f["w"], f["p"])
        d.buoyancy_force(f["force"], f["T"], f["Ta"])
        d.add_source(f["ov"], f["force"], artss_amd.V)
        return {k: t[k] for k in ("ev", "div", "ou", "ov", "ow", "force")}
    if kind == "vcycle":
        f, t = s["a"].f, s["a"].t
        t["p"].copy_(t["start"])
        torch.cuda.current_stream().synchronize()
        s["mg"].pressure(f["p"], f["rhs"], 2 * DT)
        return {"p": t["p"], "residual": s["mg"].residual(f["p"], f["rhs"])}
    if kind == "step":
        s["n"] += 1
        s["solver"].step(s["n"] * s["dt"])
        return s["out"]
    if kind == "ensemble":
        s["n"] += 1
        s["ensemble"].step(s["n"])
        return s["out"]
    if kind == "unet_forward":
        s["net"].forward(s["x"], s["y"])
        return s["out"]
    loss, grads = s["net"].gradients(s["x"], s["target"])
    s["net"].adam_step(1e-3)
    return {"loss": loss, "gradients": grads}


# ---------------------------------------------------------------- work and tolerance
def _cells(case):
    return case["nx"] * case["ny"] * case["nz"]


def work(case):
    """each input field read once, each output field written once"""
    kind = case["kind"]
    if kind == "ensemble":
        cells = case["members"] * (64 + case["max_nx"]) // 2 * (64 + case["max_ny"]) // 2 * (32 + case["max_nz"]) // 2
        return {"bytes": 88 * cells, "flops": 1500 * cells}
    n = _cells(case)
    if kind == "advect":
        return {"bytes": 40 * n, "flops": 45 * n}
    if kind == "diffuse":
        return {"bytes": (40 if case["turbulent"] else 32) * n, "flops": 80 * n}
    if kind == "explicit":
        return {"bytes": 112 * n, "flops": 90 * n}
    if kind == "vcycle":
        return {"bytes": 24 * n, "flops": 250 * n}
    if kind == "step":  # velocity, pressure, temperature and eddy viscosity in and out
        fields = 4 if case["flow"] == "tg" else 5.5
        return {"bytes": int(16 * fields * n), "flops": (1500 if case["accelerated"] else 600) * n}
    flops = sum(2 * 27 * ci * co * (n >> (3 * level)) for ci, co, level in CHANNELS)
    weights = sum(4 * (27 * ci * co + co) for ci, co, _ in CHANNELS)
    if kind == "unet_forward":
        return {"bytes": 12 * n + weights, "flops": flops}
    return {"bytes": 12 * n + 6 * weights, "flops": 3 * flops}


def tolerance(case):
    """each about four times what was measured"""
    kind = case["kind"]
    if kind == "unet_forward":  # BF16 activations: 0.2 to 1.4 % from 64 bits, by how far the outputs cancel
        return {"rel": 0.02, "max": 0.2}
    if kind == "unet_train":  # gradients: 0.3 to 2.8 % from 64 bits
        return {"rel": 0.03, "max": 0.3}
    if kind == "ensemble" or case.get("accelerated"):
        # the iteration stops at a residual, not at one iterate: other sweeps
        # and starts, or all in 64 bits, end within rel 1.1e-8, max 6.2e-8 (p)
        return {"rel": 5e-8, "max": 2.5e-7}
    if kind in ("vcycle", "step"):  # sums and sweeps in another order: 5e-16
        return {"rel": 1e-13, "max": 1e-10}
    return {"rel": 4e-15, "max": 1e-12}  # 7e-16


# ---------------------------------------------------------------- the same in plain torch
class _Level:
    """one grid level: spacing, fluid cells, obstacle boxes and the fill"""

    def __init__(self, n, h, boxes):
        self.n, self.h, self.boxes = n, h, boxes
        m = torch.zeros(n[2] + 2, n[1] + 2, n[0] + 2, dtype=torch.bool, device="cuda")
        m[1:-1, 1:-1, 1:-1] = True
        for b in boxes:
            m[b[4]:b[5] + 1, b[2]:b[3] + 1, b[0]:b[1] + 1] = False
        self.fluid = m

    def fill(self, f, bc):
        """obstacle faces, then the domain's patches; bc: "p", "T", velocity
        "v", or "tg" (periodic); left, right, bottom, top, front, back"""
        for b in self.boxes:
            s = -1.0 if bc == "v" else 1.0
            z, y, x = slice(b[4], b[5] + 1), slice(b[2], b[3] + 1), slice(b[0], b[1] + 1)
            if b[0] > 1:
                f[z, y, b[0]] = s * f[z, y, b[0] - 1]
            if b[1] < self.n[0]:
                f[z, y, b[1]] = s * f[z, y, b[1] + 1]
            if b[2] > 1:
                f[z, b[2], x] = s * f[z, b[2] - 1, x]
            if b[3] < self.n[1]:
                f[z, b[3], x] = s * f[z, b[3] + 1, x]
            if b[4] > 1:
                f[b[4], y, x] = s * f[b[4] - 1, y, x]
            if b[5] < self.n[2]:
                f[b[5], y, x] = s * f[b[5] + 1, y, x]
        for patch in range(6):
            d = f.transpose(0, 2 - patch // 2)  # the patch's axis first (a view)
            ghost, near, far = (0, 1, -2) if patch % 2 == 0 else (-1, -2, 1)
            if bc == "tg":
                d[ghost] = d[far]
            elif bc == "v":
                d[ghost] = d[near] if patch == 3 else -d[near]
            elif bc == "p":
                d[ghost] = -d[near] if patch == 3 else d[near]
            else:
                d[ghost] = d[near] if patch in (2, 3) else 2 * T_AMBIENT - d[near]
        return f


def _sh(f, dx=0, dy=0, dz=0):
    """f at the cell's neighbour (wrapping reaches no fluid cell)"""
    return torch.roll(f, (-dz, -dy, -dx), (0, 1, 2))


def _pairs(f):
    return _sh(f, 1) + _sh(f, -1), _sh(f, 0, 1) + _sh(f, 0, -1), _sh(f, 0, 0, 1) + _sh(f, 0, 0, -1)


def _hierarchy(case, levels):
    n = (case["nx"], case["ny"], case["nz"])
    length = (1.0, 1.0, 1.0) if case.get("flow") == "tg" else tuple(H * m for m in n)
    boxes, out = _obstacle_boxes(case), []
    for _ in range(levels + 1):
        out.append(_Level(n, [length[a] / n[a] for a in range(3)], boxes))
        n = tuple(1 if m == 1 else m // 2 for m in n)
        boxes = [tuple((e + 1) // 2 for e in b) for b in boxes]
    return out


def _advect(L, f, u, v, w, dt):
    nz, ny, nx = f.shape
    pos = torch.meshgrid(*(torch.arange(m, device="cuda") for m in f.shape), indexing="ij")
    near, off, frac = [], [], []
    for axis, vel in ((2, u), (1, v), (0, w)):
        c = vel * (dt / L.h[2 - axis])
        shift = torch.trunc(c)
        still = c.abs() <= 1e-6
        i0 = (pos[axis] - shift.to(torch.int64)).clamp(1, f.shape[axis] - 2)
        near.append(torch.where(still, pos[axis], i0))
        off.append(torch.where(still, near[-1], i0 - torch.sign(c).to(torch.int64)))
        frac.append(torch.where(still, torch.ones_like(c), (c - shift).abs()))

    def at(a, b, c):
        i, j, k = ((off if s else near)[n].clamp(0, m - 1) for n, (s, m) in enumerate(zip((a, b, c), (nx, ny, nz))))
        return f[k, j, i]

    r, s, t = frac
    line = {}
    for b in (0, 1):
        for c in (0, 1):
            lo = at(0, b, c)
            line[b, c] = lo + r * (at(1, b, c) - lo)
    plane = [line[0, c] + s * (line[1, c] - line[0, c]) for c in (0, 1)]
    return plane[0] + t * (plane[1] - plane[0])


def _diffuse(L, method, x, b, D, ev, dt, bc):
    """the implicit loop from x: out and in as the loop leaves them, and its iterations"""
    e = D if ev is None else D + ev
    ax, ay, az = (e * dt / (h * h) for h in L.h)
    rb = 1.0 + 2.0 * (ax + ay + az)
    parity = sum(torch.meshgrid(*(torch.arange(m, device="cuda") for m in x.shape), indexing="ij")) % 2
    shell = torch.ones_like(L.fluid)
    shell[1:-1, 1:-1, 1:-1] = False
    start, it, res = x, 0, 1.0
    while res > DIFF_TOL and it < DIFF_MAX:
        new = x.clone()
        for color in ((0, 1) if method != "Jacobi" else (None,)):
            px, py, pz = _pairs(new)
            at = L.fluid if color is None else L.fluid & (parity == color)
            new = torch.where(at, (b + ax * px + ay * py + az * pz) / rb, new)
        L.fill(new, bc)
        res = float((rb * (new - x))[L.fluid].square().sum().sqrt())
        # Jacobi's in follows out except in its obstacle cells
        before, x, it = x, torch.where(L.fluid | shell, new, start) if method == "Jacobi" else new, it + 1
    return new, x if method == "Jacobi" else before, it


def _lap(L, x):
    px, py, pz = _pairs(x)
    rx, ry, rz = (1.0 / (h * h) for h in L.h)
    return rx * (px - 2 * x) + ry * (py - 2 * x) + rz * (pz - 2 * x)


def _residual(L, x, b):
    return float((b - _lap(L, x))[L.fluid].square().sum().sqrt())


def _sweep(L, x, b, bc, w=0.6666666667):
    px, py, pz = _pairs(x)
    rx, ry, rz = (1.0 / (h * h) for h in L.h)
    return L.fill(torch.where(L.fluid, (1 - w) * x + w * (-b + rx * px + ry * py + rz * pz) / (2 * (rx + ry + rz)), x),
                  bc)


def _fine(a):
    """the eight fine cells of every coarse inner cell, (2, 2, 2) slices"""
    return [slice(1 + d, 1 + d + 2 * (a - 1) + 1, 2) for d in (0, 1)]


def _vcycle(levels, p, b, bc):
    """one V-cycle of the reference's schedule: four relaxations per
    smoothing, of which the pointer swaps return the third"""
    top = len(levels) - 1
    err, rhs = [p.clone()], [b]
    for l in range(top):
        L, C = levels[l], levels[l + 1]
        err[l] = L.fill(err[l], bc)
        for _ in range(3):
            err[l] = _sweep(L, err[l], rhs[l], bc)
        r = torch.where(L.fluid, rhs[l] - _lap(L, err[l]), torch.zeros_like(err[l]))
        sx, sy, sz = (_fine(m) for m in C.n)
        c = sum(r[z, y, x] for z in sz for y in sy for x in sx) * 0.125
        full = torch.zeros_like(C.fluid, dtype=torch.float64)
        full[1:-1, 1:-1, 1:-1] = c
        rhs.append(torch.where(C.fluid, full, torch.zeros_like(full)))
        err.append(torch.zeros_like(full))
    for l in range(top, 0, -1):
        F, C = levels[l - 1], levels[l]
        e = torch.zeros_like(err[l - 1])
        sx, sy, sz = (_fine(m) for m in C.n)
        for k in (0, 1):
            for j in (0, 1):
                for i in (0, 1):
                    d = [2 * q - 1 for q in (i, j, k)]
                    c, v = err[l], 27 * err[l]
                    v = v + 9 * (_sh(c, d[0]) + _sh(c, 0, d[1]) + _sh(c, 0, 0, d[2]))
                    v = v + 3 * (_sh(c, d[0], d[1]) + _sh(c, d[0], 0, d[2]) + _sh(c, 0, d[1], d[2]))
                    v = torch.where(C.fluid, (v + _sh(c, *d)) / 64, torch.zeros_like(c))
                    e[sz[k], sy[j], sx[i]] = v[1:-1, 1:-1, 1:-1]
        x = F.fill(err[l - 1] + F.fill(e, bc), bc)
        if l < top or (F.n[0] <= 2 and F.n[1] <= 2):
            for _ in range(3):
                x = _sweep(F, x, rhs[l - 1], bc)
        else:
            it, before = 0, x
            while it == 0 or (_residual(F, x, rhs[l - 1]) > 1e-8 and it < 100):
                before, x, it = x, _sweep(F, x, rhs[l - 1], bc), it + 1
            x = before if it % 2 == 0 else x
        err[l - 1] = x
    return levels[0].fill(err[0], bc)


def _keep(L, new, old):
    return torch.where(L.fluid, new, old)


def _diff(L, f, axis):
    d = [0, 0, 0]
    d[axis] = 1
    return (_sh(f, *d) - _sh(f, *[-q for q in d])) * 0.5 / L.h[axis]


def _conv(x, W, b):
    """3x3x3 convolution, zero padding, channels last: 27 products"""
    Z, Y, X, ci = x.shape
    xp = torch.nn.functional.pad(x, (0, 0, 1, 1, 1, 1, 1, 1))
    out = b.expand(Z * Y * X, -1)
    for t in range(27):
        dz, dy, dx = t // 9, (t // 3) % 3, t % 3
        out = out + xp[dz:dz + Z, dy:dy + Y, dx:dx + X].reshape(-1, ci) @ W[t]
    return out.reshape(Z, Y, X, -1)


def _down(x):
    Z, Y, X, C = x.shape
    return x.reshape(Z // 2, 2, Y // 2, 2, X // 2, 2, C).mean((1, 3, 5))


def _up(x):
    for a in range(3):
        x = x.repeat_interleave(2, a)
    return x


def _net(params, x):
    p = [(params[2 * q], params[2 * q + 1]) for q in range(9)]
    relu = torch.relu
    h0 = relu(_conv(x, *p[0]))
    e0 = relu(_conv(h0, *p[1]))
    e1 = relu(_conv(_down(e0), *p[2]))
    e2 = relu(_conv(_down(e1), *p[3]))
    e3 = relu(_conv(_down(e2), *p[4]))
    d2 = relu(_conv(_up(e3), *p[5])) + e2
    d1 = relu(_conv(_up(d2), *p[6])) + e1
    d0 = relu(_conv(_up(d1), *p[7])) + e0
    return _conv(d0, *p[8])


def _exact_net(case, seed):
    flat, params, off = torch.tensor(_net_params(seed), dtype=torch.float64, device="cuda"), [], 0
    for ci, co, _ in CHANNELS:
        for shape in ((27, ci, co), (co,)):
            m = math.prod(shape)
            params.append(flat[off:off + m].reshape(shape).clone())
            off += m
    x, t = (torch.tensor(a, dtype=torch.float64, device="cuda") for a in _net_volumes(case, seed))
    if case["kind"] == "unet_forward":
        with torch.no_grad():
            return _net(params, x)
    for q in params:
        q.requires_grad_(True)
    loss = (_net(params, x) - t).square().mean()
    grads = torch.autograd.grad(loss, params)
    return {"loss": float(loss), "gradients": torch.cat([g.reshape(-1) for g in grads]).cpu().numpy()}


def exact(case, seed):
    kind = case["kind"]
    if kind in ("unet_forward", "unet_train"):
        return _exact_net(case, seed)
    if kind == "ensemble" or case.get("flow") == "plume":
        # whole plume steps: hundreds of V-cycles to the residual target, and
        # the heat source's lines of sight past the obstacles for every cell
        return None
    if kind == "step":
        levels = _hierarchy(case, case["levels"])
        L, f = levels[0], _tg_inputs(case, seed)
        vel = {c: L.fill(_keep(L, _advect(L, f[c], f["u"], f["v"], f["w"], TG_DT), f[c]), "tg") for c in "uvw"}
        vel = {c: _diffuse(L, "Jacobi", v, v, TG_NU, None, TG_DT, "tg")[0] for c, v in vel.items()}
        div = sum(_diff(L, vel[c], a) for a, c in enumerate("uvw"))
        p = torch.zeros_like(div)
        for _ in range(2):
            p = _vcycle(levels, p, div, "tg")
        out = {c: L.fill(_keep(L, vel[c] - _diff(L, p, a), vel[c]), "tg") for a, c in enumerate("uvw")}
        out["p"] = p
        return {c: v.reshape(-1) for c, v in out.items()}
    levels = _hierarchy(case, case.get("levels", 1) if kind == "vcycle" else 0)
    L, f = levels[0], _inputs(case, seed)
    zero = torch.zeros_like(f["u"])
    if kind == "advect":
        return L.fill(_keep(L, _advect(L, f["T"], f["u"], f["v"], f["w"], DT), zero), "T")
    if kind == "diffuse":
        out, before, it = _diffuse(L, case["method"], f["T"], f["T"], KAPPA, f["nu_t"] if case["turbulent"] else None,
                                   DT, "T")
        return {"out": out, "in": before, "iterations": it}
    if kind == "explicit":
        g = {c: [_diff(L, f[c], a) for a in range(3)] for c in "uvw"}
        s12, s13, s23 = (0.5 * (g[a][i] + g[b][j]) for a, i, b, j in (("u", 1, "v", 0), ("u", 2, "w", 0),
                                                                     ("v", 2, "w", 1)))
        size = (2 * (g["u"][0] ** 2 + g["v"][1] ** 2 + g["w"][2] ** 2 + 2 * (s12 ** 2 + s13 ** 2 + s23 ** 2))).sqrt()
        delta = (L.h[0] * L.h[1] * L.h[2]) ** (1.0 / 3.0)
        out = {"ev": _keep(L, CS * CS * delta * delta * size, zero),
               "div": _keep(L, g["u"][0] + g["v"][1] + g["w"][2], zero)}
        for a, c in enumerate("uvw"):
            out["o" + c] = L.fill(_keep(L, f[c] - _diff(L, f["p"], a), zero), "v")
        force = -BETA * (f["T"] - T_AMBIENT) * G
        shell = torch.ones_like(L.fluid)
        shell[1:-1, 1:-1, 1:-1] = False
        out["force"] = torch.where(L.fluid | shell, force, zero)
        out["ov"] = L.fill(_keep(L, out["ov"] + DT * out["force"], out["ov"]), "v")
        return out
    p = f["p"]
    for _ in range(2):
        p = _vcycle(levels, p, f["rhs"], "p")
    return {"p": p, "residual": _residual(L, p, f["rhs"])}
