"""The work users of hyperboliconvergence_amd have it do, as measurable cases.

Every case is one pass of a time integration (or of its gradient) through the Python entry points,
with the state on the GPU, as a program holds it that runs many of them:

* an initial state goes in (`set_state_device`, or the device state of a batch), the steps run from
  replayed graphs (`set_graph_steps`), the final state and time come out;
* steady marching with its residual checks (`step_steady`);
* the K-step trajectory and its gradient (`adjoint.trajectory`), forward and backward.

`exact` restates the scheme in plain float64 torch: MUSCL with LSQ-biased slopes, the flux, the
boundary conditions and the Runge-Kutta step on [variable][i][j] tensors; gradients by autograd.
"""
import math

import numpy as np
import torch
import torch.utils.checkpoint

import hyperboliconvergence_amd as hca
from hyperboliconvergence_amd import adjoint, cases as drivers

GAMMA = 1.4
FLUX = {"rusanov": hca.FLUX_RUSANOV, "roe": hca.FLUX_ROE, "slau": hca.FLUX_SLAU, "ausmpup": hca.FLUX_AUSMPUP,
        "roe_faceframe": hca.FLUX_ROE_FACEFRAME}
LIMITER = {"nolimit1": hca.LIM_NOLIMIT1, "nolimit3": hca.LIM_NOLIMIT3, "vanalbada2": hca.LIM_VANALBADA2,
           "minmod2": hca.LIM_MINMOD2, "mc2": hca.LIM_MC2,
           "smooth_vanalbada": hca.LIM_SMOOTHVANALBADA}
DT = {"global": hca.DT_GLOBAL, "local": hca.DT_LOCAL, "fixed": hca.DT_FIXED}
PERIODIC, RIEMANN, FIXED, WALL = hca.BC_PERIODIC, hca.BC_RIEMANN, hca.BC_FIXED, hca.BC_WALL
STAGES = {"ssp11": 1, "ssp22": 2, "ssp33": 3, "ssp34": 4, "rk4": 4}
# families whose whole state lives on a periodic box
BOX = {"scalar": (0.0, 1.0), "gresho": (-1.0, 1.0), "vortex": (-10.0, 10.0)}
# (n_theta, n_r) of a batch's meshes, as the cylinder sweep uses them
BATCH_MESHES = ((128, 64), (256, 128), (384, 192), (512, 256))


def listed():
    """i is the radial (streamwise) index, j the contiguous one."""
    def case(name, family, ni, nj, flux, limiter, rk, dt, cfl, steps, basis="primitive", precision="fp64"):
        return {"name": name, "family": family, "ni": ni, "nj": nj, "flux": flux, "limiter": limiter, "basis": basis,
                "rk": rk, "dt": dt, "cfl": cfl, "precision": precision, "steps": steps}

    return [
        # the plain method at its smallest: scalar advection, latency and launches (van Leer, the other limiter it is
        # run with, amplifies rounding to order one within 20 steps: nothing to compare its results with)
        case("scalar 128x128", "scalar", 128, 128, "rusanov", "vanalbada2", "ssp33", "global", 0.5, 50, "conserved"),
        # the channel-with-bump driver: one-stage steps, first order, fixed states and walls
        case("bump 144x96", "bump", 144, 96, "rusanov", "nolimit1", "ssp11", "global", 0.4, 50),
        # the Gresho vortex driver: low Mach, four stages, global step
        case("gresho 256x256", "gresho", 256, 256, "rusanov", "nolimit3", "ssp34", "global", 1.6, 20),
        # the cylinder O-grid at its configured size, both precisions
        case("cylinder 256x512 fp64", "cylinder", 256, 512, "roe_faceframe", "minmod2", "rk4", "local", 1.0, 20),
        case("cylinder 256x512 mixed", "cylinder", 256, 512, "roe_faceframe", "minmod2", "rk4", "local", 1.0, 20,
             precision="mixed"),
        # steady marching with residual checks on an odd-sized O-grid, conserved variables
        case("steady 147x301 fp64", "steady", 147, 301, "roe_faceframe", "vanalbada2", "rk4", "local", 0.8, 40, "conserved"),
        # the isentropic vortex: a large box whose spacing is exact in binary, and a ragged one that is not
        case("vortex 2048x2048 fp64", "vortex", 2048, 2048, "ausmpup", "vanalbada2", "ssp33", "global", 0.8, 4),
        case("vortex 1000x901 fp64", "vortex", 1000, 901, "ausmpup", "vanalbada2", "ssp33", "global", 0.8, 6),
        # the sweep of cylinder flows, all cases in one launch per stage, both precisions
        {"name": "batch 96 fp64", "family": "batch", "count": 96, "meshes": 4, "precision": "fp64", "steps": 10},
        {"name": "batch 48 mixed", "family": "batch", "count": 48, "meshes": 4, "precision": "mixed", "steps": 10},
        # the gradient of K steps of the cylinder flow, forward and backward
        {"name": "adjoint 256x512", "family": "adjoint", "ni": 256, "nj": 512, "steps": 12, "every": 4},
        {"name": "adjoint 512x1024", "family": "adjoint", "ni": 512, "nj": 1024, "steps": 6, "every": 3},
    ]


def draw(rng):
    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    family = rng.choice(["scalar", "bump", "gresho", "cylinder", "cylinder", "steady", "vortex", "vortex", "batch",
                         "batch", "adjoint"])
    if family == "batch":
        return {"family": "batch", "count": rng.randint(4, 90), "meshes": rng.randint(2, 4),
                "precision": rng.choice(["fp64", "mixed"]), "steps": rng.randint(4, 10)}
    if family == "adjoint":
        return {"family": "adjoint", "ni": size(48, 480), "nj": size(64, 960), "steps": rng.randint(3, 8),
                "every": rng.randint(2, 4)}
    c = {"family": family, "basis": "primitive", "precision": "fp64", "steps": rng.randint(4, 20)}
    if family == "scalar":
        n = size(48, 512)
        c.update(ni=n, nj=n + rng.randint(0, 9), flux="rusanov", limiter=rng.choice(["vanalbada2", "minmod2", "nolimit3"]),
                 basis="conserved", rk=rng.choice(["ssp33", "ssp22"]), dt="global", cfl=0.5)
    elif family == "bump":
        c.update(ni=3 * size(16, 160), nj=size(24, 300), flux=rng.choice(["rusanov", "slau"]),
                 limiter=rng.choice(["nolimit1", "mc2"]), rk=rng.choice(["ssp11", "ssp33"]), dt="global", cfl=0.4)
        if c["limiter"] != "nolimit1":
            c["rk"] = "ssp33"
    elif family == "gresho":
        n = size(64, 768)
        c.update(ni=n, nj=n, flux="rusanov", limiter=rng.choice(["nolimit3", "vanalbada2"]), rk="ssp34", dt="global",
                 cfl=1.6)
    elif family in ("cylinder", "steady"):
        c.update(ni=size(32, 400), nj=size(64, 800), flux=rng.choice(["roe_faceframe", "roe", "rusanov"]),
                 limiter=rng.choice(["minmod2", "vanalbada2", "mc2"]), basis=rng.choice(["primitive", "conserved"]),
                 rk=rng.choice(["rk4", "ssp34"]), dt="local", cfl=0.8)
        if family == "cylinder" and c["flux"] in ("roe_faceframe", "rusanov"):
            c["precision"] = rng.choice(["fp64", "mixed"])
        if family == "steady":
            c["steps"] = 10 * rng.randint(1, 3)
    else:
        c.update(ni=size(64, 1800), nj=size(64, 1800), flux=rng.choice(["ausmpup", "slau"]), limiter="vanalbada2",
                 rk="ssp33", dt="global", cfl=0.8, steps=rng.randint(3, 8))
    return c


# ---------------- meshes and initial states (numpy, no library code) ----------------

def _box(ni, nj, lo, hi):
    nodes = np.empty((ni + 1, nj + 1, 2))
    nodes[..., 0] = (lo + np.arange(ni + 1) * ((hi - lo) / ni))[:, None]
    nodes[..., 1] = (lo + np.arange(nj + 1) * ((hi - lo) / nj))[None, :]
    return nodes


def _ogrid(nr, nth, rc=0.5, rb=20.0, dr0=1e-3):
    """Radii geometrically stretched from the first spacing dr0, angles uniform, closed on itself."""
    lo, hi = 1.0 + 1e-12, 2.0
    for _ in range(100):
        mid = 0.5 * (lo + hi)
        if dr0 * (mid ** nr - 1.0) / (mid - 1.0) < rb - rc:
            lo = mid
        else:
            hi = mid
    s = 0.5 * (lo + hi)
    r = rc + dr0 * (s ** np.arange(nr + 1.0) - 1.0) / (s - 1.0)
    r[nr] = rb
    th = 2.0 * math.pi * (np.arange(nth + 1) % nth) / nth
    return np.stack([r[:, None] * np.cos(th)[None, :], r[:, None] * np.sin(th)[None, :]], axis=-1)


def _bump(ni, nj):
    """A channel of height 2 and length 8 with a cosine bump of height 0.1 on the middle quarter of its lower wall."""
    x = -4.0 + np.arange(ni + 1) * (8.0 / ni)
    yl = np.where(np.abs(x) <= 1.0, 0.05 * (1.0 + np.cos(math.pi * x)), 0.0)
    eta = np.arange(nj + 1) / nj
    return np.stack([np.broadcast_to(x[:, None], (ni + 1, nj + 1)), yl[:, None] + (2.0 - yl)[:, None] * eta[None, :]],
                    axis=-1).copy()


def _centres(nodes):
    return 0.25 * (nodes[:-1, :-1] + nodes[1:, :-1] + nodes[:-1, 1:] + nodes[1:, 1:])


def _conserved(q):
    u, v, r, p = (q[..., k] for k in range(4))
    return np.stack([r * u, r * v, r, p / (GAMMA - 1.0) + 0.5 * r * (u * u + v * v)], axis=-1)


def _ripple(shape, rng, amplitude):
    """A smooth periodic field of zero mean, a different one for each variable: a few low modes."""
    ni, nj = shape
    i = (np.arange(ni) + 0.5)[:, None] / ni
    j = (np.arange(nj) + 0.5)[None, :] / nj
    out = np.zeros((ni, nj, 4))
    for k in range(4):
        for m in range(1, 4):
            a, b, c = rng.uniform(-1.0, 1.0), rng.uniform(0.0, 2 * math.pi), rng.uniform(0.0, 2 * math.pi)
            out[..., k] += a * np.cos(2 * math.pi * m * i + b) * np.cos(2 * math.pi * m * j + c)
    return (amplitude / 3.0) * out


def _freestream(rng):
    """A flow condition of the cylinder sweep: Mach number and primitive free stream."""
    mach, alpha = rng.uniform(0.2, 0.8), math.radians(rng.uniform(-5.0, 5.0))
    return mach, np.array([mach * math.cos(alpha), mach * math.sin(alpha), 1.0, 1.0 / GAMMA])


def _problem(c, seed, member=0):
    """(nodes, initial state, boundary reference row, boundary types, minf) of one case."""
    rng = np.random.default_rng([int(seed), member])
    family = c["family"]
    ni, nj = c["ni"], c["nj"]
    if family in BOX:
        nodes = _box(ni, nj, *BOX[family])
        bc, minf = (PERIODIC,) * 4, 1.0
        xy = _centres(nodes)
        x, y = xy[..., 0] - 0.05 * rng.uniform(-1, 1), xy[..., 1] - 0.05 * rng.uniform(-1, 1)
        if family == "scalar":
            q = np.empty((ni, nj, 3))
            q[..., 0], q[..., 1] = 1.0, 0.5
            q[..., 2] = np.exp(-((x - 0.5) ** 2 + (y - 0.5) ** 2) / (0.01 * rng.uniform(0.8, 1.2)))
            return nodes, q, np.zeros(3), bc, 1.0
        if family == "gresho":
            minf = 0.3
            q = _gresho(x, y, minf)
        else:
            minf = 0.5
            q = _vortex(x, y, rng.uniform(4.0, 5.0), minf)
        ref = np.array([0.0, 0.0, 1.0, 1.0])
    elif family == "bump":
        nodes, bc, minf = _bump(ni, nj), (FIXED, FIXED, WALL, WALL), rng.uniform(0.3, 0.5)
        ref = np.array([minf * math.sqrt(GAMMA), 0.0, 1.0, 1.0])
        q = ref + _ripple((ni, nj), rng, 0.01)
    else:
        nodes, bc = _ogrid(ni, nj), (WALL, RIEMANN, PERIODIC, PERIODIC)
        minf, ref = (0.4, np.array([0.4, 0.0, 1.0, 1.0 / GAMMA])) if family == "adjoint" else _freestream(rng)
        q = ref + _ripple((ni, nj), rng, 1e-3 if family == "adjoint" else 0.01)
    if c.get("basis", "primitive") == "conserved":
        q, ref = _conserved(q), _conserved(ref)
    return nodes, q, ref, bc, minf


def _gresho(x, y, mach):
    """Gresho vortex: solid-body core, a linear decay to rest at r = 0.4, the pressure that balances them."""
    r = np.maximum(np.sqrt(x * x + y * y), 1e-12)
    p0 = 1.0 / (GAMMA * mach * mach)
    ring = (r >= 0.2) & (r < 0.4)
    ut = np.where(r < 0.2, 5.0 * r, np.where(ring, 2.0 - 5.0 * r, 0.0))
    p = np.where(r < 0.2, p0 + 12.5 * r * r,
                 np.where(ring, p0 + 12.5 * r * r + 4.0 * (1.0 - 5.0 * r - math.log(0.2) + np.log(r)),
                          p0 - 2.0 + 4.0 * math.log(2.0)))
    return np.stack([0.1 - ut * y / r, ut * x / r, np.ones_like(r), p], axis=-1)


def _vortex(x, y, strength, mach):
    """Isentropic vortex at the origin of a uniform stream along the diagonal."""
    u0 = mach * math.sqrt(GAMMA) / math.sqrt(2.0)
    r2 = x * x + y * y
    e = strength / (2.0 * math.pi) * np.exp(0.5 * (1.0 - r2))
    t = 1.0 - (GAMMA - 1.0) / (2.0 * GAMMA) * e * e
    rho = t ** (1.0 / (GAMMA - 1.0))
    return np.stack([u0 - e * y, u0 + e * x, rho, rho ** GAMMA], axis=-1)


def _members(c):
    """The single cases of a batch: the sweep's meshes in turn."""
    for k in range(c["count"]):
        nth, nr = BATCH_MESHES[k % c["meshes"]]
        yield {"family": "cylinder", "ni": nr, "nj": nth, "flux": "roe_faceframe", "limiter": "minmod2",
               "basis": "primitive", "rk": "rk4", "dt": "local", "cfl": 1.0, "precision": c["precision"],
               "steps": c["steps"]}


def _adjoint_single(c):
    # a fixed step well inside the stability limit of the first radial spacing (1e-3, volumes of area / 4)
    return {"family": "adjoint", "ni": c["ni"], "nj": c["nj"], "flux": "ausmpup", "limiter": "smooth_vanalbada",
            "basis": "conserved", "rk": "ssp33", "dt": "fixed", "cfl": 0.1 * min(1e-3, 3.0 / c["nj"]), "steps": c["steps"]}


# ---------------- prepare and run ----------------

def _descriptor(c, bc, minf):
    lo, hi = BOX.get(c["family"], (0.0, 0.0))
    scalar = c["family"] == "scalar"
    return drivers.make_case(hca.LAW_SCALAR if scalar else hca.LAW_EULER,
                             hca.BASIS_CONSERVED if c["basis"] == "conserved" else hca.BASIS_PRIMITIVE,
                             FLUX[c["flux"]], LIMITER[c["limiter"]], bc, c["rk"], c["cfl"], DT[c["dt"]],
                             hca.Species() if scalar else drivers.air_species(minf), (hi - lo, 0.0), (0.0, hi - lo))


def _bref(c, ref):
    return np.tile(ref, (2 * c["nj"] + 2 * c["ni"], 1))


class _DeviceMemory:
    """A device address as torch takes it (no copy)."""

    def __init__(self, address, n):
        self.__cuda_array_interface__ = {"shape": (n,), "typestr": "<f8", "data": (address, False), "version": 2}


def _state_of(ctx, n):
    """The context's device state as a tensor (packed: case after case, [variable][cell] in each)."""
    return torch.as_tensor(_DeviceMemory(ctx.device_state_ptr(), n), device="cuda:0")


def prepare(case, seed):
    if case["family"] == "batch":
        return _prepare_batch(case, seed)
    if case["family"] == "adjoint":
        single = _adjoint_single(case)
        nodes, q, ref, bc, minf = _problem(single, seed)
        solver = adjoint.TrajectorySolver(nodes, _descriptor(single, bc, minf), case["steps"], case["every"])
        w = np.random.default_rng([int(seed), 77]).standard_normal(q.shape)
        on_gpu = [torch.from_numpy(a).cuda() for a in (q, _bref(single, ref), w)]
        return {"kind": "adjoint", "solver": solver, "q0": on_gpu[0].requires_grad_(), "w": on_gpu[2],
                "bref": on_gpu[1].requires_grad_(),
                "minf": torch.tensor(minf, dtype=torch.float64, requires_grad=True)}
    nodes, q, ref, bc, minf = _problem(case, seed)
    ctx = hca.Context(0)
    ctx.set_precision(hca.PRECISION_MIXED if case["precision"] == "mixed" else hca.PRECISION_FP64)
    ctx.set_mesh(nodes)
    ctx.set_case(_descriptor(case, bc, minf))
    ctx.set_boundary_refs(_bref(case, ref))
    ctx.set_graph_steps(10)
    q0 = torch.from_numpy(q).cuda()
    torch.cuda.synchronize()
    return {"kind": "steady" if case["family"] == "steady" else "single", "ctx": ctx, "q0": q0,
            "q": torch.empty_like(q0), "steps": case["steps"], "timed": case["dt"] == "global"}


def _prepare_batch(case, seed):
    batch = hca.Batch(0)
    batch.set_precision(hca.PRECISION_MIXED if case["precision"] == "mixed" else hca.PRECISION_FP64)
    batch.begin()
    meshes, q0, refs = {}, [], []
    for k, c in enumerate(_members(case)):
        rng = np.random.default_rng([int(seed), k])
        minf, ref = _freestream(rng)
        key = (c["ni"], c["nj"])
        if key not in meshes:
            meshes[key] = _ogrid(*key)
        batch.add_case(meshes[key], _descriptor(c, (WALL, RIEMANN, PERIODIC, PERIODIC), minf))
        q0.append(ref)
        refs.append(_bref(c, ref))
    batch.end()
    for k, c in enumerate(_members(case)):
        batch.set_case_boundary_refs(k, refs[k])
        batch.set_case_state(k, np.tile(q0[k], (c["ni"], c["nj"], 1)))
    batch.set_graph_steps(case["steps"])
    n = 4 * sum(c["ni"] * c["nj"] for c in _members(case))
    start = _state_of(batch, n).clone()
    torch.cuda.synchronize()
    return {"kind": "batch", "ctx": batch, "q0": start, "q": torch.empty_like(start), "n": n, "steps": case["steps"]}


def run(state):
    kind = state["kind"]
    if kind == "adjoint":
        wrt = (state["q0"], state["bref"], state["minf"])
        qk = adjoint.trajectory(state["solver"], *wrt)
        grads = torch.autograd.grad(qk, wrt, state["w"])
        return {"q": qk.detach(), "q0_grad": grads[0], "bref_grad": grads[1]}
    ctx = state["ctx"]
    if kind == "batch":   # restart the sweep from its free streams
        _state_of(ctx, state["n"]).copy_(state["q0"])
        torch.cuda.current_stream().synchronize()
        ctx.step(state["steps"])
        ctx.synchronize()
        return {"q": state["q"].copy_(_state_of(ctx, state["n"]))}   # the context's buffers go with it
    ctx.set_state_device(state["q0"].data_ptr())
    if kind == "steady":
        _, drop = ctx.step_steady(state["steps"], 1e-12, 10)
        ctx.get_state_device(state["q"].data_ptr())
        return {"q": state["q"], "drop": drop}
    ctx.step(state["steps"])
    ctx.get_state_device(state["q"].data_ptr())
    return {"q": state["q"], "t": ctx.time()} if state["timed"] else {"q": state["q"]}


# operations of one cell and stage (two faces, the cell update), divisions and roots counted once
FLOPS = {"scalar": 130.0, "rusanov": 420.0, "slau": 480.0, "ausmpup": 560.0, "roe": 640.0, "roe_faceframe": 660.0}


def work(case):
    """Per cell and stage: the stage's state and the step's start state read, the new state written, and on
    curvilinear meshes one mesh node; a gradient needs the trajectory and, per stage, the adjoint of the
    state read and written beside the state (about three times the operations of the forward stage)."""
    if case["family"] == "batch":
        ws = [work(c) for c in _members(case)]
        return {k: sum(w[k] for w in ws) for k in ("bytes", "flops")}
    if case["family"] == "adjoint":
        stages = case["ni"] * case["nj"] * 3.0 * case["steps"]
        return {"bytes": stages * (112.0 + 112.0), "flops": stages * 4.0 * FLOPS["ausmpup"]}
    nv = 1 if case["family"] == "scalar" else 4   # the advection velocity does not change
    stages = float(case["ni"] * case["nj"] * STAGES[case["rk"]] * case["steps"])
    geometry = 0.0 if case["family"] in BOX else 16.0
    return {"bytes": stages * (24.0 * nv + geometry),
            "flops": stages * FLOPS["scalar" if nv == 1 else case["flux"]]}


# ---------------- the scheme in plain float64 torch ----------------

def _rk(name):
    third, sixth = 1.0 / 3.0, 1.0 / 6.0
    return {"ssp11": ([[1.0]], [1.0]),
            "ssp22": ([[1.0], [0.5, 0.5]], [1.0, 1.0]),
            "ssp33": ([[1.0], [0.5, 0.5], [sixth, sixth, 2.0 / 3.0]], [1.0, 0.5, 1.0]),
            "ssp34": ([[1.0], [0.5, 0.5], [third] * 3, [sixth, sixth, sixth, 0.5]], [0.5, 1.0, 0.5, 1.0]),
            "rk4": ([[1.0], [0.0, 1.0], [0.0, 0.0, 1.0], [sixth, third, third, sixth]], [0.5, 0.5, 1.0, 1.0])}[name]


def _limited(name, a, b):
    """The limiter of the centred slope a and the upwind-biased slope b."""
    zero = torch.zeros((), dtype=a.dtype, device=a.device)
    tiny = float(np.finfo(np.float64).tiny)
    if name == "nolimit3":
        return (2.0 * a + b) / 3.0
    if name == "minmod2":
        return torch.where(a > 0, torch.minimum(a, torch.maximum(b, zero)), torch.maximum(a, torch.minimum(b, zero)))
    if name == "mc2":
        up = torch.maximum(zero, torch.minimum(0.5 * (a + b), torch.minimum(2 * b, 2 * a)))
        down = torch.minimum(zero, torch.maximum(0.5 * (a + b), torch.maximum(2 * b, 2 * a)))
        return torch.where(a > 0, up, down)
    s = (b * (a * a) + a * (b * b)) / (a * a + b * b + tiny)
    return torch.where(a * b < 0, zero, s) if name == "vanalbada2" else s


class _Gas:
    """Pressure, sound speed and enthalpy of a set of states in the solution basis."""

    def __init__(self, q, basis):
        if basis == "conserved":
            self.r = q[2]
            self.u, self.v = q[0] / q[2], q[1] / q[2]
            self.k = 0.5 * (self.u * self.u + self.v * self.v)
            self.p = (GAMMA - 1.0) * (q[3] - self.r * self.k)
        else:
            self.u, self.v, self.r, self.p = q[0], q[1], q[2], q[3]
            self.k = 0.5 * (self.u * self.u + self.v * self.v)
        self.a2 = GAMMA * self.p / self.r
        self.h = self.a2 / (GAMMA - 1.0) + self.k
        self.a = torch.sqrt(self.a2)

    def conserved(self):
        return torch.stack([self.r * self.u, self.r * self.v, self.r, self.r * self.h - self.p])


def _euler_flux(name, basis, minf, area, n0, n1, ql, qr):
    """(flux [4], spectral radius) times the area of faces with unit normal (n0, n1), left to right."""
    L, R = _Gas(ql, basis), _Gas(qr, basis)
    unl, unr = n0 * L.u + n1 * L.v, n0 * R.u + n1 * R.v
    nx = torch.stack([n0.expand_as(unl), n1.expand_as(unl), torch.zeros_like(unl), torch.zeros_like(unl)])
    if name in ("rusanov", "roe", "roe_faceframe"):
        fl = L.r * unl * torch.stack([L.u, L.v, torch.ones_like(unl), L.h]) + L.p * nx
        fr = R.r * unr * torch.stack([R.u, R.v, torch.ones_like(unr), R.h]) + R.p * nx
        lam = torch.maximum(unl.abs() + L.a, unr.abs() + R.a)
        dq = R.conserved() - L.conserved()
        if name == "rusanov":
            return (0.5 * (fl + fr) - 0.5 * lam * dq) * area, lam * area
        w = 1.0 / (1.0 + torch.sqrt(R.r / L.r))
        r = torch.sqrt(R.r / L.r) * L.r
        u, v, h = (w * x + (1.0 - w) * y for x, y in ((L.u, R.u), (L.v, R.v), (L.h, R.h)))
        k = 0.5 * (u * u + v * v)
        a2 = (GAMMA - 1.0) * (h - k)
        a = torch.sqrt(a2)
        un = n0 * u + n1 * v
        speeds = [un.abs()]
        for x, xl, xr in ((un - a, unl - L.a, unr - R.a), (un + a, unl + L.a, unr + R.a)):
            e = 0.05 * torch.clamp(torch.maximum(x - xl, xr - x), min=0.0)
            y = x.abs()
            speeds.append(torch.where(y > e, y, 0.5 * (e + y * y / e)))
        # the jump in the face frame; the plain Roe functor keeps the averaged velocity in the global frame
        uf, vf = (un, -n1 * u + n0 * v) if name == "roe_faceframe" else (u, v)
        d0, d1, dr, de = n0 * dq[0] + n1 * dq[1], -n1 * dq[0] + n0 * dq[1], dq[2], dq[3]
        du, dv = (d0 - uf * dr) / r, (d1 - vf * dr) / r
        dp = (GAMMA - 1.0) * (k * dr + de - uf * d0 - vf * d1)
        w0 = speeds[0] * GAMMA * (dp / a2 - dr) / r
        w1, w2, w3 = speeds[1] * (du - dp / (r * a)), speeds[2] * (du + dp / (r * a)), speeds[0] * dv
        dp = 0.5 * r * a * (w2 - w1)
        dr, du, dv = dp / a2 - r * w0 / GAMMA, 0.5 * (w1 + w2), w3
        d0, d1 = r * du + uf * dr, r * dv + vf * dr
        de = dp / (GAMMA - 1.0) + r * (uf * du + vf * dv) + k * dr
        fd = torch.stack([n0 * d0 - n1 * d1, n1 * d0 + n0 * d1, dr, de])
        return (0.5 * (fl + fr) - 0.5 * fd) * area, torch.maximum(lam, un.abs() + a) * area
    one = torch.ones_like(unl)
    if name == "slau":
        ua = torch.sqrt(L.k + R.k)
        a = 0.5 * (L.a + R.a)
        m, ml, mr = ua / a, unl / a, unr / a
        una = (L.r * unl.abs() + R.r * unr.abs()) / (L.r + R.r)
        chi = (1.0 - torch.minimum(one, m)) ** 2
        g = -torch.clamp(ml, -1.0, 0.0) * torch.clamp(mr, 0.0, 1.0)
        mdot = 0.5 * ((L.r * unl + R.r * unr - una * (R.r - L.r)) * (1.0 - g) - chi * (R.p - L.p) / a) * area
        bl = torch.where(ml.abs() > 1.0, one, 0.25 * (ml + 1.0) ** 2 * (2.0 - ml))
        br = torch.where(mr.abs() > 1.0, one, 0.25 * (mr - 1.0) ** 2 * (2.0 + mr))
        p = 0.5 * ((L.p + R.p) - (bl - br) * (R.p - L.p) + m * (bl + br - 1.0) * (L.p + R.p)) * area
        left = ua > 0
        lam = torch.maximum(L.a, R.a) + torch.maximum(unl.abs(), unr.abs())
    else:
        c = 2.0 * (GAMMA - 1.0) / (GAMMA + 1.0)
        al, ar = c * L.h / torch.maximum(unl, torch.sqrt(c * L.h)), c * R.h / torch.maximum(-unr, torch.sqrt(c * R.h))
        a = torch.minimum(al, ar)
        ml, mr = unl / a, unr / a
        r = 0.5 * (L.r + R.r)
        mm = 0.5 * (ml * ml + mr * mr)
        m0 = torch.clamp(torch.sqrt(mm), max=1.0)
        m0 = torch.maximum(m0, minf * one)
        fa = m0 * (2.0 - m0)
        supl, supr = ml.abs() > 1.0, mr.abs() > 1.0
        m2 = [0.25 * (ml + 1.0) ** 2, -0.25 * (ml - 1.0) ** 2, 0.25 * (mr + 1.0) ** 2, -0.25 * (mr - 1.0) ** 2]
        mp = torch.where(supl, 0.5 * (ml + ml.abs()), m2[0] * (1.0 - 2.0 * m2[1]))
        mn = torch.where(supr, 0.5 * (mr - mr.abs()), m2[3] * (1.0 + 2.0 * m2[2]))
        ua = a * (mp + mn - 0.25 * torch.clamp(1.0 - mm, min=0.0) * (R.p - L.p) / (fa * r * a * a)) * area
        al5 = 0.1875 * (5.0 * fa * fa - 4.0)
        pl = torch.where(supl, one, m2[0] * (2.0 - ml) - 16.0 * al5 * ml * m2[0] * m2[1])
        pr = torch.where(supr, one, m2[3] * (-2.0 - mr) + 16.0 * al5 * mr * m2[3] * m2[2])
        p = (pl * L.p + pr * R.p - 1.5 * pl * pr * r * fa * a * (unr - unl)) * area
        left = ua > 0
        mdot = ua * torch.where(left, L.r, R.r)
        amax = torch.sqrt(torch.maximum(a * a, torch.maximum(L.a2, R.a2)))
        lam = 0.5 * (m0 + 1.0) / fa * amax + torch.maximum(ua.abs(), torch.maximum(unl.abs(), unr.abs()))
    up = torch.stack([torch.where(left, L.u, R.u), torch.where(left, L.v, R.v), one, torch.where(left, L.h, R.h)])
    return mdot * up + p * nx, lam * area


class _Scheme:
    """Residual and time step of one case on [variable][i][j] tensors."""

    def __init__(self, c, nodes, bref, bc, minf, device):
        self.c, self.bc, self.minf, self.bref = c, bc, minf, bref
        x = torch.from_numpy(nodes).to(device)
        lo, hi = BOX.get(c["family"], (0.0, 0.0))
        self.cen = 0.25 * (x[:-1, :-1] + x[1:, :-1] + x[:-1, 1:] + x[1:, 1:])
        a, b = (x[1:, 1:] - x[:-1, :-1]), (x[:-1, 1:] - x[1:, :-1])
        self.vol = (0.125 * (a[..., 0] * b[..., 1] - a[..., 1] * b[..., 0])).abs()
        self.dirs = []
        for d in (0, 1):
            # node line l of direction d: face l lies between cells l - 1 and l
            p0, p1 = (x[:, :-1], x[:, 1:]) if d == 0 else (x[1:], x[:-1])
            t = p1 - p0
            area = t.norm(dim=-1)
            shift = torch.zeros(2, dtype=x.dtype, device=device)
            shift[d] = hi - lo
            self.dirs.append({"d": d, "area": area, "n": torch.stack([t[..., 1], -t[..., 0]]) / area, "mid": 0.5 * (p0 + p1),
                              "per": bc[2 * d] == PERIODIC, "shift": shift})
        X = torch.zeros(3, *self.vol.shape, dtype=x.dtype, device=device)
        for f in self.dirs:
            f["lo"], f["hi"] = (0, None) if f["per"] else (1, -1)   # node lines that hold two-sided faces
            cl, cr = self._sides(f, self.cen.movedim(-1, 0))
            if f["per"]:
                cl = cl.clone()
                cl.select(f["d"] + 1, 0).sub_(f["shift"].reshape(2, 1))
            f["dx"] = cr - cl
            dd = torch.stack([f["dx"][0] ** 2, f["dx"][0] * f["dx"][1], f["dx"][1] ** 2])
            X = X + self._add(f, dd, dd)
            if not f["per"]:
                # mirror points beyond the two sides
                ax = f["d"] + 1
                for k, e in ((0, 0), (-1, -1)):
                    X.select(ax, k).add_(dd.select(ax, e))
            line = [slice(None)] * 2
            line[f["d"]] = slice(f["lo"], f["area"].shape[f["d"]] - 1)
            f["farea"], f["fn"], mid = f["area"][tuple(line)], f["n"][:, line[0], line[1]], f["mid"][tuple(line)].movedim(-1, 0)
            f["dl"], f["dr"] = (mid - cl).norm(dim=0), (cr - mid).norm(dim=0)
        for f in self.dirs:
            for side, Xs in zip(("wl", "wr"), self._sides(f, X)):
                xx, xy, yy = Xs[0] - f["dx"][0] ** 2, Xs[1] - f["dx"][0] * f["dx"][1], Xs[2] - f["dx"][1] ** 2
                det = xx * yy - xy * xy
                f[side] = torch.stack([yy * f["fn"][0] - xy * f["fn"][1], xx * f["fn"][1] - xy * f["fn"][0]]) / det

    def _sides(self, f, q):
        """Left and right cells of a direction's two-sided faces."""
        ax = f["d"] + 1
        if f["per"]:
            return q.roll(1, ax), q
        n = q.shape[ax]
        return q.narrow(ax, 0, n - 1), q.narrow(ax, 1, n - 1)

    def _add(self, f, left, right):
        """Per cell: what its faces give it as their left cell and as their right cell."""
        ax = f["d"] + 1
        if f["per"]:
            return left.roll(-1, ax) + right
        pad = [0, 0, 0, 0]
        a, b = list(pad), list(pad)
        a[3 - 2 * f["d"]], b[2 - 2 * f["d"]] = 1, 1
        return torch.nn.functional.pad(left, a) + torch.nn.functional.pad(right, b)

    def _flux(self, area, n, ql, qr):
        if self.c["family"] == "scalar":
            unl, unr = n[0] * ql[0] + n[1] * ql[1], n[0] * qr[0] + n[1] * qr[1]
            lam = torch.maximum(unl.abs(), unr.abs())
            f = torch.stack([torch.zeros_like(unl), torch.zeros_like(unl), 0.5 * (unl * ql[2] + unr * qr[2])])
            return (f - 0.5 * lam * (qr - ql)) * area, lam * area
        return _euler_flux(self.c["flux"], self.c["basis"], self.minf, area, n[0], n[1], ql, qr)

    def _far(self, n, qi, qf):
        """Characteristic far field: the interior state where the flow leaves, else from the Riemann invariants."""
        basis = self.c["basis"]

        def turned(q):
            return torch.stack([n[0] * q[0] + n[1] * q[1], -n[1] * q[0] + n[0] * q[1], q[2], q[3]])

        I, F = _Gas(turned(qi), basis), _Gas(turned(qf), basis)
        w = 1.0 / (1.0 + torch.sqrt(F.r / I.r))
        u, v, h = (w * x + (1.0 - w) * y for x, y in ((I.u, F.u), (I.v, F.v), (I.h, F.h)))
        k = 0.5 * (u * u + v * v)
        ma = u / torch.sqrt((GAMMA - 1.0) * (h - k))
        minus, plus = I.u - 2.0 * I.a / (GAMMA - 1.0), F.u + 2.0 * F.a / (GAMMA - 1.0)
        ub, ab = 0.5 * (minus + plus), 0.25 * (GAMMA - 1.0) * (plus - minus)
        s = F.a2 / (GAMMA * F.r ** (GAMMA - 1.0))
        r = (ab * ab / (GAMMA * s)) ** (1.0 / (GAMMA - 1.0))
        g = torch.stack([ub, F.v, r, r * ab * ab / GAMMA])
        if basis == "conserved":
            g = _Gas(g, "primitive").conserved()
        g = torch.stack([n[0] * g[0] - n[1] * g[1], n[1] * g[0] + n[0] * g[1], g[2], g[3]])
        return torch.where(u / torch.sqrt(2.0 * k) < 0.001, qi, torch.where(ma.abs() > 1.0, qf, g))

    def residual(self, q):
        nv, ni, nj = q.shape
        R, lam = torch.zeros_like(q), torch.zeros_like(q[0])
        Q = None
        if self.c["limiter"] != "nolimit1":
            Q = torch.zeros(2, *q.shape, dtype=q.dtype, device=q.device)
            for f in self.dirs:
                ql, qr = self._sides(f, q)
                Q = Q + torch.stack([self._add(f, (qr - ql) * f["dx"][k], (qr - ql) * f["dx"][k]) for k in (0, 1)])
        for f in self.dirs:
            ql, qr = self._sides(f, q)
            if Q is not None:
                dq = qr - ql
                slopes = []
                for w, Qk in (("wl", 0), ("wr", 1)):
                    s = [self._sides(f, Q[k])[Qk] - dq * f["dx"][k] for k in (0, 1)]
                    slopes.append(_limited(self.c["limiter"], dq / (f["dl"] + f["dr"]), s[0] * f[w][0] + s[1] * f[w][1]))
                ql, qr = ql + slopes[0] * f["dl"], qr - slopes[1] * f["dr"]
            F, lf = self._flux(f["farea"], f["fn"], ql, qr)
            R = R + self._add(f, -F, F)
            lam = lam + self._add(f, lf[None], lf[None])[0]
            if not f["per"]:
                R, lam = self._boundaries(f, q, R, lam)
        return R, lam

    def _boundaries(self, f, q, R, lam):
        d, nv = f["d"], q.shape[0]
        ni, nj = q.shape[1:]
        for side in (0, 1):
            b = 2 * d + side
            line = -1 if side else 0
            area, n = f["area"].select(d, line), f["n"].select(d + 1, line)
            inward = -n if side else n
            qi = q.select(d + 1, line)
            if self.bc[b] == WALL:
                s = _Gas(qi, self.c["basis"])
                F = torch.stack([area * s.p * inward[0], area * s.p * inward[1], torch.zeros_like(area), torch.zeros_like(area)])
                lf = area * ((n[0] * s.u + n[1] * s.v).abs() + s.a)
            else:
                start = (0, nj, 2 * nj, 2 * nj + ni)[b]
                qf = self.bref[start:start + area.shape[0]].T
                g = self._far(inward, qi, qf) if self.bc[b] == RIEMANN else qf
                F, lf = self._flux(area, n, qi, g) if side else self._flux(area, n, g, qi)
                F = -F if side else F
            pad = [0, 0, 0, 0]
            pad[2 - 2 * d + (0 if side else 1)] = q.shape[d + 1] - 1
            R = R + torch.nn.functional.pad(F.unsqueeze(d + 1), pad)
            lam = lam + torch.nn.functional.pad(lf.unsqueeze(d), pad)
        return R, lam

    def step(self, q0):
        """(state after one step, its time step or None)."""
        alpha, beta = _rk(self.c["rk"])
        euler_primitive = self.c["family"] != "scalar" and self.c["basis"] == "primitive"
        c0 = _Gas(q0, "primitive").conserved() if euler_primitive else q0
        q, done, dt, lam0 = q0, [], None, None
        for s, row in enumerate(alpha):
            r, lam = self.residual(q)
            done.append(r)
            if s == 0:
                lam0 = lam
                dt = self.c["cfl"] / float((lam / self.vol).max()) if self.c["dt"] == "global" else None
            total = sum(a * x for a, x in zip(row, done) if a != 0.0)
            per = lam0 if self.c["dt"] == "local" else self.vol
            c1 = c0 + total * (beta[s] * (self.c["cfl"] if dt is None else dt) / per)
            if euler_primitive:
                g = _Gas(c1, "conserved")
                c1 = torch.stack([g.u, g.v, g.r, g.p])
            q = c1
        return q, dt


def _march(c, seed, member, device):
    nodes, q, ref, bc, minf = _problem(c, seed, member)
    scheme = _Scheme(c, nodes, torch.from_numpy(_bref(c, ref)).to(device), bc, minf, device)
    q = torch.from_numpy(q).to(device).permute(2, 0, 1).contiguous()
    first, t = scheme.residual(q)[0][2] / scheme.vol if c["family"] == "steady" else None, 0.0
    for _ in range(c["steps"]):
        q, dt = scheme.step(q)
        t += dt or 0.0
    return scheme, q, t, first


def exact(case, seed):
    device = "cuda:0" if torch.cuda.is_available() else "cpu"
    if case["family"] == "batch":
        with torch.no_grad():
            out = []
            for k, c in enumerate(_members(case)):
                _, ref = _freestream(np.random.default_rng([int(seed), k]))
                scheme = _Scheme(c, _ogrid(c["ni"], c["nj"]), torch.from_numpy(_bref(c, ref)).to(device),
                                 (WALL, RIEMANN, PERIODIC, PERIODIC), 0.0, device)
                q = torch.from_numpy(ref).to(device).reshape(4, 1, 1).expand(4, c["ni"], c["nj"])
                for _ in range(c["steps"]):
                    q, _ = scheme.step(q)
                out.append(q.reshape(-1))
            return {"q": torch.cat(out)}
    if case["family"] == "adjoint":
        c = _adjoint_single(case)
        nodes, q, ref, bc, minf = _problem(c, seed)
        q0 = torch.from_numpy(q).to(device).requires_grad_()
        bref = torch.from_numpy(_bref(c, ref)).to(device).requires_grad_()
        scheme = _Scheme(c, nodes, bref, bc, minf, device)
        q = q0.permute(2, 0, 1)
        for _ in range(c["steps"]):
            q = torch.utils.checkpoint.checkpoint(lambda x: scheme.step(x)[0], q, use_reentrant=False)
        qk = q.permute(1, 2, 0)
        w = torch.from_numpy(np.random.default_rng([int(seed), 77]).standard_normal(qk.shape)).to(device)
        grads = torch.autograd.grad(qk, (q0, bref), w)
        return {"q": qk.detach(), "q0_grad": grads[0], "bref_grad": grads[1]}
    with torch.no_grad():
        scheme, q, t, first = _march(case, seed, 0, device)
        out = {"q": q.permute(1, 2, 0).contiguous()}
        if case["family"] == "steady":
            last = scheme.residual(q)[0][2] / scheme.vol
            out["drop"] = float(last.square().mean().sqrt() / first.square().mean().sqrt())
        elif case["dt"] == "global":
            out["t"] = t
        return out
