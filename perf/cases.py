"""What is timed of this solver: whole timesteps, the pressure solve with the
projection that follows it, the flow kernels around it, the particle side of
a Lamb pass, and the network of the learned initial guess, each through the
entry points that a program calls (bbhip.Simulation and the C ABI of
include/bluebottle.h; the network's calls as bench.py makes them).

The library keeps its simulation in globals, so each state has a copy of the
library of its own: several runs can be held side by side.  Inputs are made
from the seed on the GPU, smooth velocity modes with a little noise, and
written into the library's arrays.
"""
import ctypes
import math
import os
import shutil
import sys
import tempfile

import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "bluebottle-3.0_amd"))

import bbconfig  # noqa: E402
import bbhip  # noqa: E402

F64 = torch.float64
DT = 1e-3                               # of the flow and solve cases
NET_STEPS = 4                           # Adam steps of a training pass
NET_RATE = 3e-4
# cin, cout, taps, level of the network's layers
NET = [(2, 16, 27, 0), (16, 16, 27, 0), (16, 32, 27, 1), (32, 32, 27, 1),
       (32, 64, 27, 2), (64, 64, 27, 2), (96, 32, 27, 1), (32, 32, 27, 1),
       (48, 16, 27, 0), (16, 16, 27, 0), (16, 1, 1, 0)]


def case(name, kind, flow, n, spheres=0, radius=0.0, precision="PLAIN",
         history=False):
    c = dict(kind=kind, flow=flow, nx=n[0], ny=n[1], nz=n[2],
             spheres=spheres, radius=radius, precision=precision,
             history=history)
    return dict(name=name, **c) if name else c


def listed():
    return [
        # a timestep of the smallest box a user runs (the smoke test's):
        # launches and host checks are all there is
        case("step_cavity_16", "step", "cavity", (16, 16, 16)),
        # a timestep of a small channel of odd sizes, which the row kernels
        # do not take
        case("step_channel_65x33x31", "step", "channel", (65, 33, 31)),
        # sedimentation at the default box of the input writer: eight
        # spheres, a Lamb loop of several pressure solves
        case("step_sediment_64", "step", "sediment", (64, 64, 64), 8, 6.0),
        # convection between hot and cold walls with the scalar transport
        case("step_convection_96x80x48", "step", "convection", (96, 80, 48)),
        # the benchmark's channel, with the mixed-precision solve
        case("step_channel_256_mixed", "step", "channel", (256, 128, 128),
             precision="MIXED"),
        # the benchmark's box: 500 spheres, mixed precision, the initial
        # guess from earlier solutions
        case("step_sediment_256_mixed", "step", "sediment", (256, 256, 256),
             500, 6.0, "MIXED", True),
        # one plain pressure solve with particles, and the projection
        case("solve_sediment_128", "solve", "sediment", (128, 128, 128), 62,
             6.0),
        # one mixed-precision solve of a singular, anisotropic, ragged grid
        case("solve_channel_150_mixed", "solve", "channel", (150, 130, 94),
             precision="MIXED"),
        # everything of a Lamb pass but the pressure solve, single phase
        case("flow_channel_256", "flow", "channel", (256, 256, 128)),
        # the particle side of a Lamb pass and of the end of a step
        case("particles_128", "particles", "sediment", (128, 128, 128), 90,
             6.0),
        # the network's inference on the coarse grid of a 256^3 box
        case("net_forward_128", "net_forward", "", (128, 128, 128)),
        # its training on 64^3 crops: forward, backward and Adam
        case("net_train_64", "net_train", "", (64, 64, 64)),
    ]


def draw(rng):
    def size(lo, hi, step=1):
        v = math.exp(rng.uniform(math.log(lo), math.log(hi + 0.99)))
        return max(step, int(v) // step * step)

    kind = rng.choice(["step", "step", "step", "solve", "solve", "flow",
                       "particles", "net_forward", "net_train"])
    if kind == "net_forward":
        return case("", kind, "", tuple(size(16, 128, 4) for _ in range(3)))
    if kind == "net_train":
        return case("", kind, "", tuple(size(16, 64, 4) for _ in range(3)))
    precision = rng.choice(["PLAIN", "MIXED"])
    flow = "sediment" if kind == "particles" else rng.choice(
        ["channel", "sediment"] if kind == "solve" else
        ["channel", "convection"] if kind == "flow" else
        ["cavity", "channel", "sediment", "sediment", "convection"])
    if kind == "flow":
        precision = "PLAIN"
    if flow == "cavity":
        return case("", kind, flow, tuple(size(12, 64) for _ in range(3)),
                    precision=precision)
    if flow == "convection":
        return case("", kind, flow, (size(32, 160), size(32, 128),
                                     size(24, 64)), precision=precision)
    if flow == "channel":
        return case("", kind, flow, (size(48, 256), size(32, 128),
                                     size(32, 128)), precision=precision)
    history = kind == "step" and precision == "MIXED" and rng.random() < 0.5
    step = 8 if history else 1
    n = tuple(size(48, 160, step) for _ in range(3))
    # radii that the grid resolves: runs with smaller ones diverge in time
    radius = rng.choice([6.0, 6.5, 7.0, 8.0])
    share = rng.uniform(0.005, 0.03) * n[0] * n[1] * n[2]
    return case("", kind, flow, n,
                max(1, int(share / (4 / 3 * math.pi * radius ** 3))), radius,
                "PLAIN" if kind == "particles" else precision, history)


# ------------------------------- set-up -----------------------------------
_idle = []                              # library copies no state holds


def _library():
    if _idle:
        return _idle.pop()
    torch.cuda.init()
    with tempfile.TemporaryDirectory(prefix="bb_lib_") as d:
        path = shutil.copy(bbhip.LIB_PATH, d)
        lib = ctypes.CDLL(path, mode=os.RTLD_LOCAL | os.RTLD_DEEPBIND)
    vp = ctypes.c_void_p
    lib.bb_unet_create.argtypes = [ctypes.c_ulonglong]
    lib.bb_unet_volume.argtypes = [ctypes.c_int] * 3
    lib.bb_unet_forward.argtypes = [vp, vp]
    lib.bb_unet_backward.argtypes = [vp]
    lib.bb_unet_backward.restype = ctypes.c_double
    lib.bb_unet_adam.argtypes = [ctypes.c_float]
    lib.bb_unet_get.argtypes = [ctypes.c_int, ctypes.c_int, vp]
    lib.cuda_exchange.argtypes = [vp, ctypes.c_int]
    lib.cuda_dom_BC_p.argtypes = [vp]
    return lib


class _Memory:
    """A device array of a state's library, for torch.as_tensor; the tensor
    keeps the state alive."""

    def __init__(self, state, ptr, shape, strides, kind="<f8"):
        self.state = state
        self.__cuda_array_interface__ = dict(
            data=(ptr, False), shape=tuple(shape), strides=tuple(strides),
            typestr=kind, version=2)


class State:
    """One simulation in a library copy of its own."""

    def __init__(self, c, config, parts):
        self.case = c
        self.n = config["n"]
        self.dir = tempfile.TemporaryDirectory(prefix="bb_case_")
        bbconfig.write_case(self.dir.name, **config)
        if parts:
            bbconfig.write_parts(self.dir.name, parts)
        self.lib = _library()
        bbhip._lib = self.lib
        self.sim = bbhip.Simulation(self.dir.name, self.n)
        # the guess's span of earlier solutions without the network
        ctypes.c_int.in_dll(self.lib, "bb_warm_use_net").value = 0
        self.sim.setup()
        self.views = {}

    def __del__(self):
        self.views = {}
        self.sim.teardown()
        _idle.append(self.lib)

    def ptr(self, name):
        return ctypes.c_void_p.in_dll(self.lib, name)

    def view(self, name, grid, ghosts=False):
        """Array `name` as a [k, j, i] tensor (rows are padded to 32)."""
        ptr = self.ptr(name).value
        key = (ptr, grid, ghosts)
        if key not in self.views:
            ib, jb, kb = (m + 2 for m in bbhip.grid_dims(grid, self.n))
            sy = (ib + 31) // 32 * 32
            t = torch.as_tensor(_Memory(_Weak(self), ptr, (kb, jb, ib),
                                        (8 * sy * jb, 8 * sy, 8)),
                                device="cuda")
            self.views[key] = t if ghosts else t[1:-1, 1:-1, 1:-1]
        return self.views[key]

    def out(self, name, grid):
        """`name`'s interior, for the caller: keeps this state alive."""
        t = self.view(name, grid)
        t = torch.as_tensor(_Memory(self, t.data_ptr(), t.shape,
                                    [8 * s for s in t.stride()]),
                            device="cuda")
        return t

    def parts(self):
        """The particles' motion, forces and Lamb coefficients."""
        P = bbhip.PartStruct
        size, n = ctypes.sizeof(P), self.case["spheres"]
        res = {}
        for what, lo, hi in (("motion", P.r.offset, P.nodes.offset),
                             ("coeffs", P.pnm_re.offset, P.pnm_re0.offset)):
            res[what] = torch.as_tensor(
                _Memory(self, self.ptr("_parts").value + lo,
                        (n, (hi - lo) // 8), (size, 8)), device="cuda")
        return res


class _Weak:
    """A state's own views must not keep it alive."""

    def __init__(self, state):
        pass


GRID = {"u": bbhip.GFX, "v": bbhip.GFY, "w": bbhip.GFZ, "p": bbhip.GCC}


def configuration(c, seed):
    """Input file values and spheres of a case."""
    n = (c["nx"], c["ny"], c["nz"])
    ext = {"pp_precision": c["precision"]}
    parts = None
    if c["flow"] == "cavity":
        kw = bbconfig.cavity(n=16, steps=10 ** 9)
        kw["n"] = n
        ext["fixed_dt"] = 1e-3
    elif c["flow"] == "channel":
        kw = bbconfig.channel(n=n)
        kw["init_cond"] = "QUIESCENT"   # the fields are written below
    elif c["flow"] == "convection":
        kw = bbconfig.rayleigh_benard(n=n)
    else:
        kw, parts = bbconfig.sediment(n=n, nparts=c["spheres"],
                                      a=c["radius"], seed=seed + 1)
    if c["kind"] != "step":
        ext["fixed_dt"] = DT
    if c["history"]:
        ext["pp_warmstart"] = "LEARNED"
    kw["extensions"] = ext
    return kw, parts


def periodic(kw):
    return tuple(kw["p_bc"][f][0] == "PERIODIC" for f in "WSB")


def spacing(kw):
    return tuple((kw["hi"][d] - kw["lo"][d]) / kw["n"][d] for d in range(3))


def smooth(gen, comp, kw, amp):
    """A velocity component (comp 0..2) or cell field (3) over the interior
    points, [k, j, i]: six modes of a few wavelengths per box with 2 % of
    noise; periodic duplicates equal."""
    n = kw["n"]
    dev = gen.device
    shape = [n[d] + (comp == d) for d in (2, 1, 0)]
    f = 0.02 * amp * torch.randn(shape, generator=gen, device=dev, dtype=F64)
    for _ in range(6):
        term = torch.ones((), device=dev, dtype=F64)
        k = torch.randint(0, 4, (3,), generator=gen, device=dev)
        ph = torch.rand(4, generator=gen, device=dev, dtype=F64)
        for d in range(3):
            x = torch.arange(n[d] + (comp == d), device=dev, dtype=F64)
            x = (x + (0.0 if comp == d else 0.5)) / n[d]
            s = [1, 1, 1]
            s[2 - d] = -1
            term = term * torch.cos(2 * math.pi * (k[d] * x + ph[d])).view(s)
        f += amp * (2 * ph[3] - 1) * term
    for d, per in enumerate(periodic(kw)):
        if per and comp == d:
            f.select(2 - d, n[d]).copy_(f.select(2 - d, 0))
    return f


# near rest with spheres, which start at rest too
AMPLITUDE = {"cavity": 0.3, "channel": 1.0, "sediment": 0.002,
             "convection": 0.05}


def inputs(c, kw, seed):
    """The fields a case starts from, interior points."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    amp = AMPLITUDE[c["flow"]]
    f = {q: smooth(gen, d, kw, amp) for d, q in enumerate("uvw")}
    if c["flow"] == "channel":          # the laminar profile
        z = (torch.arange(c["nz"], device="cuda", dtype=F64) + 0.5)
        z = z * spacing(kw)[2] - 1.0
        f["u"] = 0.2 * f["u"] + (90.0 * (1 - z * z)).view(-1, 1, 1)
    f["p"] = smooth(gen, 3, kw, amp * amp)
    if c["kind"] == "flow":
        f["phi"] = smooth(gen, 3, kw, amp * amp)
        for d, q in enumerate("uvw"):
            f["conv0_" + q] = smooth(gen, d, kw, amp)
            f["diff0_" + q] = smooth(gen, d, kw, amp)
    return f


# ------------------------------ prepare, run -------------------------------
def prepare(c, seed):
    if c["kind"].startswith("net_"):
        return Net(c, seed)
    kw, parts = configuration(c, seed)
    s = State(c, kw, parts)
    lib = s.lib
    f = inputs(c, kw, seed)
    lib.compute_vel_BC()                # walls at their speeds
    star = "_star" if c["kind"] == "solve" else ""
    for q in "uvw":
        s.view("_" + q + star, GRID[q]).copy_(f[q])
        lib.cuda_exchange(s.ptr("_" + q + star), GRID[q])
    if star:
        lib.cuda_dom_BC_star()
    lib.cuda_dom_BC()
    for q in "uvw":                     # the start of the step: u0 = u
        s.view("_" + q + "0", GRID[q], True).copy_(
            s.view("_" + q, GRID[q], True))
    if c["kind"] != "step":             # a start of a run has p = 0
        for p in ("_p", "_p0") + (("_phi",) if "phi" in f else ()):
            s.view(p, bbhip.GCC).copy_(f["phi" if p == "_phi" else "p"])
            lib.cuda_exchange(s.ptr(p), bbhip.GCC)
            lib.cuda_dom_BC_p(s.ptr(p))
    if c["kind"] == "flow":
        for q in "uvw":
            for h in ("conv0_", "diff0_"):
                s.view("_" + h + q, GRID[q]).copy_(f[h + q])
        s.sim.set_scalar("dt0", DT)
        lib.cuda_compute_forcing()
        if c["flow"] == "convection":
            lib.cuda_compute_boussinesq()
    lib.cuda_find_dt()
    return s


def run(s):
    return RUN[s.case["kind"]](s)


def _outputs(state, names, **more):
    o = {q: state.out("_" + q, GRID[q[-1]] if q[-1] in GRID else GRID[q[0]])
         for q in names}
    o.update(more)
    return o


def _run_step(s):
    """One timestep of a running simulation."""
    s.sim.step()
    more = {"dt": s.sim.scalar("dt")}
    if s.case["flow"] == "convection":
        more["s"] = s.out("_s", bbhip.GCC)
    if s.case["spheres"]:
        more.update(s.parts())
    # the history that the next step starts from is _conv0, _diff0
    return _outputs(s, ["u", "v", "w", "p", "conv0_u", "conv0_v", "conv0_w",
                        "diff0_u", "diff0_v", "diff0_w"], **more)


def _run_solve(s):
    """The pressure solve and the corrector that it is for."""
    lib, c = s.lib, s.case
    if c["precision"] == "MIXED":
        lib.cuda_PP_cg_mixed()
    elif c["spheres"]:
        lib.cuda_PP_cg()
    else:
        lib.cuda_PP_cg_noparts()
    lib.cuda_exchange(s.ptr("_phi"), bbhip.GCC)
    lib.cuda_dom_BC_p(s.ptr("_phi"))
    _corrector(s)
    return _outputs(s, ["u", "v", "w", "p"])


def _corrector(s):
    lib = s.lib
    lib.cuda_project()
    for q in "uvw":
        lib.cuda_exchange(s.ptr("_" + q), GRID[q])
    lib.cuda_dom_BC()
    for q in "uvw":
        lib.cuda_exchange(s.ptr("_" + q), GRID[q])
    lib.cuda_update_p()
    lib.cuda_dom_BC_p(s.ptr("_p"))
    lib.cuda_exchange(s.ptr("_p"), bbhip.GCC)


def _exchange_star(s):
    for q in "uvw":
        s.lib.cuda_exchange(s.ptr("_" + q + "_star"), GRID[q])


def _run_flow(s):
    """u*, its boundary values and solvability correction; projection and
    pressure update with the phi that the state holds."""
    lib = s.lib
    lib.cuda_U_star()
    _exchange_star(s)
    lib.cuda_dom_BC_star()
    _exchange_star(s)
    lib.cuda_solvability()
    lib.cuda_dom_BC_star()
    _exchange_star(s)
    _corrector(s)
    return _outputs(s, ["u_star", "v_star", "w_star", "conv_u", "conv_v",
                        "conv_w", "diff_u", "diff_v", "diff_w", "u", "v",
                        "w", "p"])


def _run_particles(s):
    """The calls of a Lamb pass that follow u* and the projection, and the
    new cages at the end of a step."""
    lib = s.lib
    err, num = ctypes.c_double(), ctypes.c_int()
    lib.cuda_part_BC_star()
    lib.cuda_part_BC()
    lib.cuda_part_p_fill()
    lib.cuda_move_parts_sub()
    lib.cuda_lamb()
    lib.cuda_lamb_err(ctypes.byref(err), ctypes.byref(num))
    lib.cuda_parts_internal()
    lib.cuda_build_cages()
    lib.cuda_PP_init_jacobi_preconditioner()
    return _outputs(s, ["u", "v", "w", "p", "u_star", "v_star", "w_star"],
                    err=err.value, **s.parts())


class Net:
    """The network of the learned guess and the data it is given."""

    def __init__(self, c, seed):
        self.case, self.dims = c, (c["nx"], c["ny"], c["nz"])
        self.lib = _library()
        self.lib.bb_unet_create(seed + 1)
        self.lib.bb_unet_volume(*self.dims)
        nv = math.prod(self.dims)
        gen = torch.Generator(device="cuda").manual_seed(seed)
        # a scaled defect and the fluid fraction, and a smooth target
        self.x = torch.randn(nv, 2, generator=gen, device="cuda")
        self.x[:, 1] = (torch.rand(nv, generator=gen, device="cuda") >
                        0.03).float()
        self.t = smooth(gen, 3, dict(n=self.dims, p_bc={
            f: ("PERIODIC",) for f in "WSB"}), 1.0).float().reshape(-1)
        self.y = torch.zeros(nv, device="cuda")
        self.weights = [torch.zeros(taps, -(-co // 16) * 16, -(-ci // 16) * 16)
                        for ci, co, taps, _ in NET]

    def __del__(self):
        self.lib.bb_unet_destroy()
        _idle.append(self.lib)

    def get(self):
        for l, w in enumerate(self.weights):
            self.lib.bb_unet_get(l, 0, w.data_ptr())
        return self.weights


def _run_net_forward(s):
    s.lib.bb_unet_forward(s.x.data_ptr(), s.y.data_ptr())
    return s.y


def _run_net_train(s):
    """Adam steps on one crop, as a training round takes them, and the
    weights that they lead to."""
    for _ in range(NET_STEPS):
        s.lib.bb_unet_forward(s.x.data_ptr(), s.y.data_ptr())
        s.lib.bb_unet_backward(s.t.data_ptr())
        s.lib.bb_unet_adam(NET_RATE)
    return {"y": s.y, "weights": s.get()}


RUN = {"step": _run_step, "solve": _run_solve, "flow": _run_flow,
       "particles": _run_particles, "net_forward": _run_net_forward,
       "net_train": _run_net_train}


# ------------------------------ work, tolerance ----------------------------
def work(c):
    cells = c["nx"] * c["ny"] * c["nz"]
    kind = c["kind"]
    if kind.startswith("net_"):
        flops = sum(2 * taps * ci * co * cells / 8 ** lv
                    for ci, co, taps, lv in NET)
        nw = sum(taps * ci * co for ci, co, taps, _ in NET)
        if kind == "net_forward":
            return {"bytes": 12 * cells + 2 * nw, "flops": flops}
        # forward, backward data and weight gradient; Adam's three arrays
        return {"bytes": NET_STEPS * (16 * cells + 28 * nw),
                "flops": 3 * NET_STEPS * flops}
    if kind == "step":      # u, v, w, p and both histories in and out
        arrays = 20 + (6 if c["flow"] == "convection" else 0)
        return {"bytes": 8 * arrays * cells, "flops": 300 * cells}
    if kind == "solve":     # u*, p0 in; u, v, w, p out
        return {"bytes": 64 * cells, "flops": 60 * cells}
    if kind == "flow":      # u0, p0, phi, histories in; star, conv, diff, u out
        return {"bytes": (8 * (11 + 13) + 4) * cells, "flops": 200 * cells}
    # faces and cells of the cages, and the mask, flags and p they change
    return {"bytes": (3 * 4 + 2 * 4 + 1) * cells + 3128 * 2 * c["spheres"],
            "flops": 3000 * c["spheres"] * c["radius"] ** 2}


def tolerance(c):
    """About four times what correct variants of the same precision differ
    by after one or two passes: the mixed solve with other inner tolerances
    and restarts against the plain one, and each against exact().  A solve
    ends anywhere in the ball of its stopping test, (r, M^-1 r) <= 1e-16
    (b, b); without spheres the pressure's longest waves are free in it."""
    kind, flow = c["kind"], c["flow"]
    if kind == "net_forward":           # 16-bit weights and activations
        return {"rel": 3e-3, "max": 0.06}
    if kind == "net_train":             # and Adam's steps on their gradients
        return {"rel": 0.02, "max": 0.5}
    if kind == "flow":                  # 64-bit stencils, no reduction
        return {"rel": 1e-12}
    if kind == "particles":             # and sin, cos, acos of the device
        return {"rel": 1e-9}
    if flow == "sediment":
        return {"rel": 2e-6}
    if kind == "solve":
        return {"rel": 2e-5}
    if flow == "cavity":
        return {"rel": 1e-5}
    return {"rel": 5e-3 if c["precision"] == "MIXED" else 1e-4}


# --------------------------------- exact -----------------------------------
class Reference:
    """The single-phase step in torch, 64 bits: fields are [k, j, i] with
    one ghost layer."""

    def __init__(self, c, kw):
        self.c, self.kw = c, kw
        self.n, self.h, self.per = kw["n"], spacing(kw), periodic(kw)
        self.nu, self.rho = kw["nu"], kw["rho_f"]

    def pad(self, f):
        g = torch.zeros([m + 2 for m in f.shape], device=f.device, dtype=F64)
        g[1:-1, 1:-1, 1:-1] = f
        return g

    @staticmethod
    def at(f, axis, i):
        """Plane i across `axis`, interior points of the other two."""
        ix = [slice(1, -1)] * 3
        ix[axis] = i
        return f[tuple(ix)]

    def wrap(self, f, comp):
        for d in range(3):
            if not self.per[d]:
                continue
            a, e, o = 2 - d, f.shape[2 - d] - 2, int(comp == d)
            self.at(f, a, 0).copy_(self.at(f, a, e - o))
            self.at(f, a, e + 1).copy_(self.at(f, a, 1 + o))
        return f

    def bc(self, f, comp):
        """Walls: comp 0..2 a velocity component, 3 a Neumann cell field."""
        for d in range(3):
            if self.per[d]:
                continue
            a, e = 2 - d, f.shape[2 - d] - 2
            for g, s0, s1, face in ((0, 1, 2, "WSB"[d]),
                                    (e + 1, e, e - 1, "ENT"[d])):
                if comp == 3:
                    self.at(f, a, g).copy_(self.at(f, a, s0))
                    continue
                v = self.kw["vel_bc"]["uvw"[comp]][face][1]
                if comp == d:
                    self.at(f, a, g).copy_(2 * v - self.at(f, a, s1))
                    self.at(f, a, s0).fill_(v)
                else:
                    self.at(f, a, g).copy_(8 / 3 * v - 2 * self.at(f, a, s0)
                                           + self.at(f, a, s1) / 3)
        return f

    def sh(self, f, comp, off):
        """Interior of component grid `comp` of the field f shifted by `off`
        (x, y, z)."""
        ix = []
        for d in (2, 1, 0):
            m = self.n[d] + (comp == d)
            ix.append(slice(1 + off[d], 1 + off[d] + m))
        return f[tuple(ix)]

    def star(self, vel, p, comp, dt, dt0, conv0, diff0, sfield=None):
        c, ih = comp, [1 / h for h in self.h]
        e = [[int(a == b) for a in range(3)] for b in range(3)]

        def u(q, *offs):
            o = [sum(x) for x in zip(*offs)] if offs else [0, 0, 0]
            return self.sh(vel[q], c, o)

        def m(v):
            return [-x for x in v]

        me = u(c)
        conv = torch.zeros_like(me)
        diff = torch.zeros_like(me)
        for d in range(3):
            up, dn = u(c, e[d]), u(c, m(e[d]))
            if d == c:
                t = (up + me) ** 2 - (me + dn) ** 2
            else:
                t = ((up + me) * (u(d, e[d]) + u(d, e[d], m(e[c]))) -
                     (me + dn) * (u(d) + u(d, m(e[c]))))
            conv += 0.25 * ih[d] * t
            diff += (up - 2 * me + dn) * ih[d] ** 2
        diff *= self.nu
        grad = (self.sh(p, c, m(e[c])) - self.sh(p, c, [0, 0, 0])) * ih[c]
        s = grad / self.rho - self.kw.get("gradP", [(0., 0.)] * 3)[c][0] / \
            self.rho
        if dt0 > 0:
            b = 0.5 * dt / dt0
            s = s - (1 + b) * conv + b * conv0 + (1 + b) * diff - b * diff0
        else:
            s = s - conv + diff
        if sfield is not None:
            sc = self.kw["scalar"]
            face = 0.5 * (self.sh(sfield, c, m(e[c])) +
                          self.sh(sfield, c, [0, 0, 0]))
            s = s - self.kw["g"][c][0] * sc["s_beta"] * (face - sc["s_ref"])
        return me + dt * s, conv, diff

    def solvable(self, st):
        """The net flux through each pair of faces, taken off in halves."""
        for d in range(3):
            a, e = 2 - d, st[d].shape[2 - d] - 2
            lo, hi = self.at(st[d], a, 1), self.at(st[d], a, e)
            eps = 0.5 * (hi.mean() - lo.mean())
            lo += eps
            hi -= eps

    def basis(self, n, per):
        """Orthonormal eigenvectors (columns) and eigenvalues of the 1-D
        second difference, sign reversed."""
        i = torch.arange(n, device="cuda", dtype=F64).view(-1, 1)
        k = torch.arange(n, device="cuda", dtype=F64).view(1, -1)
        if not per:
            q = torch.cos(math.pi * (i + 0.5) * k / n) * math.sqrt(2 / n)
            q[:, 0] /= math.sqrt(2)
            return q, 2 - 2 * torch.cos(math.pi * k[0] / n)
        half = torch.floor((k + 1) / 2)
        arg = 2 * math.pi * half * i / n
        q = torch.where(k % 2 == 1, torch.cos(arg), torch.sin(arg))
        q[:, 0] = 1
        q = q / q.norm(dim=0)
        return q, 2 - 2 * torch.cos(2 * math.pi * half[0] / n)

    def poisson(self, b):
        """phi of -lap phi = b with zero mean, by its eigenvectors."""
        lam = 0
        qs = []
        for d in range(3):
            q, ev = self.basis(self.n[d], self.per[d])
            qs.append(q)
            s = [1, 1, 1]
            s[2 - d] = -1
            lam = lam + (ev / self.h[d] ** 2).view(s)
        lam = lam.clone()
        lam[0, 0, 0] = 1

        def along(f, way):
            for d in range(3):
                f = f.movedim(2 - d, 2)
                q = qs[d] if way else qs[d].t().contiguous()
                f = torch.matmul(f.reshape(-1, f.shape[2]).contiguous(), q
                                 ).reshape(f.shape).movedim(2, 2 - d)
            return f

        f = along(b, True) / lam
        f[0, 0, 0] = 0
        return along(f, False)

    def masked_poisson(self, b, fluid):
        """The same in the fluid cells with phi = 0 in the others: CG far
        past the solver's own test."""
        def lap(x):
            y = torch.zeros_like(x)
            for d in range(3):
                a = 2 - d
                y += (2 * x - x.roll(1, a) - x.roll(-1, a)) / self.h[d] ** 2
            return y * fluid

        x = torch.zeros_like(b)
        r = b * fluid
        p, rr = r.clone(), (r * r).sum()
        stop = 1e-26 * float(rr)
        for it in range(4000):
            ap = lap(p)
            alpha = rr / (p * ap).sum()
            x += alpha * p
            r -= alpha * ap
            new = (r * r).sum()
            if it % 20 == 0 and float(new) <= stop:
                break
            p = r + (new / rr) * p
            rr = new
        return x

    def divergence(self, st):
        b = 0
        for d in range(3):
            o = [int(a == d) for a in range(3)]
            b = b + (self.sh(st[d], 3, o) -
                     self.sh(st[d], 3, [0, 0, 0])) / self.h[d]
        return b

    def correct(self, st, p0, phi, dt, fluid=None):
        """u, v, w and p from u* and phi (interior)."""
        ph = self.bc(self.wrap(self.pad(phi), 3), 3)
        vel = []
        for d in range(3):
            o = [-int(a == d) for a in range(3)]
            grad = (self.sh(ph, d, [0, 0, 0]) - self.sh(ph, d, o)) / self.h[d]
            if not self.per[d]:
                for i in (0, -1):
                    grad.select(2 - d, i).zero_()
            f = self.pad(self.sh(st[d], d, [0, 0, 0]) - dt / self.rho * grad)
            vel.append(self.wrap(self.bc(self.wrap(f, d), d), d))
        p = p0 + phi
        if fluid is not None:
            p = p * fluid
        return vel, p - p.mean()

    def predict(self, vel, p, dt, dt0, hist, sfield=None):
        st, conv, diff = [], [], []
        for d in range(3):
            s, cv, df = self.star(vel, p, d, dt, dt0, *hist[d], sfield)
            st.append(self.pad(s))
            conv.append(cv)
            diff.append(df)

        def edges():
            for d in range(3):
                self.wrap(self.bc(self.wrap(st[d], d), d), d)

        edges()
        self.solvable(st)
        edges()
        return st, conv, diff

    def time_step(self, vel):
        if "fixed_dt" in self.kw["extensions"]:
            return self.kw["extensions"]["fixed_dt"]
        nu = self.nu
        if self.c["flow"] == "convection":
            nu = max(nu, self.kw["scalar"]["s_D"])
        top = [float(self.sh(vel[d], d, [0, 0, 0]).abs().max())
               for d in range(3)]
        return self.kw["CFL"] / sum(t / h + 2 * nu / h ** 2
                                    for t, h in zip(top, self.h))

    def scalar_bc(self, s):
        for g, i, v in ((0, 1, 0.5), (s.shape[0] - 1, -2, -0.5)):
            self.at(s, 0, g).copy_(2 * v - self.at(s, 0, i))
        return self.wrap(s, 3)

    def scalar(self, s, vel, dt):
        """One Euler step of the flux form."""
        D = self.kw["scalar"]["s_D"]
        me, rate = self.sh(s, 3, [0, 0, 0]), 0
        for d in range(3):
            o = [int(a == d) for a in range(3)]
            up, dn = self.sh(s, 3, o), self.sh(s, 3, [-x for x in o])
            hi = self.sh(vel[d], 3, o)
            lo = self.sh(vel[d], 3, [0, 0, 0])
            rate = rate - (hi * 0.5 * (up + me) -
                           lo * 0.5 * (me + dn)) / self.h[d] + \
                D * (up - 2 * me + dn) / self.h[d] ** 2
        return me + dt * rate


def exact(c, seed):
    if c["kind"].startswith("net_"):
        return exact_net(c, seed)
    # no plain form of the particle path (Lamb series, quadrature, cages)
    # that is not a second solver
    if c["kind"] == "particles" or (c["kind"] == "step" and c["spheres"]):
        return None
    kw, parts = configuration(c, seed)
    R = Reference(c, kw)
    f = inputs(c, kw, seed)
    vel = [R.bc(R.wrap(R.pad(f[q]), d), d) for d, q in enumerate("uvw")]
    inner = [slice(1, -1)] * 3

    def out(names, arrays, **more):
        o = dict(zip(names, arrays))
        o.update(more)
        return o

    def whole(fields):
        return [g[tuple(inner)] for g in fields]

    if c["kind"] == "solve":
        b = -R.rho / DT * R.divergence(vel)
        fluid = None
        if c["spheres"]:
            fluid = fluid_cells(kw, parts)
            phi = R.masked_poisson(b, fluid)
        else:
            phi = R.poisson(b)
        vel, p = R.correct(vel, f["p"], phi, DT, fluid)
        return out("uvwp", whole(vel) + [p])
    dt = R.time_step(vel)
    zero = [(0.0, 0.0)] * 3
    sfield = None
    if c["flow"] == "convection":
        sfield = R.scalar_bc(R.pad(initial_scalar(kw)))
    if c["kind"] == "flow":
        p = R.bc(R.wrap(R.pad(f["p"]), 3), 3)
        hist = [(f["conv0_" + q], f["diff0_" + q]) for q in "uvw"]
        st, conv, diff = R.predict(vel, p, dt, DT, hist, sfield)
        vel, p = R.correct(st, f["p"], f["phi"], dt)
        return out(["u_star", "v_star", "w_star", "conv_u", "conv_v",
                    "conv_w", "diff_u", "diff_v", "diff_w", "u", "v", "w",
                    "p"], whole(st) + conv + diff + whole(vel) + [p])
    st, conv, diff = R.predict(vel, torch.zeros_like(R.pad(f["p"])), dt, 0.0,
                               zero, sfield)
    phi = R.poisson(-R.rho / dt * R.divergence(st))
    new, p = R.correct(st, torch.zeros_like(f["p"]), phi, dt)
    more = {"dt": R.time_step(new)}
    if sfield is not None:
        more["s"] = R.scalar(sfield, vel, dt)
    return out(["u", "v", "w", "p", "conv0_u", "conv0_v", "conv0_w",
                "diff0_u", "diff0_v", "diff0_w"],
               whole(new) + [p] + conv + diff, **more)


def initial_scalar(kw):
    """The scalar's seeded noise: the C library generator, seeded with each
    cell's index in the ghosted grid."""
    libc = ctypes.CDLL(None)
    s0, amp = kw["scalar"]["init_s"]
    nx, ny, nz = kw["n"]
    f = torch.empty(nz, ny, nx, dtype=F64)
    for k in range(nz):
        rows = []
        for j in range(ny):
            base = (nx + 2) * (j + 1 + (ny + 2) * (k + 1)) + 1
            for i in range(nx):
                libc.srand(base + i)
                rows.append(libc.rand())
        f[k] = torch.tensor(rows, dtype=F64).view(ny, nx)
    return (s0 + amp * (2.0 * f / 2147483647.0 - 1.0)).cuda()


def fluid_cells(kw, parts):
    """1.0 in cells whose centre lies outside every sphere (periodic box of
    unit cells)."""
    n = kw["n"]
    fluid = torch.ones(n[2], n[1], n[0], device="cuda", dtype=F64)
    for P in parts:
        d2 = 0
        for d, q in enumerate("xyz"):
            x = torch.arange(n[d], device="cuda", dtype=F64) + 0.5 - P[q]
            x = x - n[d] * torch.round(x / n[d])
            s = [1, 1, 1]
            s[2 - d] = -1
            d2 = d2 + (x * x).view(s)
        fluid[torch.sqrt(d2) < P["r"]] = 0.0
    return fluid


def exact_net(c, seed):
    """The network, its gradients and Adam in 64 bits without the 16-bit
    rounding of weights and activations."""
    s = Net(c, seed)
    nx, ny, nz = s.dims
    train = c["kind"] == "net_train"
    W = [w[:, :co, :ci].to("cuda", F64).requires_grad_(train)
         for w, (ci, co, _, _) in zip(s.get(), NET)]
    B = [torch.zeros(co, device="cuda", dtype=F64, requires_grad=train)
         for _, co, _, _ in NET]

    def conv(l, x):                     # x: [z, y, x, channel]
        z, y, xx, ci = x.shape
        if NET[l][2] == 1:
            return x.reshape(-1, ci) @ W[l][0].t() + B[l]
        xp = torch.nn.functional.pad(x, (0, 0, 1, 1, 1, 1, 1, 1))
        o = B[l]
        for tap in range(27):
            a, b, d = tap % 3, tap // 3 % 3, tap // 9
            part = xp[d:d + z, b:b + y, a:a + xx].reshape(-1, ci)
            o = o + part @ W[l][tap].t()
        return torch.relu(o).reshape(z, y, xx, -1)

    def pool(x):
        z, y, xx, ch = x.shape
        return x.reshape(z // 2, 2, y // 2, 2, xx // 2, 2, ch).mean((1, 3, 5))

    def up(x):
        for a in range(3):
            x = x.repeat_interleave(2, a)
        return x

    def forward():
        x = s.x.double().reshape(nz, ny, nx, 2)
        e0 = conv(1, conv(0, x))
        e1 = conv(3, conv(2, pool(e0)))
        b = conv(5, conv(4, pool(e1)))
        d1 = conv(7, conv(6, torch.cat([up(b), e1], 3)))
        d0 = conv(9, conv(8, torch.cat([up(d1), e0], 3)))
        return conv(10, d0).reshape(-1)

    if not train:
        with torch.no_grad():
            return forward()
    par = W + B
    m = [torch.zeros_like(p) for p in par]
    v = [torch.zeros_like(p) for p in par]
    for step in range(1, NET_STEPS + 1):
        y = forward()
        loss = 0.5 * ((y - s.t.double()) ** 2).mean()
        grads = torch.autograd.grad(loss, par)
        with torch.no_grad():
            for p, g, a, b in zip(par, grads, m, v):
                a.mul_(0.9).add_(g, alpha=0.1)
                b.mul_(0.999).add_(g * g, alpha=0.001)
                p -= NET_RATE * (a / (1 - 0.9 ** step)) / (
                    torch.sqrt(b / (1 - 0.999 ** step)) + 1e-8)
    full = []
    for w, z in zip(W, s.weights):
        z = torch.zeros(z.shape, dtype=F64)
        z[:, :w.shape[1], :w.shape[2]] = w.detach().cpu()
        full.append(z)
    return {"y": y.detach(), "weights": full}
