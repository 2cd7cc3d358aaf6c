"""The V-cycle that preconditions the mixed form's sweeps on large grids
(bb_mg.h) against the Jacobi factor: the same timestep with both.  Grids whose
levels take every path of the level kernels: runs of four cells and single
ones, tiles that end inside a run, each combination of coarsened directions
that a spacing can ask for, walls and periodic faces, a last level of more than
4096 cells, more partials than tiles, particles."""
import ctypes

import numpy as np
import pytest

import bbconfig
import bbhip
from helpers import bitwise_equal

pytestmark = pytest.mark.gpu


def box(n, per, h):
    """Walls, one of them moving, where a direction is not periodic."""
    P = ("PERIODIC",)
    face = {f: P if per["WESNBT".index(f) // 2] else None for f in "WESNBT"}
    wall = ("DIRICHLET", 0.0, 0.0)
    vel = {c: {f: face[f] or wall for f in "WESNBT"} for c in "uvw"}
    for c, f in (("v", "T"), ("w", "E"), ("u", "N")):
        if not face[f]:
            vel[c][f] = ("DIRICHLET", 0.4, 0.0)
    return dict(n=n, lo=(0.0, 0.0, 0.0),
                hi=tuple(a * m for a, m in zip(h, n)), rho_f=1.0, nu=0.01,
                duration=1.0, pp_max_iter=100000, pp_residual=1e-8,
                p_bc={f: face[f] or ("NEUMANN", 0.0) for f in "WESNBT"},
                vel_bc=vel, init_cond="QUIESCENT",
                extensions={"fixed_dt": 1e-3, "perturb": (7, 0.2),
                            "pp_precision": "MIXED"})


def run(case_dir, kw, parts, mg):
    lib = bbhip.load()
    on = ctypes.c_int.in_dll(lib, "bb_mg")
    saved = on.value
    on.value = mg
    try:
        bbconfig.write_case(case_dir, **kw)
        if parts:
            bbconfig.write_parts(case_dir, parts)
        with bbhip.Simulation(case_dir, kw["n"]) as s:
            s.step()
            s.pull()
            return dict(
                s.pp_stats(), dt=s.scalar("dt"),
                levels=ctypes.c_int.in_dll(lib, "bb_mg_last").value,
                **{f: np.array(s.field(f)) for f in ("u", "v", "w", "phi")})
    finally:
        on.value = saved


def inner(a, n):
    """The cells (faces) of the domain, without the ghosts."""
    lo = [(s - m) // 2 for s, m in zip(a.shape, n)]
    return a[tuple(slice(l, l + m) for l, m in zip(lo, n))]


def difference_bound(out, h, low):
    """Both solves leave residuals with (r, D^-1 r) <= 1e-16 (b, b), so their
    difference e has A e = r1 - r2 and (A e, e) <= (2e-8)^2 (b, b) / low, low
    the smallest eigenvalue of D^-1 A (without the constant).  The velocities
    differ by dt / rho times the differences of e, whose squares sum to
    (A e, e)."""
    return out["dt"] * 2e-8 * np.sqrt(out["sp_rhs"] / low)


def velocity_difference(a, b, n):
    return np.sqrt(sum(np.sum((inner(a[f], n) - inner(b[f], n)) ** 2)
                       for f in "uvw"))


@pytest.mark.parametrize("n,per,h,levels", [
    ((128, 96, 96), (1, 1, 1), (1.0, 1.0, 1.0), 4),
    ((216, 72, 72), (0, 1, 0), (1.0, 0.8, 1.2), 4),
    ((200, 200, 28), (0, 0, 1), (1.0, 1.0, 1.0), 4),
    ((129, 96, 96), (1, 0, 0), (20.0, 1.0, 1.0), 5),
    ((64, 256, 72), (1, 0, 1), (1.0, 0.2, 1.0), 6),
    ((512, 48, 48), (1, 1, 0), (0.2, 1.0, 1.0), 6),
    ((48, 48, 512), (0, 0, 0), (1.0, 0.45, 0.2), 5),
    ((130, 96, 96), (1, 1, 1), (1.0, 1.0, 1.0), 0),
    ((100, 96, 96), (1, 0, 1), (1.0, 1.0, 1.0), 4),
    ((64, 8, 1024), (1, 1, 1), (1.0, 8.0, 1.0), 5),
    ((64, 64, 64), (1, 1, 1), (1.0, 1.0, 1.0), 0)])
def test_same_step(case_dir, n, per, h, levels):
    """levels: 0 where Jacobi stays (sizes with too few factors of two, no more
    than 2^18 cells)."""
    kw = box(n, per, h)
    ref, out = run(case_dir, kw, None, 0), run(case_dir, kw, None, 1)
    print("levels", out["levels"], "iterations", ref["niter"], out["niter"])
    assert ref["levels"] == 0 and bool(out["levels"]) == bool(levels)
    if not levels:
        assert ref["niter"] == out["niter"]
        return
    assert out["levels"] == levels
    assert out["resid"] <= 1e-8 and out["niter"] <= 30 < ref["niter"]
    c = [1.0 / a ** 2 for a in h]
    low = min((2 - 2 * np.cos((2 if p else 1) * np.pi / m)) * a
              for a, m, p in zip(c, n, per)) / (2 * sum(c))
    assert velocity_difference(ref, out, n) <= difference_bound(out, h, low)
    # the constant that the singular system leaves open: the mean of D phi is
    # 0 in both, to the FP32 rounding of the sweeps' phi (8 units)
    D = sum(a * np.where(
        (np.arange(m) % (m - 1) == 0) & (not p), 1.0, 2.0).reshape(
            [-1 if d == i else 1 for d in range(3)])
        for i, (a, m, p) in enumerate(zip(c, n, per)))
    for s in (ref, out):
        phi = inner(s["phi"], n)
        assert abs(np.sum(D * phi)) <= 8 * 2.0 ** -24 * np.sum(D * np.abs(phi))


@pytest.mark.parametrize("n,per,h", [
    ((1153, 2, 128), (1, 1, 1), (16.0, 16.0, 1.0)),
    ((1153, 2, 128), (0, 0, 0), (16.0, 16.0, 1.0)),
    ((2, 1153, 128), (1, 0, 1), (16.0, 16.0, 1.0)),
    ((2, 128, 1153), (0, 1, 1), (16.0, 1.0, 16.0)),
    ((128, 2, 1027), (1, 1, 0), (1.0, 16.0, 16.0))])
def test_long_last_level(case_dir, n, per, h):
    """A last level of more than 1024 cells in one direction (1153 x 2 x 4 and
    its like), against the plain form: FP32 sweeps with the Jacobi factor
    stall on such boxes.  Their condition number is up to 1.6e6 on the last
    level; its polynomial of degree 32 leaves 1 / (4 32^2) of it, 400, which
    is some 190 iterations (sqrt(400) / 2 times ln(2e8))."""
    kw = box(n, per, h)
    out = run(case_dir, kw, None, 1)
    kw["extensions"]["pp_precision"] = "PLAIN"
    ref = run(case_dir, kw, None, 1)
    print("levels", out["levels"], "iterations", ref["niter"], out["niter"])
    assert out["levels"] > 1
    assert out["resid"] <= 1e-8 and out["niter"] <= 200
    c = [1.0 / a ** 2 for a in h]
    low = min((2 - 2 * np.cos((2 if p else 1) * np.pi / m)) * a
              for a, m, p in zip(c, n, per)) / (2 * sum(c))
    assert velocity_difference(ref, out, n) <= difference_bound(out, h, low)


@pytest.mark.parametrize("n,walls", [((128, 96, 96), ""), ((144, 96, 80), "z")])
def test_same_step_particles(case_dir, n, walls):
    """Particle cells masked on every level.  The smallest eigenvalue is that
    of absorbing spheres in a box, at least the one of a single sphere: 4 pi a
    / V (its capacity), over 6 for D^-1.  Twice the bound for the particles'
    answer to the difference."""
    a = 8.0
    kw, parts = bbconfig.sediment(n=n, nparts=3, a=a, seed=13, walls=walls)
    for P, c in zip(parts, ((20., 20., 20.), (64., 50., 53.), (94., 70., 45.))):
        P.update(x=c[0], y=c[1], z=c[2])
    kw["extensions"] = {"pp_precision": "MIXED"}
    assert run(case_dir, kw, parts, 1)["levels"] == 0       # on request only
    ref, out = run(case_dir, kw, parts, 0), run(case_dir, kw, parts, 2)
    print("levels", out["levels"], "iterations", ref["niter"], out["niter"])
    assert ref["levels"] == 0 and out["levels"] > 1
    assert out["resid"] <= 1e-8 and out["niter"] <= 30 < ref["niter"]
    low = 4 * np.pi * a / np.prod(n) / 6
    assert velocity_difference(ref, out, n) <= \
        2 * difference_bound(out, (1., 1., 1.), low)


def test_steps_with_moving_particles(case_dir):
    """Three timesteps with spheres that move by part of a cell in each: the
    levels' masks follow, and the same bits come out where the solver's buffers
    are freed before each step (void bb_solver_free(void)), which builds the
    levels anew."""
    lib = bbhip.load()
    on = ctypes.c_int.in_dll(lib, "bb_mg")
    free = getattr(lib, "_Z14bb_solver_freev")
    kw, parts = bbconfig.sediment(n=(80, 64, 64), nparts=2, a=8.0, seed=13)
    for P, c, v in zip(parts, ((20., 20., 20.), (60., 40., 45.)), (0.3, -0.3)):
        P.update(x=c[0], y=c[1], z=c[2], u=v, w=v)
    kw["extensions"] = {"pp_precision": "MIXED"}
    out, saved = [], on.value
    on.value = 2
    try:
        for anew in (0, 1):
            bbconfig.write_case(case_dir, **kw)
            bbconfig.write_parts(case_dir, parts)
            with bbhip.Simulation(case_dir, kw["n"]) as s:
                steps, phase = [], []
                for _ in range(3):
                    if anew:
                        s.sync()
                        free()
                    s.step()
                    st = s.pp_stats()
                    assert ctypes.c_int.in_dll(lib, "bb_mg_last").value == 4
                    assert st["resid"] <= 1e-8 and st["niter"] <= 30
                    s.pull()
                    phase.append(np.array(s.field("phase")) >= 0)
                    steps.append({f: np.array(s.field(f))
                                  for f in ("u", "v", "w", "phi")})
                    steps[-1]["niter"] = st["niter"]
                assert all((a != b).any() for a, b in zip(phase, phase[1:]))
            out.append(steps)
    finally:
        on.value = saved
    for a, b in zip(*out):
        assert a["niter"] == b["niter"]
        for f in ("u", "v", "w", "phi"):
            assert bitwise_equal(a[f], b[f]), f


def test_steps_warm_start(case_dir):
    """Three timesteps from earlier solutions (the guess without its network)
    with the V-cycle and with the Jacobi factor.  Each solve leaves a velocity
    difference B (difference_bound) and one in dt / rho grad p, which the next
    steps start from: n B of the n steps before, so 1 + 2 + 3 B after three
    (seven: convection and diffusion change it by less than a sixth)."""
    lib = bbhip.load()
    h = (1.0, 1.0, 1.0)
    kw = box((128, 96, 96), (1, 1, 1), h)
    kw["extensions"]["pp_warmstart"] = "LEARNED"
    on = ctypes.c_int.in_dll(lib, "bb_mg")
    net = ctypes.c_int.in_dll(lib, "bb_warm_use_net")
    saved = on.value, net.value
    net.value = 0
    out = []
    try:
        for mg in (0, 1):
            on.value = mg
            bbconfig.write_case(case_dir, **kw)
            with bbhip.Simulation(case_dir, kw["n"]) as s:
                stats = []
                for _ in range(3):
                    s.step()
                    stats.append(s.pp_stats())
                    assert stats[-1]["resid"] <= 1e-8
                assert ctypes.c_int.in_dll(lib, "bb_mg_last").value == 4 * mg
                s.pull()
                out.append({f: np.array(s.field(f)) for f in "uvw"})
                out[-1].update(dt=s.scalar("dt"), n=[t["niter"] for t in stats],
                               sp_rhs=max(t["sp_rhs"] for t in stats))
    finally:
        on.value, net.value = saved
    ref, got = out
    print("iterations", ref["n"], got["n"])
    assert max(got["n"]) <= 30 < ref["n"][0] and got["n"][-1] < got["n"][0]
    low = min((2 - 2 * np.cos(2 * np.pi / m)) for m in kw["n"]) / 6
    assert velocity_difference(ref, got, kw["n"]) <= \
        7 * difference_bound(got, h, low)


def test_without_memory(case_dir):
    """Where the levels cannot be allocated the solve keeps the Jacobi factor:
    the bits of a solve that does not ask for them."""
    kw = box((128, 96, 96), (1, 0, 1), (1.0, 1.0, 1.0))
    most = ctypes.c_long.in_dll(bbhip.load(), "bb_optional_max")
    most.value = 1 << 20                # fewer bytes than the grid's vector
    try:
        out = run(case_dir, kw, None, 1)
    finally:
        most.value = -1
    ref = run(case_dir, kw, None, 0)
    assert out["levels"] == 0 and out["niter"] == ref["niter"]
    for f in ("u", "v", "w", "phi"):
        assert bitwise_equal(out[f], ref[f]), f


def test_which_way(case_dir):
    """bb_mg_last and bb_resident_last speak of the last solve alone."""
    lib = bbhip.load()
    levels, tiles, spins = (ctypes.c_int.in_dll(lib, "bb_" + n) for n in
                            ("mg_last", "resident_last", "resident_spins"))
    kw = box((128, 96, 96), (1, 0, 1), (1.0, 1.0, 1.0))
    bbconfig.write_case(case_dir, **kw)
    polls = spins.value
    try:
        with bbhip.Simulation(case_dir, kw["n"]) as s:
            s.step()
            assert (levels.value, tiles.value) == (4, 0)
            lib.cuda_PP_cg_noparts()
            assert (levels.value, tiles.value) == (0, 2)
            lib.cuda_PP_cg_mixed()
            assert (levels.value, tiles.value) == (4, 0)
            spins.value = 0             # the one-launch sweep gives up
            lib.cuda_PP_cg_noparts()
            assert (levels.value, tiles.value) == (0, 0)
    finally:
        spins.value = polls
