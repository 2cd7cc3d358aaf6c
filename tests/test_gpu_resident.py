"""The PCG sweep that runs in one launch (bb_resident.h) against the same
solve kernel by kernel: the arithmetic and the order of the dot products are
the same, so iterations and fields agree bit for bit, in the plain and the
mixed form.  Sizes: one tile that is its own neighbour on every side, rows,
columns and planes that end inside a tile, one cell past a tile, one, two and
four tiles per workgroup with a last group that is not full; walls and
periodic faces in each direction, particles, more than 50 iterations (the
plain form's recomputed residual)."""
import ctypes

import numpy as np
import pytest

import bbconfig
import bbhip
from helpers import bitwise_equal

pytestmark = pytest.mark.gpu

FIELDS = ("u", "v", "w", "p", "phi")


def box(n, per, precision):
    """Walls, one of them moving, where a direction is not periodic."""
    P = ("PERIODIC",)
    face = {f: P if per["WESNBT".index(f) // 2] else None for f in "WESNBT"}
    wall = ("DIRICHLET", 0.0, 0.0)
    vel = {c: {f: face[f] or wall for f in "WESNBT"} for c in "uvw"}
    for c, f in (("v", "T"), ("w", "E"), ("u", "N")):
        if not face[f]:
            vel[c][f] = ("DIRICHLET", 0.4, 0.0)
    return dict(n=n, lo=(0.0, 0.0, 0.0),
                hi=tuple(h * m for h, m in zip((0.05, 0.04, 0.06), n)),
                rho_f=1.0, nu=0.01, duration=1.0, pp_max_iter=100000,
                pp_residual=1e-8,
                p_bc={f: face[f] or ("NEUMANN", 0.0) for f in "WESNBT"},
                vel_bc=vel, init_cond="QUIESCENT",
                extensions={"fixed_dt": 1e-3, "perturb": (7, 0.2),
                            "pp_precision": precision})


def run(case_dir, kw, parts, resident, nsteps=2, spins=None):
    lib = bbhip.load()
    on = ctypes.c_int.in_dll(lib, "bb_resident")
    most = ctypes.c_int.in_dll(lib, "bb_resident_spins")
    saved = on.value, most.value
    on.value = resident
    if spins is not None:
        most.value = spins
    try:
        bbconfig.write_case(case_dir, **kw)
        if parts:
            bbconfig.write_parts(case_dir, parts)
        out = {"iters": [], "tiles": [], "resid": []}
        with bbhip.Simulation(case_dir, kw["n"]) as s:
            for _ in range(nsteps):
                s.step()
                out["iters"].append(s.pp_stats()["niter"])
                out["resid"].append(s.pp_stats()["resid"])
                out["tiles"].append(
                    ctypes.c_int.in_dll(lib, "bb_resident_last").value)
            s.pull()
            out["f"] = {f: np.array(s.field(f)) for f in FIELDS}
    finally:
        on.value, most.value = saved
    return out


def same(a, b):
    assert a["iters"] == b["iters"]
    for f in FIELDS:
        assert bitwise_equal(a["f"][f], b["f"][f]), f


@pytest.mark.parametrize("n,per,tiles", [
    ((64, 8, 8), (1, 1, 1), (1, 1)), ((3, 2, 2), (0, 0, 0), (1, 1)),
    ((65, 9, 9), (0, 1, 0), (1, 1)), ((65, 9, 17), (1, 0, 1), (1, 1)),
    ((40, 30, 23), (0, 0, 1), (1, 1)), ((128, 24, 33), (1, 1, 0), (1, 1)),
    ((64, 128, 130), (1, 0, 0), (2, 2)), ((100, 70, 131), (0, 1, 1), (2, 2)),
    ((129, 16, 40), (1, 0, 0), (0, 1)), ((130, 126, 100), (0, 0, 0), (0, 4)),
    ((256, 64, 129), (1, 1, 0), (0, 4)), ((60, 512, 137), (1, 0, 1), (0, 0))])
@pytest.mark.parametrize("precision", ["PLAIN", "MIXED"])
def test_one_launch_same_bits(case_dir, n, per, tiles, precision):
    """tiles: tiles per workgroup of the plain and of the mixed form, 0 where
    the grid does not fit."""
    kw = box(n, per, precision)
    ref = run(case_dir, kw, None, 0)
    out = run(case_dir, kw, None, 1)
    assert ref["tiles"][-1] == 0
    assert out["tiles"][-1] == tiles[precision == "MIXED"]
    print("iterations", out["iters"])
    same(out, ref)


@pytest.mark.parametrize("n,walls", [((64, 64, 64), ""), ((72, 60, 70), "z")])
@pytest.mark.parametrize("precision", ["PLAIN", "MIXED"])
def test_one_launch_particles_same_bits(case_dir, n, walls, precision):
    """Particle cells masked out, several Lamb passes per step."""
    kw, parts = bbconfig.sediment(n=n, nparts=3, a=5.0, seed=13, walls=walls)
    for P, c in zip(parts, ((20., 20., 20.), (44., 30., 33.), (24., 46., 45.))):
        P.update(x=c[0], y=c[1], z=c[2])
    kw["extensions"] = {"pp_precision": precision}
    ref = run(case_dir, kw, parts, 0)
    out = run(case_dir, kw, parts, 1)
    assert out["tiles"][-1] > 0
    same(out, ref)


@pytest.mark.parametrize("precision", ["PLAIN", "MIXED"])
def test_one_launch_warm_start_same_bits(case_dir, precision):
    """From earlier solutions instead of phi = 0 (the guess without its
    network)."""
    kw, parts = bbconfig.sediment(n=(64, 32, 48), nparts=2, a=5.0, seed=13)
    kw["extensions"] = {"pp_precision": precision, "pp_warmstart": "LEARNED"}
    net = ctypes.c_int.in_dll(bbhip.load(), "bb_warm_use_net")
    saved, net.value = net.value, 0
    try:
        ref = run(case_dir, kw, parts, 0, nsteps=3)
        out = run(case_dir, kw, parts, 1, nsteps=3)
    finally:
        net.value = saved
    assert out["tiles"][-1] > 0 and ref["tiles"][-1] == 0
    assert out["iters"][-1] < out["iters"][0]
    same(out, ref)


@pytest.mark.parametrize("precision", ["PLAIN", "MIXED"])
def test_wait_that_gives_up(case_dir, precision):
    """With no poll allowed the sweep gives up at its first meeting and the
    solve runs kernel by kernel: the same bits for the plain form, the same
    stopping test for the mixed one."""
    kw = box((64, 24, 24), (1, 0, 1), precision)
    ref = run(case_dir, kw, None, 0)
    out = run(case_dir, kw, None, 1, spins=0)
    assert out["tiles"][-1] == 0
    assert max(out["resid"]) <= 1e-8
    if precision == "PLAIN":
        same(out, ref)


@pytest.mark.parametrize("precision", ["PLAIN", "MIXED"])
def test_without_memory(case_dir, precision):
    """Where the slots cannot be allocated: kernel by kernel."""
    kw = box((64, 24, 24), (1, 0, 1), precision)
    most = ctypes.c_long.in_dll(bbhip.load(), "bb_optional_max")
    most.value = 0
    try:
        out = run(case_dir, kw, None, 1)
    finally:
        most.value = -1
    assert out["tiles"][-1] == 0
    same(out, run(case_dir, kw, None, 0))
