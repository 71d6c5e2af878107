"""The neighbour passes with several lanes per particle, bit for bit against the
FP32 oracle (the precision form, which has none, against its other forms) where
they can go wrong: both group sizes; particle counts that leave
partial groups, waves and blocks; lists that overflow (the cell sweep); pairs
outside the fast arithmetic's range (coincident and nearly coincident
particles, an infinite temperature, fluid at rest), whose targets are done
again with IEEE operations; tiny and large lengths that switch it off; particle
counts on either side of the sizes where a pass takes another form."""
import subprocess
from pathlib import Path

import numpy as np
import pytest

import cabi

pytestmark = pytest.mark.gpu

FIELDS = ("x", "v", "rho", "T", "p", "a", "ab", "fw", "mw", "drho", "dTdt", "kappa")


def test_fast_arithmetic_rounds_as_ieee():
    """Reciprocal, division and square root of the pair loops over the range they
    are used in: all significands, no result differs from the IEEE operation's."""
    exe = Path(__file__).resolve().parent / "cpp" / "fast_math"
    assert exe.exists(), "tests/cpp/fast_math is built by __graft_entry__.build()"
    print("fast arithmetic", flush=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=100)
    print(r.stdout, flush=True)
    assert r.returncode == 0 and r.stdout.split() == ["0", "0", "0"], r.stdout + r.stderr


def tank(scale=1.0, model="csf", seed=0):
    fluid = cabi.hip_fluid_preset("LN2")
    dx = float(np.float32(0.005 * scale))
    kw = dict(dx=dx, gravity=(0, 0, -0.5), contact_angle_deg=20, velocity_scale=1.0)
    if model == "column":
        kw.update(surface_tension=0, thermal=0, phase_change=0, density_mode=1)
    elif model == "akinci":
        kw.update(surface_tension=2, thermal=0, phase_change=0, contact_angle_deg=60)
    elif model == "sps":
        kw.update(surface_tension=0, thermal=0, phase_change=0, density_mode=1, sps_turbulence=1)
    cfg = cabi.default_config(**kw)
    s = 0.04 * scale
    ps = cabi.hip_build_tank_particles(cabi.box(s, s, s), fluid, dx, cabi.default_fill(
        include_vapor=1 if model == "csf" else 0, T_liquid=fluid.T_sat + 1.0))
    rng = np.random.default_rng(seed)
    fl = ps.phase != cabi.WALL
    ps.x[fl] += (0.05 * dx * rng.uniform(-1, 1, (int(fl.sum()), 3))).astype(np.float32)
    ps.v[fl] = rng.normal(0, 0.05, (int(fl.sum()), 3)).astype(np.float32)
    return fluid, cfg, ps, dx


def take(ps, keep):
    return cabi.ParticleSet(ps.x[keep], ps.v[keep], ps.nrm[keep], ps.m[keep], ps.rho[keep], ps.T[keep], ps.phase[keep],
                            ps.flags[keep], None)


def check(fluid, cfg, ps, dx, variant, steps=2):
    lo, hi = ps.x.min(0) - 4 * dx, ps.x.max(0) + 4 * dx
    gpu, cpu = cabi.HipSolver(cfg, fluid), cabi.CpuSolver("orc", cfg, fluid, 32)
    gpu.set_launch_variant(variant)
    for s in (gpu, cpu):
        s.set_particles(ps, lo, hi)
        s.next_dt()
    for k in range(2):
        for f in FIELDS:
            a, b = gpu.field(f), cpu.field(f)
            assert np.array_equal(a, b, equal_nan=True), (f, k, int((a != b).sum()))
        if k == 0 and steps:
            gpu.run_steps(steps)
            cpu.run_steps(steps)


@pytest.mark.parametrize("variant", [0, 1])
@pytest.mark.parametrize("model", ["csf", "column", "akinci", "sps"])
@pytest.mark.parametrize("drop", [0, 1, 63])
def test_group_sizes_and_remainders(model, variant, drop):
    fluid, cfg, ps, dx = tank(model=model)
    n = len(ps) // 64 * 64 + 1 - drop
    print("lanes", model, variant, n, flush=True)
    walls = np.flatnonzero(ps.phase == cabi.WALL)
    keep = np.ones(len(ps), bool)
    keep[walls[:len(ps) - n]] = False
    check(fluid, cfg, take(ps, keep), dx, variant)


@pytest.mark.parametrize("variant", [0, 1])
@pytest.mark.parametrize("case", ["crowd", "coincident", "close", "hot", "rest"])
def test_particles_outside_the_fast_range(case, variant):
    fluid, cfg, ps, dx = tank()
    fl = np.flatnonzero(ps.phase == cabi.LIQUID)
    steps = 2
    print("lanes", case, variant, flush=True)
    if case == "crowd":  # more than 96 neighbours each
        ps.x[fl[:160]] = ps.x[fl[80]] + (0.4 * dx * np.random.default_rng(1).uniform(-1, 1, (160, 3))).astype(np.float32)
        assert len(fl) >= 160
        steps = 0
    elif case == "coincident":
        ps.x[fl[10]] = ps.x[fl[11]]
        steps = 0
    elif case == "close":
        ps.x[fl[10]] = np.nextafter(ps.x[fl[11]], np.float32(1))
        steps = 0
    elif case == "hot":
        ps.T[fl[20]] = np.float32(np.inf)
        steps = 0
    else:
        ps.v[:] = 0
    check(fluid, cfg, ps, dx, variant, steps)


@pytest.mark.parametrize("scale", [2e-4, 1e6])
def test_lengths_beyond_the_fast_range(scale):
    fluid, cfg, ps, dx = tank(scale=scale, model="column")
    print("lanes scale", scale, flush=True)
    check(fluid, cfg, ps, dx, 0, steps=1)


@pytest.mark.parametrize("n", [2047, 2049, 59_999, 60_000, 79_999, 80_000, 99_999, 100_000, 119_999, 139_999, 140_000,
                               249_999, 250_000, 299_999, 300_000, 399_999, 400_000, 599_999, 600_000, 700_000])
def test_both_sides_of_the_size_rules(n):
    """A heated, superheated two-phase tank of exactly n particles: every pass of
    a step with phase change.  Without transport velocity, whose wall density
    takes a powf that the oracle's libm rounds differently in its last bit for
    a few walls; the other tests here run the passes with it."""
    fluid = cabi.hip_fluid_preset("LN2")
    dx = float(np.float32(0.1 / (round(n ** (1 / 3)) - 4)))
    cfg = cabi.default_config(dx=dx, gravity=(0, 0, -0.5), contact_angle_deg=20, velocity_scale=1.0, thermo_mode=1,
                              lee_evaporation=5.0, lee_condensation=5.0, heater_power=5.0,
                              transport_velocity=0)
    ps = cabi.hip_build_tank_particles(cabi.box(0.1, 0.1, 0.1), fluid, dx, cabi.default_fill(
        T_liquid=fluid.T_sat + 2.0, heater_zmax=-0.05))
    print("lanes sizes", n, len(ps), flush=True)
    keep = np.ones(len(ps), bool)
    assert len(ps) >= n
    walls = np.flatnonzero(ps.phase == cabi.WALL)
    keep[walls[:len(ps) - n]] = False
    ps = take(ps, keep)
    assert len(ps) == n
    lo, hi = ps.x.min(0) - 4 * dx, ps.x.max(0) + 4 * dx
    gpu, cpu = cabi.HipSolver(cfg, fluid), cabi.CpuSolver("orc", cfg, fluid, 32)
    for s in (gpu, cpu):
        s.set_particles(ps, lo, hi)
        s.run_steps(2)
    for f in FIELDS + ("m", "alpha", "wall_w", "heat_w", "nrm", "ns", "id"):
        a, b = gpu.field(f), cpu.field(f)
        assert np.array_equal(a, b, equal_nan=True), (f, int((a != b).sum()))


def beside(ps, dx, n):
    """ps and a block of isolated walls (1.2 dx apart, none within reach of the tank) that makes n particles of it."""
    pad = n - len(ps)
    assert pad >= 0
    side = int(np.ceil(max(pad, 1) ** (1 / 3)))
    g = np.stack(np.meshgrid(*[np.arange(side)] * 3, indexing="ij"), -1).reshape(-1, 3)[:pad]
    x = ps.x.max(0) + np.float32(6 * dx) + (1.2 * dx * g).astype(np.float32)
    cat = lambda a, b: np.concatenate([a, np.asarray(b, a.dtype)])  # noqa: E731
    z = np.zeros(pad)
    return cabi.ParticleSet(cat(ps.x, x), cat(ps.v, 0 * x), cat(ps.nrm, 0 * x), cat(ps.m, z + ps.m.max()),
                            cat(ps.rho, z + ps.rho.max()), cat(ps.T, z + ps.T[0]), cat(ps.phase, z + cabi.WALL),
                            cat(ps.flags, z), None)


@pytest.mark.parametrize("n", [21_000, 30_000, 65_000, 81_000, 160_000, 310_000, 610_000, 2_999_999, 3_000_000])
@pytest.mark.parametrize("compensated", [0, 1])
@pytest.mark.parametrize("crowd", [False, True])
def test_the_form_a_size_selects_changes_no_bit(crowd, compensated, n):
    """A superheated two-phase tank of 13 k particles, alone and beside enough
    walls, out of its reach, that every pass takes the form it has for n
    particles: the tank's fields are the same bits, in the precision form too
    (which has no FP32 oracle), and where lists overflow."""
    fluid = cabi.hip_fluid_preset("LN2")
    dx = 0.004
    cfg = cabi.default_config(dx=dx, gravity=(0, 0, -0.5), contact_angle_deg=20, velocity_scale=1.0, thermo_mode=0,
                              lee_evaporation=5.0, lee_condensation=5.0, compensated_sums=compensated)
    ps = cabi.hip_build_tank_particles(cabi.box(0.07, 0.07, 0.07), fluid, dx, cabi.default_fill(T_liquid=fluid.T_sat + 2.0))
    rng = np.random.default_rng(5)
    fl = ps.phase != cabi.WALL
    ps.x[fl] += (0.05 * dx * rng.uniform(-1, 1, (int(fl.sum()), 3))).astype(np.float32)
    ps.v[fl] = rng.normal(0, 0.05, (int(fl.sum()), 3)).astype(np.float32)
    if crowd:  # more than 96 neighbours each, liquid and vapour, at the interface
        for ph, side in ((cabi.LIQUID, -1), (cabi.VAPOR, 1)):
            at = np.flatnonzero(ps.phase == ph)
            at = at[np.argsort(side * ps.x[at, 2], kind="stable")[:120]]
            ps.x[at] = ps.x[at].mean(0) + (0.5 * dx * rng.uniform(-1, 1, (120, 3))).astype(np.float32)
    print("lanes form", crowd, compensated, n, len(ps), flush=True)
    big = beside(ps, dx, n)
    lo, hi = big.x.min(0) - 4 * dx, big.x.max(0) + 4 * dx
    edge = ps.x.max() + 3 * dx

    def fields(p, variant):
        s = cabi.HipSolver(cfg, fluid)
        s.set_launch_variant(variant)
        s.set_particles(p, lo, hi)
        s.run_steps(1 if crowd else 3)
        assert s.diagnostics().evaporated_mass > 0
        tank = s.field("x").max(1) < edge
        return {f: s.field(f)[tank] for f in FIELDS + ("m", "alpha", "wall_w", "out_m", "out_h", "w_norm", "nrm", "ns", "rmin")}

    alone = fields(ps, 0)
    assert np.isfinite(alone["x"]).all()
    for variant in (0, 1):
        got = fields(big, variant)
        for f, a in alone.items():
            assert np.array_equal(a, got[f], equal_nan=True), (f, variant, int((a != got[f]).sum()))
