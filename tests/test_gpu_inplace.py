"""The particle passes with pinned options against the generic passes (every
option at run time), which a run with a magnetic field takes: a field too weak
to change a bit of any velocity must end in the same state, bit for bit, at
particle counts around a block's edges, with one and with four particles a
thread (stores above 262 144), for the collisionless, the electrons' and the
ions' collisional passes, with and without per-particle weights, through
in-place and sort passes (sort 2: every second), and with more collision
candidates than one round of a block's lanes."""
import numpy as np
import pytest

import pic2d
import workloads

pytestmark = pytest.mark.gpu


def by_id(sim, s):
    d = sim.get_state(s)
    d["w"] = sim.get_weights(s)
    o = np.argsort(d["id"])
    return {k: v[o] for k, v in d.items()}


WEAK = 1e-30  # [T]: the generic passes, the same bits
CELL_REMOVED = -16001  # pic_dev.h CELL_DEAD


def run(n, gas, pressure, wall, weights, bfield=0.0, sort=16, steps=4, te=4.0,
        emit=False, removed=False):
    p = workloads.discharge(16, 4, te=te)
    p.init_particle_no = n
    if pressure:
        workloads.with_gas(p, gas, pressure)
        p.gas = gas
    p.wall = wall
    if emit:
        p.e_impact_see = p.ion_impact_see = p.reflection = p.backscatter = 1
    p.sort_interval = sort
    p.magnetic_field, p.angle = bfield, 0.0
    with pic2d.Pic(p) as sim:
        if removed:
            for s in (0, 1):
                d = sim.get_state(s)
                d["cell"][d["id"] % 7 == 0] = (CELL_REMOVED & 0xFFFF) | (3 << 16)
                sim.set_state(s, d)
        if weights is not None:
            for s in (0, 1):
                sim.set_weights(s, weights[s][sim.get_state(s)["id"]])
        sim.advance(steps)
        return ([by_id(sim, s) for s in (0, 1)], [sim.get_qfixed(s) for s in (0, 1)],
                [sim.loss_counts(s) for s in (0, 1)], [sim.collision_counts(s) for s in (0, 1)])


@pytest.mark.parametrize("n", [1, 63, 256, 1023, 1024, 1025, 5000, 263000])
@pytest.mark.parametrize("kind", ["plain", "spawn", "argon", "hydrogen", "dense"])
@pytest.mark.parametrize("sort", [16, 2])
def test_pinned_passes_match_the_generic_pass(n, kind, sort):
    gas, pressure, wall = {
        "plain": (pic2d.GAS_ARGON, 0.0, pic2d.WALL_ABSORB),
        "spawn": (pic2d.GAS_ARGON, 0.0, pic2d.WALL_STEADY),
        "argon": (pic2d.GAS_ARGON, 66.0, pic2d.WALL_STEADY),
        "hydrogen": (pic2d.GAS_HYDROGEN, 66.0, pic2d.WALL_STEADY),
        # most particles are candidates: the queue holds whole blocks
        "dense": (pic2d.GAS_ARGON, 60000.0, pic2d.WALL_ABSORB),
    }[kind]
    print(f"in-place {kind} n={n} sort={sort}", flush=True)
    compare(run(n, gas, pressure, wall, None, sort=sort),
            run(n, gas, pressure, wall, None, sort=sort, bfield=WEAK), kind, n)


def compare(a, b, kind, n):
    for s in (0, 1):
        for k in ("id", "cell", "ox", "oy", "vx", "vy", "vz", "w"):
            assert np.array_equal(a[0][s][k], b[0][s][k]), (s, k)
        for q in (1, 2, 3):
            assert np.array_equal(a[q][s], b[q][s]), (s, q)
    if kind == "dense" and n >= 5000:
        # a quarter of the electrons a step at least: with four particles a
        # thread more than a round of a block's 256 lanes
        assert a[3][0].sum() > n


@pytest.mark.parametrize("n", [1, 1023, 1025, 5000, 263000])  # (the last: four particles a thread)
@pytest.mark.parametrize("kind", ["absorb", "steady", "emit", "argon", "hydrogen", "argon_emit", "dense"])
@pytest.mark.parametrize("sort", [16, 2])
def test_weighted_passes_match_the_generic_pass(n, kind, sort):
    gas, pressure, wall, emit = {
        "absorb": (pic2d.GAS_ARGON, 0.0, pic2d.WALL_ABSORB, False),
        "steady": (pic2d.GAS_ARGON, 0.0, pic2d.WALL_STEADY, False),
        "emit": (pic2d.GAS_ARGON, 0.0, pic2d.WALL_ABSORB, True),
        "argon": (pic2d.GAS_ARGON, 66.0, pic2d.WALL_STEADY, False),
        "hydrogen": (pic2d.GAS_HYDROGEN, 66.0, pic2d.WALL_STEADY, False),
        "argon_emit": (pic2d.GAS_ARGON, 66.0, pic2d.WALL_ABSORB, True),
        "dense": (pic2d.GAS_ARGON, 60000.0, pic2d.WALL_ABSORB, False),
    }[kind]
    rng = np.random.default_rng(n)
    w = [rng.integers(0, 9, n).astype(np.float32) / 4 for _ in range(2)]
    print(f"weighted {kind} n={n} sort={sort}", flush=True)
    kw = dict(sort=sort, te=40.0 if emit else 4.0, emit=emit)
    compare(run(n, gas, pressure, wall, w, **kw), run(n, gas, pressure, wall, w, bfield=WEAK, **kw),
            kind, n)


@pytest.mark.parametrize("weighted", [False, True])
@pytest.mark.parametrize("kind", ["steady", "argon", "emit"])
def test_uploaded_removed_particles_reach_no_wall(kind, weighted):
    """a particle uploaded with the cell of one a collision removed is counted
    as such and dropped by the next pass; it has not reached a wall, so no
    pair is re-injected for it and the surface pass does not see it"""
    n = 2000
    gas, pressure, wall, emit = {
        "steady": (pic2d.GAS_ARGON, 0.0, pic2d.WALL_STEADY, False),
        "argon": (pic2d.GAS_ARGON, 66.0, pic2d.WALL_STEADY, False),
        "emit": (pic2d.GAS_ARGON, 0.0, pic2d.WALL_ABSORB, True),
    }[kind]
    print(f"removed {kind} weighted={weighted}", flush=True)
    w = [np.full(n, 0.5, dtype=np.float32)] * 2 if weighted else None
    kw = dict(sort=16, steps=1, emit=emit, removed=True)
    a = run(n, gas, pressure, wall, w, **kw)
    assert all(a[2][s][4] >= n // 7 for s in (0, 1))
    compare(a, run(n, gas, pressure, wall, w, bfield=WEAK, **kw), kind, n)
