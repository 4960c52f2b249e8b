"""The in-place particle passes with pinned options against the generic pass
(every option at run time), which a species with per-particle weights takes:
the same run with every weight set to 1 must end in the same state, bit for
bit, at particle counts around a block's edges, for the collisionless, the
electrons' and the ions' collisional passes, and with more collision candidates
than one round of a block's lanes."""
import numpy as np
import pytest

import pic2d
import workloads

pytestmark = pytest.mark.gpu


def by_id(sim, s):
    d = sim.get_state(s)
    o = np.argsort(d["id"])
    return {k: v[o] for k, v in d.items()}


def run(n, gas, pressure, wall, weighted, steps=4, te=4.0):
    p = workloads.discharge(16, 4, te=te)
    p.init_particle_no = n
    if pressure:
        workloads.with_gas(p, gas, pressure)
        p.gas = gas
    p.wall = wall
    p.sort_interval = 16
    with pic2d.Pic(p) as sim:
        if weighted:
            for s in (0, 1):
                sim.set_weights(s, np.ones(n, dtype=np.float32))
        sim.advance(steps)
        return ([by_id(sim, s) for s in (0, 1)], [sim.get_qfixed(s) for s in (0, 1)],
                [sim.loss_counts(s) for s in (0, 1)], [sim.collision_counts(s) for s in (0, 1)])


@pytest.mark.parametrize("n", [1, 63, 256, 1023, 1024, 1025, 5000])
@pytest.mark.parametrize("kind", ["plain", "spawn", "argon", "hydrogen", "dense"])
def test_pinned_passes_match_the_generic_pass(n, kind):
    gas, pressure, wall = {
        "plain": (pic2d.GAS_ARGON, 0.0, pic2d.WALL_ABSORB),
        "spawn": (pic2d.GAS_ARGON, 0.0, pic2d.WALL_STEADY),
        "argon": (pic2d.GAS_ARGON, 66.0, pic2d.WALL_STEADY),
        "hydrogen": (pic2d.GAS_HYDROGEN, 66.0, pic2d.WALL_STEADY),
        # most particles are candidates: the queue holds whole blocks
        "dense": (pic2d.GAS_ARGON, 60000.0, pic2d.WALL_ABSORB),
    }[kind]
    print(f"in-place {kind} n={n}", flush=True)
    a, b = (run(n, gas, pressure, wall, w) for w in (False, True))
    for s in (0, 1):
        for k in ("id", "cell", "ox", "oy", "vx", "vy", "vz"):
            assert np.array_equal(a[0][s][k], b[0][s][k]), (s, k)
        for q in (1, 2, 3):
            assert np.array_equal(a[q][s], b[q][s]), (s, q)
    if kind == "dense" and n == 5000:
        assert a[3][0].sum() > n  # a quarter of the electrons a step at least
