"""The commit of staged particles at the counts where its sort changes form (a
wavefront, one, two and four values a thread, the sort in memory): the first c of a
step's injected particles do not depend on how many are injected, so each
commit must append what the largest one appends first, in the same order."""
import numpy as np
import pytest

import pic2d
import workloads

pytestmark = pytest.mark.gpu

LARGEST = 5000


def appended(c, species):
    p = workloads.discharge(16, 4)
    p.number_to_inject = c
    with pic2d.Pic(p) as sim:
        n = sim.particle_size(species)
        sim.inject_particles(species)
        d = sim.get_state(species)
        return {k: v[n:] for k, v in d.items()}


@pytest.fixture(scope="module")
def largest():
    return [appended(LARGEST, s) for s in (0, 1)]


@pytest.mark.parametrize("c", [1, 2, 63, 64, 65, 128, 129, 1000, 1024, 1025, 2048, 2049, 4096, 4097])
def test_commit_order(c, largest):
    print(f"commit c={c}", flush=True)
    for s in (0, 1):
        d = appended(c, s)
        assert len(d["id"]) == c and np.array_equal(np.diff(d["id"]), np.ones(c - 1))
        for k in ("id", "cell", "ox", "oy", "vx", "vy", "vz"):
            assert np.array_equal(d[k], largest[s][k][:c]), (s, k)


def test_largest_commit_is_in_key_order(largest):
    for s in (0, 1):
        assert np.array_equal(np.diff(largest[s]["id"]), np.ones(LARGEST - 1))
        assert len(np.unique(largest[s]["vx"])) > LARGEST // 2


@pytest.mark.parametrize("n", [1, 1024, 1025, 4_300_000, 17_000_000])
def test_wall_pass_keeps_the_store_order(n):
    """The absorbing walls' compaction, whose scan takes one workgroup up to four
    tiles of block counts (16.8 M particles) and three launches beyond: the
    particles inside stay, in order."""
    print(f"wall pass n={n}", flush=True)
    p = workloads.discharge(16, 4, te=40.0)
    p.init_particle_no = n
    with pic2d.Pic(p) as sim:
        sim.get_particle_electric_field(0)
        sim.move_particles(0)
        a = sim.get_state(0)
        sim.boundary(1)
        b = sim.get_state(0)
        jx, jy = pic2d.cell_unpack(a["cell"])
        keep = (jx >= 0) & (jx <= p.nodes - 2) & (jy >= 0) & (jy <= p.nodes - 2)
        assert n < 1000 or 0 < keep.sum() < n
        for k in ("id", "cell", "ox", "vx"):
            assert np.array_equal(a[k][keep], b[k]), k


@pytest.mark.parametrize("fused", [4, 0])
def test_gather_sorts_a_store_whose_order_nobody_knows(fused):
    """phase by phase, from a new handle or after fused steps, a gather after
    sort_interval moves sorts the particles by tile, unless the store's order
    has been read since its last sort pass or it has not passed the walls
    since the move; the particles are the same"""
    out = []
    for read, walls in ((False, True), (True, True), (True, False), (False, False)):
        print(f"gather sort, fused {fused}, read {read}, walls {walls}", flush=True)
        p = workloads.discharge(64, 4, te=40.0)
        p.sort_key = 6  # one tile
        p.sort_interval = 2
        with pic2d.Pic(p) as sim:
            sim.advance(fused)
            if read:
                sim.get_state(0)
            for k in range(2):
                sim.get_particle_electric_field(0)
                sim.move_particles(0)
                if walls:
                    sim.boundary(1)
            sim.get_particle_electric_field(0)
            d = sim.get_state(0)
        jx, jy = pic2d.cell_unpack(d["cell"])
        tile = (jy + 1) // 8 * 64 + (jx + 1) // 8  # of the halo grid
        out.append((d, int((np.diff(tile) < 0).sum())))
    n = len(out[0][0]["id"])
    down = [x[1] for x in out]
    print(f"steps down in {n} particles: {down}", flush=True)
    assert down[0] < min(down[1], n // 16)
    for i, j in ((0, 1), (2, 3)):
        a, b = out[i][0], out[j][0]
        oa, ob = np.argsort(a["id"]), np.argsort(b["id"])
        for k in ("id", "cell", "ox", "oy", "vx", "vy", "vz"):
            assert np.array_equal(a[k][oa], b[k][ob]), (i, j, k)
    assert len(out[2][0]["id"]) > n  # without the wall pass nobody left
