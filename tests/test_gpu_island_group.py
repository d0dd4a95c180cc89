"""The step's island pass at the edge of its one-workgroup form (8,192 rows): chains of touching balls in
shuffled row order that fall asleep, and are woken at one end by a ball and by each other. Each step's
islands, sleeps, wakes and resting contacts against the oracle's step."""

from __future__ import annotations

import numpy as np
import pytest

from dynamis_amd.world import World
from tests.worlds import DT, BodyDesc, encode, static_config

pytestmark = pytest.mark.gpu

COUNTERS = ["CONTACTS", "RESTING", "SLEPT", "WOKE", "WOKE_DEFERRED", "ISLANDS", "ISLAND_FAULTS", "LIVE"]


def chains(rows):
    """Up to three chains along x and a ball that reaches the first one's end after 40 steps; the chains'
    first ball is a static one."""
    rng = np.random.default_rng(rows)
    place = [(0.995 * i + 30.0 * (i * 3 // rows), 0.0, 0.0) for i in range(rows - 1)]
    bodies = [BodyDesc.sphere(0.5, position=p) for p in place[1:]]
    bodies.append(BodyDesc.sphere(0.5, position=(place[-1][0] + 5.0, 0.0, 0.0), velocity=(-6.3, 0.0, 0.0)))
    order = rng.permutation(len(bodies))
    return [BodyDesc.sphere(0.5, position=place[0]).fixed()] + [bodies[i] for i in order]


@pytest.mark.parametrize("rows", [9, 1023, 8192, 8193])
def test_chains(device, oracle, rows):
    scene = encode(chains(rows), static_config())
    world, ref = World(), oracle.world(scene)
    world.create(scene)
    assert len(scene.states) == rows
    seen = dict.fromkeys(COUNTERS, 0)
    for frame in range(60):
        world.step(DT)
        ref.step(DT)
        got, want = world.measured(), ref.measured()
        assert {k: got[k] for k in COUNTERS} == {k: want[k] for k in COUNTERS}, frame
        seen = {k: max(seen[k], got[k]) for k in COUNTERS}
        assert np.array_equal(world.states()["sleeping"], ref.states()["sleeping"]), frame
    assert seen["SLEPT"] and seen["WOKE"] and seen["RESTING"] and not seen["ISLAND_FAULTS"]
    world.close()
    ref.close()
