"""The narrowphase's pair lists and its two kinds of GJK at their edges: pair capacities on both sides of
the one-workgroup grouping, and lists long enough for one thread a pair (above 90,112 GJK pairs, above
81,920 resumed ones). The same pairs repeated give the same contacts in every copy, and the first copy is
held to the oracle by the stage's own tests."""

from __future__ import annotations

import numpy as np
import pytest

from dynamis_amd import abi
from dynamis_amd.narrowphase import Narrowphase
from dynamis_amd.world import World
from tests.narrow_cases import DT, pile_scene, with_states

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def settled(device):
    scene = pile_scene(3000, seed=5, hull_sources=64, spacing=1.5)
    with World() as world:
        world.create(scene)
        for _ in range(60):
            world.step(DT)
        return with_states(scene, world.states()), world.pairs(), world.convex_work()


@pytest.fixture(scope="module")
def pile(settled):
    return settled[:2]


@pytest.fixture(scope="module")
def work(settled):
    return settled[2]


def run(scene, pairs, capacity):
    stage = Narrowphase(scene, capacity)
    stage.run(pairs)
    raw, valid = stage.read()
    return raw, valid


@pytest.mark.parametrize("count,capacity", [(1, 1), (255, 256), (257, 16384), (257, 16385), (4097, 16384),
                                            (4097, 16385), (5000, 70001)])
def test_capacities(pile, count, capacity):
    scene, pairs = pile
    pairs = pairs[:: max(1, len(pairs) // count)][:count]
    want_raw, want_valid = run(scene, pairs, 65536)
    raw, valid = run(scene, pairs, capacity)
    assert np.array_equal(valid, want_valid)
    hit = valid == 1
    assert raw[hit].tobytes() == want_raw[hit].tobytes()


@pytest.mark.parametrize("count", [1, 1023, 1024, 1025, 2049])
def test_split_edges(pile, count):
    """GJK lists of just as many pairs (touching ones with a hull or a cylinder and no plane) around the
    workgroups of 1,024 that split them into the penetrating pairs and the hits."""
    scene, pairs = pile
    raw, valid = run(scene, pairs, len(pairs))
    kinds = scene.colliders["kind"][pairs]
    gjk = np.isin(kinds, (abi.SHAPE_HULL, abi.SHAPE_CYLINDER)).any(axis=1) & (kinds != abi.SHAPE_PLANE).all(axis=1)
    chosen = np.resize(np.flatnonzero(gjk & (valid == 1)), count)
    got_raw, got_valid = run(scene, pairs[chosen], 4096)
    assert (got_valid == 1).all()
    assert got_raw.tobytes() == raw[chosen].tobytes()


# the lists' limits, and a quarter more for what moved since the step whose lists are counted
LONG_GJK, LONG_RESUME, MARGIN = 11 << 13, 5 << 14, 1.25


@pytest.mark.parametrize("long_resume", [False, True])
def test_long_list(pile, work, long_resume):
    """GJK by a thread a pair, its open pairs resumed by quads, and both by threads."""
    scene, pairs = pile
    copies = 1 + int(MARGIN * max(LONG_GJK / work["gjk"], long_resume * LONG_RESUME / work["gjk_resumed"]))
    assert MARGIN * work["gjk"] < LONG_GJK < copies * work["gjk"] / MARGIN * 1.01
    assert (copies * work["gjk_resumed"] > LONG_RESUME * MARGIN) == long_resume
    assert long_resume or copies * work["gjk_resumed"] * MARGIN < LONG_RESUME
    want_raw, want_valid = run(scene, pairs, len(pairs))
    hit = want_valid == 1
    assert hit.sum() > 1000
    raw, valid = run(scene, np.tile(pairs, (copies, 1)), copies * len(pairs))
    for c in range(copies):
        part = slice(c * len(pairs), (c + 1) * len(pairs))
        assert np.array_equal(valid[part], want_valid)
        assert raw[part][hit].tobytes() == want_raw[hit].tobytes()
