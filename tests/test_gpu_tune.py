"""The autotuner on the device: every sort tiling it may choose gives the same stable order, and a
world whose sorts were tuned steps bit for bit as an untuned one; the per-GPU cache is reused."""

from __future__ import annotations

import ctypes
import pathlib
import re

import numpy as np
import pytest

from dynamis_amd import scenes, tune
from dynamis_amd._native import call
from dynamis_amd.sort import RadixSort, SortChannels, units_for
from dynamis_amd.world import World, encode
from tests.sort_cases import expected_order

pytestmark = pytest.mark.gpu

TILINGS = [(8, 512), (8, 1024), (8, 2048), (16, 512), (16, 1024), (16, 2048)]


SORT_THREADS = int(re.search(r"kSortThreads = (\d+);", (pathlib.Path(tune.__file__).parent / "csrc" / "sort.h").read_text())[1])
NARROW_BELOW = 1572864  # live records up to which every tiling runs 8 keys a lane


# 300,000 records; two tiles more than there are workgroups, so that some take a second ticket and the
# others one past the last tile; the fewest records that run 16 keys a lane
@pytest.mark.parametrize("items,groups,n", [(i, g, 300_000) for i, g in TILINGS] +
                         [(i, g, SORT_THREADS * i * (g + 1) + 77) for i, g in TILINGS] + [(16, 2048, NARROW_BELOW + 1)])
def test_every_tiling_sorts_the_same(device, items, groups, n):
    rng = np.random.default_rng(n)
    major, minor = (rng.integers(0, 1 << 32, n, dtype=np.uint64).astype(np.uint32) for _ in range(2))
    # all eight digits where numpy's sort is quick enough, else two of them
    words = (4, 4) if n < 1 << 21 else (1, 1)
    payload = np.arange(n, dtype=np.uint32)
    try:
        tune.load(np.array([[0, tune.bucket(n), items, groups]], np.uint32))
        channels = SortChannels.upload(major, minor, payload)
        RadixSort().sort(channels, units_for(n), *words)
        m, k, p = channels.download(n)
    finally:
        tune.load(np.zeros((0, 4), np.uint32))
    if words == (4, 4):
        assert np.array_equal(p, expected_order(major, minor, *words))
    else:
        key = ((major & 0xFF) << 8 | (minor & 0xFF)).astype(np.uint16)
        assert np.array_equal(p, np.argsort(key, kind="stable"))
    assert np.array_equal(m, major[p]) and np.array_equal(k, minor[p])


def test_autotuned_world_steps_identically(device, tmp_path):
    def run(tuned):
        world = World()
        world.create(encode(scenes.cube_drop(2000, seed=3)))
        info = tune.autotune_world(world, tmp_path) if tuned else None
        for _ in range(30):
            world.step(1 / 60)
        return world.states(), info

    try:
        plain, _ = run(False)
        tuned, info = run(True)
        assert not info["from_cache"]
        assert all(t in TILINGS for t in info["tilings"].values())
        assert tuned.tobytes() == plain.tobytes()
        again, info2 = run(True)
        assert info2["from_cache"] and info2["tilings"] == info["tilings"]
        assert again.tobytes() == plain.tobytes()
    finally:
        tune.load(np.zeros((0, 4), np.uint32))


def autotune(capacity):
    items, groups = ctypes.c_uint32(), ctypes.c_uint32()
    call("dyn_sort_autotune", None, capacity, 2, ctypes.byref(items), ctypes.byref(groups))
    return items.value, groups.value


def test_tuner_times_what_is_run(device, tmp_path):
    """Capacities that one workgroup sorts have no tiling and leave no entry; those whose streams are
    always short enough for 8 keys a lane are not given 16; a world of such sorts only is cached."""
    try:
        tune.load(np.zeros((0, 4), np.uint32))
        assert autotune(1) == autotune(tune.SORT_SMALL) == tune.DEFAULT_TILING
        assert len(tune.table()) == 0
        for capacity in (tune.SORT_SMALL + 1, 40_000, 150_000, 300_000, 600_000, 1_200_000, 1_572_864):
            assert autotune(capacity)[0] == 8
            assert tune.bucket(capacity) in tune.table()[:, 1]
        tune.load(np.zeros((0, 4), np.uint32))
        with World() as world:
            world.create(encode(scenes.cube_drop(100, seed=3)))
            assert world.pair_capacity <= tune.SORT_SMALL
            first = tune.autotune_world(world, tmp_path)
            again = tune.autotune_world(world, tmp_path)
        assert set(first["tilings"].values()) == {tune.DEFAULT_TILING}
        assert again["from_cache"] and again["tilings"] == first["tilings"]
        assert len(tune.table()) == 0
    finally:
        tune.load(np.zeros((0, 4), np.uint32))


@pytest.mark.parametrize("threads", [64, 128])
def test_solver_workgroup_sizes_step_identically(device, threads):
    """The solver substeps' kernels in workgroups of 64 or 128 give the 256-thread result bit for
    bit, over a settling drop with many contacts."""
    scene = encode(scenes.cube_drop(1500, seed=4))

    def run(size):
        world = World()
        world.create(scene)
        if size:
            world.set_solver_threads(size)
        for _ in range(60):
            world.step(1 / 60)
        out = world.states(), world.inspect_contacts()
        world.close()
        return out

    (s0, c0), (s1, c1) = run(None), run(threads)
    assert len(c0) > 500
    assert s1.tobytes() == s0.tobytes() and c1.tobytes() == c0.tobytes()


def test_solver_tuning_leaves_the_world_unchanged(device):
    scene = encode(scenes.cube_drop(1500, seed=5))
    plain, tuned = World(), World()
    plain.create(scene)
    tuned.create(scene)
    for _ in range(40):
        plain.step(1 / 60)
        tuned.step(1 / 60)
    before = tuned.states().copy()
    threads, ms = tuned.tune_solver(3)
    assert threads in (64, 128, 256) and all(m > 0 for m in ms)
    assert tuned.states().tobytes() == before.tobytes()
    for _ in range(20):
        plain.step(1 / 60)
        tuned.step(1 / 60)
    assert tuned.states().tobytes() == plain.states().tobytes()
    assert tuned.inspect_contacts().tobytes() == plain.inspect_contacts().tobytes()
    plain.close()
    tuned.close()


def test_solver_tuning_of_a_world_solved_whole(device, tmp_path):
    """No workgroup size is used there: nothing is timed, and no size is cached for larger worlds."""
    with World() as world:
        world.create(encode(scenes.cube_drop(100, seed=5)))
        for _ in range(40):
            world.step(1 / 60)
        world.set_solver_threads(128)
        before = world.states().copy()
        assert world.tune_solver(3) == (128, [0.0, 0.0, 0.0])
        info = tune.autotune_solver(world, tmp_path)
        assert info["threads"] == 128 and not info["from_cache"]
        assert list(tmp_path.iterdir()) == []
        assert world.states().tobytes() == before.tobytes()
