"""The solver of small worlds (k_group_solve, k_group_position) at the edges of its rules: row counts
on both sides of each workgroup size and of the limits, more contacts than its threads hold in
registers, sleeping rows, and batches whose worlds sit on both sides. Bit for bit against the
oracle's solver, and each world of a batch against itself alone."""

from __future__ import annotations

import ctypes
import threading

import numpy as np
import pytest

from dynamis_amd._native import call
from dynamis_amd.device import profile_collect, profile_enable
from dynamis_amd.solver import Solver
from dynamis_amd.world import Batch, World
from tests.solve_cases import drop_scene, solver_inputs
from tests.test_gpu_solve import check_parity
from tests.worlds import DT, config, cube_drop, encode

pytestmark = pytest.mark.gpu


# bodies (a plane more): 64 | 65 rows (256 | 512 lanes), 160 | 161 (whole | position only),
# 256 | 257 (256 | 1,024 lanes); 2304 | 2305 below (position only | launched)
@pytest.mark.parametrize("count", [1, 63, 64, 159, 160, 255, 256])
def test_row_edges(device, oracle, count):
    check_parity(oracle, drop_scene(count, footprint=1.2 + 0.35 * count ** 0.5), 60, 0 if count == 1 else count // 2)


@pytest.mark.parametrize("count", [2303, 2304])
def test_row_limit(device, oracle, count):
    # a lattice of touching cubes on the plane: contacts from the first frames on
    side = 12.0
    profile_collect()
    profile_enable(True)
    check_parity(oracle, drop_scene(count, footprint=side), 4, 4000)
    profile_enable(False)
    assert ("k_group_position" in profile_collect()) == (count == 2303)


@pytest.mark.parametrize("count", [1501, 1502])
def test_world_row_limit(device, oracle, count):
    """A world's captured steps launch their position iterations from 1,503 rows on."""
    scene = drop_scene(count, footprint=12.0)
    ref = oracle.world(scene)
    with World() as world:
        world.create(scene)
        for _ in range(6):
            ref.step(DT)
            world.step(DT)
        assert world.measured()["CONTACTS"] > 1500
        assert world.states().tobytes() == ref.states().tobytes()
        assert ("k_group_position" in kernels_of_a_step(world)) == (count == 1501)
    ref.close()


# Blocks that a workgroup of k_group_solve has a quad for each, kept in registers (64 of 256 lanes up to 64
# rows, 128 of 512 up to 160), and contacts that the position iterations hold, four a lane (1,024, 2,048;
# k_group_position 1,024 of 256 lanes up to 256 rows, 4,096 of 1,024 above): just as many and one more, and no contact.
@pytest.mark.parametrize("bodies,contacts", [
    (40, 0), (40, 64), (40, 65), (40, 1024), (40, 1025), (120, 128), (120, 129), (120, 2048), (120, 2049),
    (200, 1024), (200, 1025), (400, 4096), (400, 4097)])
def test_contacts_that_registers_hold(device, oracle, bodies, contacts):
    scene = drop_scene(bodies, footprint=1.2 + 0.35 * bodies ** 0.5)
    inputs, some, _, _ = solver_inputs(oracle, scene, 60)
    assert len(some) > bodies // 2
    given = np.resize(some, contacts) if contacts else some[:0]  # the list over and over
    ref = oracle.world(inputs, contact_capacity=max(contacts, 1))
    want_contacts = ref.solve(given, DT)
    want_states = ref.states()
    ref.close()
    solver = Solver(inputs, max(contacts, 1))
    solver.run(inputs.states, given, DT)
    states, got_contacts, _ = solver.read()
    assert states.tobytes() == want_states.tobytes()
    assert got_contacts.tobytes() == want_contacts.tobytes()


def test_sleeping_rows(device, oracle):
    scene = encode(cube_drop(120, seed=1, footprint=8.0, high=4.0), config())
    inputs, _ = check_parity(oracle, scene, 200, 100)
    assert (inputs.states["sleeping"][:scene.dynamic_count] != 0).any()


@pytest.mark.parametrize("counts", [(3, 40, 1, 150), (5, 400, 1, 70, 260), (2500, 30)])
def test_batches_on_both_sides(device, counts):
    scenes = [encode(cube_drop(n, seed=7 + i, footprint=0.9 * n ** 0.5 + 1.0, low=1.0, high=3.0), config())
              for i, n in enumerate(counts)]
    batch = Batch(scenes)
    alone = []
    for s in scenes:
        w = World()
        w.create(s)
        alone.append(w)
    for _ in range(40):
        batch.step(DT)
        for w in alone:
            w.step(DT)
    states = batch.states()
    for i, w in enumerate(alone):
        assert batch.world_states(i, states).tobytes() == w.states().tobytes(), i
    total = {k: sum(w.measured()[k] for w in alone) for k in ("CONTACTS", "SOLVER_ROWS", "LIVE")}
    got = batch.measured()
    assert {k: got[k] for k in total} == total
    batch.close()
    for w in alone:
        w.close()


def kernels_of_a_step(batch) -> set:
    batch.set_graphs(False)
    profile_collect()
    profile_enable(True)
    batch.step(DT)
    batch.wait()
    profile_enable(False)
    batch.set_graphs(True)
    return set(profile_collect())


# worlds of some bodies each: the most that are solved whole | one more; position iterations by
# workgroups | too many tiny worlds for them, by themselves and beside a larger one; 2,304 | 2,305 rows,
# the most that a workgroup holds
@pytest.mark.parametrize("parts,solve,position", [
    ([(1024, 3)], True, False), ([(1025, 3)], False, True), ([(2600, 3)], False, True), ([(2800, 3)], False, False),
    ([(1, 500), (800, 3)], False, True), ([(1, 500), (900, 3)], False, False),
    ([(20, 2303)], False, True), ([(20, 2304)], False, False)])
def test_many_worlds(device, parts, solve, position):
    """Which kernels take a batch of many worlds, and that each world steps as it does alone."""
    kinds = [[encode(cube_drop(n, seed=11 + i, footprint=0.9 * n ** 0.5 + 1.0, low=1.0, high=2.0), config())
              for i in range(3)] for _, n in parts]
    scenes = [kind[i % 3] for (count, _), kind in zip(parts, kinds) for i in range(count)]
    batch = Batch(scenes)
    for _ in range(29):
        batch.step(DT)
    names = kernels_of_a_step(batch)
    assert ("k_group_solve" in names, "k_group_position" in names) == (solve, position)
    assert ("k_position_apply" in names) == (not solve and not position)
    states, first = batch.states(), 0
    for (count, _), kind in zip(parts, kinds):
        for i in range(min(count, 3)):
            with World() as world:
                world.create(kind[i])
                for _ in range(30):
                    world.step(DT)
                alone = world.states()
            for at in range(first + i, first + count, 3):
                assert batch.world_states(at, states).tobytes() == alone.tobytes(), at
        first += count
    batch.close()


def test_sizes_side_by_side(device):
    """Worlds whose workgroups ask for different amounts of LDS, launched from two threads at once."""
    scenes = [encode(cube_drop(n, seed=n, footprint=0.5 * n ** 0.5, low=1.0, high=3.0), config()) for n in (1000, 1500)]

    def steps(scene, out, key):
        with World() as world:
            world.create(scene)
            world.set_graphs(False)
            for _ in range(60):
                world.step(DT)
            out[key] = world.states().tobytes()

    alone, beside = {}, {}
    for i, scene in enumerate(scenes):
        steps(scene, alone, i)
    threads = [threading.Thread(target=steps, args=(scene, beside, i)) for i, scene in enumerate(scenes)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert beside == alone


def batch_of(scene, colliders, owners, worlds, world_count) -> World:
    world = World()
    world.scene = scene
    colliders, owners, worlds = (np.ascontiguousarray(a) for a in (colliders, owners, worlds))
    n, k = len(scene.states), len(colliders)
    call("dyn_batch_create", ctypes.byref(world._handle), None, scene.params.ctypes.data, scene.states.ctypes.data,
         scene.descs.ctypes.data, n, scene.dynamic_count, colliders.ctypes.data, owners.ctypes.data,
         worlds.ctypes.data, k, world_count, 8 * n, 32 * n)
    return world


def test_batch_of_sparse_world_ids(device):
    """Two worlds with the ids 7 and 2^32 - 2 of 2^32 - 1: creation keeps nothing for an id without colliders."""
    scenes = [encode(cube_drop(30, seed=3 + i, footprint=4.0, low=1.0, high=3.0), config()) for i in range(2)]
    batch = Batch(scenes)
    merged, worlds = batch.scene, batch.layout.collider_worlds
    ids = np.array([7, 0xFFFFFFFE], np.uint32)[worlds]
    world = batch_of(merged, merged.colliders, merged.owners, ids, 0xFFFFFFFF)
    for _ in range(40):
        batch.step(DT)
        world.step(DT)
    assert "k_group_solve" in kernels_of_a_step(world)
    batch.step(DT)
    assert world.states().tobytes() == batch.states().tobytes()
    batch.close()
    world.close()


def test_batch_of_scattered_colliders(device):
    """Colliders of two worlds interleaved: their contacts are no runs, and the launched passes run."""
    scenes = [encode(cube_drop(30, seed=3 + i, footprint=4.0, low=1.0, high=3.0), config()) for i in range(2)]
    batch = Batch(scenes)
    merged, worlds = batch.scene, batch.layout.collider_worlds
    mixed = np.argsort(np.concatenate([np.arange(31), np.arange(31)]), kind="stable")
    world = batch_of(merged, merged.colliders[mixed], merged.owners[mixed], worlds[mixed], 2)
    for _ in range(40):
        batch.step(DT)
        world.step(DT)
    # each world's colliders keep their order, so its steps stay the same
    assert world.states().tobytes() == batch.states().tobytes()
    batch.close()
    world.close()
