"""The broadphase at the edges of its launch shapes: the one-workgroup front (2,048 colliders), the
one-workgroup entry and pair sorts, the link modes (32,768 colliders), the digits counted by the emission
(131,072 colliders), partial workgroups, a few large
boxes among small ones, and streams too short for the entries or the pairs. Against the oracle."""

from __future__ import annotations

import numpy as np
import pytest

from dynamis_amd import abi
from dynamis_amd.broadphase import Broadphase
from dynamis_amd.scenes import uniform_boxes

pytestmark = pytest.mark.gpu


def boxes_of(count, large):
    boxes = uniform_boxes(count, (count / 4.0) ** (1.0 / 3.0) * 10.0, 0.2, 2.0, count)
    for i in range(min(large, count)):
        at = (i * 37) % count
        boxes["min"][at] -= np.float32(15.0)
        boxes["max"][at] += np.float32(15.0)
    return boxes


@pytest.mark.parametrize("count", [1, 255, 256, 257, 1023, 1024, 1025, 2047, 2048, 2049, 4095, 4096, 4097, 32768,
                                   32769, 131072, 131073])
@pytest.mark.parametrize("large", [0, 5])
def test_sizes(device, oracle, count, large):
    boxes = boxes_of(count, large)
    bp = Broadphase(count)
    bp.upload(boxes)
    bp.run()
    got, want = bp.read(), oracle.broadphase(boxes)
    assert np.array_equal(got.entry_keys, want["entry_keys"])
    assert np.array_equal(got.pairs, want["pairs"])
    assert len(got.pairs) == abi.counter(got.counters, "PAIRS")


@pytest.mark.parametrize("count", [900, 5000])
def test_short_streams_count_what_they_refuse(device, count):
    boxes = boxes_of(count, 5)
    full = Broadphase(count)
    full.upload(boxes)
    full.run()
    whole = full.read()
    entries, pairs = abi.counter(whole.counters, "ENTRIES"), abi.counter(whole.counters, "PAIRS")
    short = Broadphase(count, pair_capacity=pairs // 2)
    short.upload(boxes)
    short.run()
    got = short.read()
    assert abi.counter(got.counters, "PAIRS") == pairs
    assert abi.counter(got.counters, "REFUSED_PAIRS") == pairs - pairs // 2
    assert set(map(tuple, got.pairs)) <= set(map(tuple, whole.pairs))
    few = Broadphase(count, entry_capacity=entries // 2)
    few.upload(boxes)
    few.run()
    cut = few.read()
    assert abi.counter(cut.counters, "ENTRIES") == entries
    assert abi.counter(cut.counters, "ENTRY_FAULTS") == (abi.counter(whole.counters, "ENTRY_FAULTS") + entries - entries // 2)


@pytest.mark.parametrize("count", [700, 4500])
@pytest.mark.parametrize("reach", [40.0, 3.0e4, 5.0e6])
def test_levels_of_boxes_of_every_side(device, oracle, count, reach):
    """Sides on both sides of 1 to 16 cells of every level, one long axis or all three, near the origin,
    and where a coordinate is past 2^22 of the finest cells."""
    rng = np.random.default_rng(int(reach) + count)
    boxes = uniform_boxes(count, reach, 0.2, 0.4, 3)
    centre = rng.uniform(-reach, reach, (count, 3))
    ratio = rng.choice([1.0, 1.99, 2.0, 2.01, 4.0, 7.99, 8.0, 8.01, 16.0], (count, 1))
    half = 0.1 * ratio * 2.0 ** rng.integers(0, 14, (count, 1)) * np.where(rng.random((count, 1)) < 0.5, 1.0,
                                                                          rng.uniform(0.01, 1.0, (count, 3)))
    few = rng.random((count, 1)) < 0.03  # most boxes stay small: large ones pair with everything
    half = np.where(few, half, 0.1)
    boxes["min"][:, :3] = (centre - half).astype(np.float32)
    boxes["max"][:, :3] = (centre + half).astype(np.float32)
    bp = Broadphase(count, pair_capacity=256 * count)
    bp.upload(boxes)
    bp.run()
    got, want = bp.read(), oracle.broadphase(boxes, pair_capacity=256 * count)
    assert np.array_equal(got.entry_keys, want["entry_keys"])
    assert np.array_equal(got.pairs, want["pairs"]) and len(got.pairs) < 256 * count
