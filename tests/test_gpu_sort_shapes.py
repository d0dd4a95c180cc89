"""The radix sort at the edges of its shapes: the one-workgroup sort's sizes (2, 4 and 8 records a lane,
the capacity where the passes take over), tiles of 4,096 and 8,192 keys and their remainders, live counts
on both sides of the switch between them, and a base offset. Against numpy's stable order."""

from __future__ import annotations

import ctypes

import numpy as np
import pytest

from dynamis_amd._native import call, lib
from dynamis_amd.device import DeviceBuffer

pytestmark = pytest.mark.gpu

CAPACITIES = [1, 63, 64, 1023, 1025, 2048, 2049, 4096, 4097, 8191, 8192, 8193, 12289, 65537]


def run(capacity, live, base, major_words, minor_words, seed):
    rng = np.random.default_rng(seed)
    # few distinct keys in some digits, so that equal keys show whether ties keep their order
    lanes = [rng.integers(0, 1 << 32, capacity, dtype=np.uint64).astype(np.uint32) for _ in range(2)]
    lanes[0] &= np.uint32(0xFF03FF07)
    lanes.append(np.arange(capacity, dtype=np.uint32))
    buffers = [DeviceBuffer.from_array(a) for a in lanes]
    count, first = DeviceBuffer.from_array(np.array([live], np.uint32)), DeviceBuffer.from_array(np.array([base], np.uint32))
    scratch = DeviceBuffer(lib().dyn_sort_scratch_bytes(capacity, major_words + minor_words))
    call("dyn_sort_pairs", None, *(ctypes.c_void_p(b.ptr) for b in buffers), capacity, ctypes.c_void_p(count.ptr),
         ctypes.c_void_p(first.ptr), 1, major_words, minor_words, ctypes.c_void_p(scratch.ptr), scratch.nbytes)
    n = min(live, capacity - base)
    part = [a[base:base + n].astype(np.uint64) for a in lanes]
    keys = [(part[0] & ((1 << (8 * major_words)) - 1)), (part[1] & ((1 << (8 * minor_words)) - 1))]
    order = np.lexsort((keys[1], keys[0]))
    faults = ctypes.c_uint32()
    call("dyn_sort_faults", ctypes.byref(faults), 1)
    assert faults.value == 0
    for lane, buffer in zip(lanes, buffers):
        want = lane.copy()
        want[base:base + n] = lane[base:base + n][order]
        assert np.array_equal(buffer.download(np.uint32, capacity), want)


@pytest.mark.parametrize("words", [(2, 2), (4, 1)])
@pytest.mark.parametrize("capacity", CAPACITIES)
def test_full_and_partial(device, capacity, words):
    run(capacity, capacity, 0, *words, seed=capacity)
    run(capacity, capacity - capacity // 3, min(5, capacity // 4), *words, seed=capacity + 1)
    run(capacity, 0, 0, *words, seed=capacity + 2)


@pytest.mark.parametrize("live", [1, 4097, 1572864, 1572865, 2200001])
def test_live_counts_of_a_long_stream(device, live):
    run((1 << 21) + 131072, live, 0, 2, 1, seed=live)
