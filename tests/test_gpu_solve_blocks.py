"""The solver's blocks by quads and by single lanes (above 40,960 blocks), with rolling and spin friction
and compliance, which no scene of the other solver tests has: blocks of one to four points with zero,
small and large limits, in worlds solved whole by a workgroup and by the launched passes. Bit
for bit against the oracle's solver."""

from __future__ import annotations

import numpy as np
import pytest

from dynamis_amd.solver import Solver
from tests.narrow_cases import DT
from tests.solve_cases import NO_SLEEP, solver_inputs
from tests.worlds import config, ellipsoid_hulls, encode, mixed_pile

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bodies,blocks", [(40, 0), (200, 0), (200, 5 << 13), (200, (5 << 13) + 1),
                                           (200, 1 << 17), (200, (1 << 17) + 1)])
def test_blocks(device, oracle, bodies, blocks):
    scene = encode(mixed_pile(bodies, seed=4, kinds=5, hull_sources=4, spacing=1.4), config(**NO_SLEEP),
                   ellipsoid_hulls(4, seed=3))
    inputs, contacts, _, _ = solver_inputs(oracle, scene, 50)
    assert set(contacts["point_count"]) >= {1, 4}
    contacts = np.resize(contacts, blocks or len(contacts))  # the list over and over
    rng = np.random.default_rng(bodies)
    limits = np.array([0.0, 0.0, 1e-3, 0.3, 10.0], np.float32)
    contacts["rolling_friction"] = rng.choice(limits, len(contacts))
    contacts["spin_friction"] = rng.choice(limits, len(contacts))
    contacts["relaxation"] = rng.choice(np.array([0.0, 0.0, 0.02], np.float32), len(contacts))
    contacts["damping_ratio"] = rng.choice(np.array([0.0, 1.0], np.float32), len(contacts))
    ref = oracle.world(inputs, contact_capacity=len(contacts))
    want_contacts = ref.solve(contacts, DT)
    want_states = ref.states()
    ref.close()
    solver = Solver(inputs, len(contacts))
    solver.run(inputs.states, contacts, DT)
    states, got_contacts, _ = solver.read()
    assert states.tobytes() == want_states.tobytes()
    assert got_contacts.tobytes() == want_contacts.tobytes()
