"""Step launches of every shape the env count and the cart choose: an env's
state does not depend on the wavefront or workgroup it runs in.

70 envs (checked against the oracle elsewhere) give the state hash of each of
70 action sequences; larger counts repeat the sequences and must repeat the
hashes, at counts on both sides of the rule's edges and with a partial last
block and workgroup.
"""

from __future__ import annotations

import numpy as np
import pytest

from gbxcule_amd.carts.synth import seeded_actions

from .conftest import require_gpu

pytestmark = pytest.mark.gpu

BASE, STEPS = 70, 6


def _hashes(rom, boot, n):
    import torch

    from gbxcule_amd.backend import HipVecBackend

    dut = HipVecBackend(rom, num_envs=n, frames_per_step=2, release_after_frames=1, stage="emulate_only", bootrom=boot)
    try:
        dut.reset(seed=0)
        for k in range(STEPS):
            act = np.resize(seeded_actions(7, k, BASE), n)
            dut.step_torch(torch.from_numpy(act).cuda())
        return dut.state_hash_torch().cpu().numpy(), dut.step_lanes
    finally:
        dut.close()


@pytest.mark.parametrize(
    ("cart", "n", "lanes"),
    [
        ("c1", 1, 64),
        ("c2", 65, 64),
        ("c2", 5003, 64),
        ("c4", 63, 8),
        ("c4", 2048, 8),
        ("c4", 2049, 64),
        ("c4m3", 2047, 8),
        ("c4m3", 2049, 64),
        ("c4m3", 16384, 64),  # one wavefront a workgroup
        ("c4m3", 16449, 64),  # four, the last workgroup with two
    ],
)
def test_state_is_independent_of_the_launch_shape(carts, bootstub, cart, n, lanes):
    require_gpu()
    want, _ = _hashes(carts[cart], bootstub, BASE)
    got, got_lanes = _hashes(carts[cart], bootstub, n)
    assert got_lanes == lanes
    np.testing.assert_array_equal(got, np.resize(want, n))
