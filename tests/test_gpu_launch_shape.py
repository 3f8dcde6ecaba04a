"""Step launches of every shape the env count and the cart choose: an env's
state does not depend on the wavefront or workgroup it runs in.

70 envs (checked against the oracle elsewhere) give the state hash, cartridge
RAM and serial bytes of each of 70 action sequences; larger counts repeat the
sequences and must repeat these, at counts on both sides of the rules' edges
(which follow the device's CU count) and with a partial last block and
workgroup.
"""

from __future__ import annotations

import numpy as np
import pytest

from gbxcule_amd.carts.synth import finalize_rom, seeded_actions

from .conftest import require_gpu

pytestmark = pytest.mark.gpu

BASE = 70


def _state(rom, boot, n, steps):
    """Hash of every env; cartridge RAM and serial bytes of the first and last
    BASE envs; (lanes, threads, wavefronts per SIMD) of the launches."""
    import torch

    from gbxcule_amd import _lib
    from gbxcule_amd.backend import HipVecBackend

    dut = HipVecBackend(rom, num_envs=n, frames_per_step=2, release_after_frames=1, stage="emulate_only", bootrom=boot)
    try:
        dut.reset(seed=0)
        for k in range(steps):
            act = np.resize(seeded_actions(7, k, BASE), n)
            dut.step_torch(torch.from_numpy(act).cuda())
        shape = tuple(dut._info(k) for k in (_lib.INFO_STEP_LANES, _lib.INFO_STEP_THREADS, _lib.INFO_STEP_WAVES))
        serial = dut.export_serial()
        ends = [(0, min(BASE, n)), (max(0, n - BASE), n)]
        return (
            dut.state_hash_torch().cpu().numpy(),
            [(lo, dut.export_cart_ram(lo, hi), serial[lo:hi]) for lo, hi in ends],
            shape,
        )
    finally:
        dut.close()


def _same_for_every_shape(rom, boot, n, steps=6):
    want, ((_, ram, serial), _), _ = _state(rom, boot, BASE, steps)
    got, ends, shape = _state(rom, boot, n, steps)
    np.testing.assert_array_equal(got, np.resize(want, n))
    for lo, end_ram, end_serial in ends:
        rows = (lo + np.arange(len(end_ram))) % BASE
        np.testing.assert_array_equal(end_ram, ram[rows])
        np.testing.assert_array_equal(end_serial, serial[rows])
    return shape


def _cus():
    import torch

    return torch.cuda.get_device_properties(0).multi_processor_count


@pytest.mark.parametrize(
    ("cart", "count", "shape"),
    [
        ("c1", lambda cus: 1, (64, 64, 2)),
        ("c2", lambda cus: 65, (64, 64, 2)),
        ("c2", lambda cus: 5003, (64, 64, 2)),
        ("c4", lambda cus: 63, (8, 8, 2)),
        ("c4", lambda cus: 8 * cus, (8, 8, 2)),
        ("c4", lambda cus: 8 * cus + 1, (64, 64, 2)),
        ("c4m3", lambda cus: 8 * cus - 1, (8, 8, 2)),
        ("c4m3", lambda cus: 8 * cus + 1, (64, 64, 2)),
        # one wavefront a workgroup; four, the last workgroup with two
        ("c4m3", lambda cus: 64 * cus, (64, 64, 2)),
        ("c4m3", lambda cus: 64 * cus + 65, (64, 256, 2)),
    ],
)
def test_state_is_independent_of_the_launch_shape(carts, bootstub, cart, count, shape):
    require_gpu()
    assert _same_for_every_shape(carts[cart], bootstub, count(_cus())) == shape


@pytest.mark.parametrize("cart", ["c2", "c4", "c4m3"])
@pytest.mark.parametrize(
    ("count", "waves"),
    [
        (lambda cus: 64 * 8 * cus, 2),
        (lambda cus: 64 * 8 * cus + 1, 3),
        (lambda cus: 64 * 12 * cus, 3),
        (lambda cus: 64 * 12 * cus + 1, 2),
    ],
)
def test_wavefronts_per_simd(carts, bootstub, cart, count, waves):
    """Two wavefronts per SIMD up to 512 envs a CU, three to 768, then two."""
    require_gpu()
    n = count(_cus())
    threads = 256 if cart == "c4m3" else 64
    assert _same_for_every_shape(carts[cart], bootstub, n, steps=3) == (64, threads, waves)


# (cartridge type, ROM size code, RAM size code) over a cart's program: the
# kernel variants that the carts themselves do not reach
@pytest.mark.parametrize(
    ("cart", "header"),
    [
        ("c3", None),
        ("c2", (0x00, 0x00, 0x02)),
        ("c4", (0x03, 0x04, 0x03)),
        ("c4m3", (0x11, 0x04, 0x00)),
    ],
)
def test_three_wavefronts_of_every_variant(carts, bootstub, cart, header):
    """LY polls, block copies, and each cartridge kind with and without RAM."""
    require_gpu()
    rom = carts[cart]
    if header is not None:
        rom = finalize_rom(bytearray(rom), "GBXAMD", *header)
    n = 64 * 8 * _cus() + 1
    assert _same_for_every_shape(rom, bootstub, n, steps=12)[2] == 3


def test_captured_step_of_three_wavefronts(carts, bootstub):
    """A captured step, its variant's first launch, replayed between eager
    work: the build for three wavefronts spills to scratch memory."""
    require_gpu()
    import torch

    from gbxcule_amd.backend import HipVecBackend

    n = 64 * 8 * _cus() + 1
    act = torch.from_numpy(seeded_actions(7, 0, n)).cuda()
    pair = [HipVecBackend(carts["c1"], num_envs=n, frames_per_step=1, release_after_frames=1, stage="emulate_only",
                          bootrom=bootstub) for _ in range(2)]  # fmt: skip
    try:
        for be in pair:
            be.reset(seed=0)
        captured, eager = pair
        graph = torch.cuda.CUDAGraph()
        torch.cuda.synchronize()
        with torch.cuda.graph(graph):
            captured.step_torch(act)
        for _ in range(3):
            graph.replay()
            eager.step_torch(act)
            torch.cuda.synchronize()
            assert torch.equal(captured.state_hash_torch(), eager.state_hash_torch())
    finally:
        for be in pair:
            be.close()
