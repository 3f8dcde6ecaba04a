"""The step kernel's debug variants with a trap armed that nothing reaches:
one instruction a pass, every record fetched one ahead, and the same states as
the oracle.  Code in ROM, at bank edges, in RAM and across the boot image's
end, bank switches, interrupts and HALT wakes each take or drop the record
fetched ahead."""

from __future__ import annotations

import pytest

from gbxcule_amd.carts.synth import seeded_actions
from oracle.ref import RefMachine

from ._parity import assert_same_state
from .conftest import require_gpu
from .test_gpu_fetch import bank_edge_cart, boot_edge_cart, boot_edge_image, ram_code_cart
from .test_gpu_light_loops import halt_cart, memory_cart

pytestmark = pytest.mark.gpu

PROGRAMS = {
    "c2": lambda carts: carts["c2"],
    "c4": lambda carts: carts["c4"],
    "c4m3": lambda carts: carts["c4m3"],
    "bank_edge": lambda carts: bank_edge_cart(False),
    "bank_edge_mbc3": lambda carts: bank_edge_cart(True),
    "ram_code": lambda carts: ram_code_cart(),
    "boot_edge": lambda carts: boot_edge_cart(),
    "halt": lambda carts: halt_cart(0x00, 0x07, 8, 5),
    "memory": lambda carts: memory_cart(2),
}


@pytest.mark.parametrize("name", sorted(PROGRAMS))
def test_armed_trap_leaves_the_state_alone(carts, bootstub, name):
    require_gpu()
    from gbxcule_amd.backend import HipVecBackend

    rom, n = PROGRAMS[name](carts), 66
    boot = boot_edge_image("operand_from_cart") if name == "boot_edge" else bootstub
    dut = HipVecBackend(rom, num_envs=n, frames_per_step=2, release_after_frames=1, stage="emulate_only", bootrom=boot)
    ref = RefMachine(n, rom, boot)
    try:
        dut.reset(seed=0)
        ref.step(None, 0, 0, "emulate_only")
        for k in range(4):
            # off for one step between: both variants continue the other's state
            dut.set_debug_traps(trap_pc=0 if k == 2 else 0xFEFF)
            act = seeded_actions(23, k, n)
            dut.step(act)
            ref.step(act, 2, 1, "emulate_only", threads=4)
            assert_same_state(dut, ref, step=k, tag=f"debug {name}")
        assert int(ref.field("trap_flag").sum()) == 0
    finally:
        dut.close()
        ref.close()
