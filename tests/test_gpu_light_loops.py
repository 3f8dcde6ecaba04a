"""Programs whose wavefronts take the step kernel's short ways, against the
oracle: loads, stores, calls and stack operations only (no register-only
instruction for a pass to run ahead), and the same with a register-only
instruction or four of them on one joypad-keyed path, so that some lanes of a
wavefront have what the others lack."""

from __future__ import annotations

import numpy as np
import pytest

from gbxcule_amd.carts.asm import Asm
from gbxcule_amd.carts.synth import PROGRAM_ORIGIN, finalize_rom, seeded_actions
from oracle.ref import RefMachine

from ._parity import assert_same_state
from .conftest import require_gpu

pytestmark = pytest.mark.gpu


def _check(rom, boot, n, steps, frames, tag):
    from gbxcule_amd.backend import HipVecBackend

    dut = HipVecBackend(rom, num_envs=n, frames_per_step=frames, release_after_frames=1, stage="emulate_only", bootrom=boot)
    ref = RefMachine(n, rom, boot)
    try:
        dut.reset(seed=0)
        ref.step(None, 0, 0, "emulate_only")
        for k in range(steps):
            act = seeded_actions(17, k, n)
            dut.step(act)
            ref.step(act, frames, 1, "emulate_only", threads=4)
            assert_same_state(dut, ref, step=k, tag=tag, mem=k == steps - 1)
        assert int(ref.field("trap_flag").sum()) == 0
        return ref.mem.reshape(n, -1).copy()
    finally:
        dut.close()
        ref.close()


def _joypad(a: Asm) -> None:
    """A = the direction keys' bits (active low)."""
    a.ld_r_d8("A", 0x20)
    a.ldh_a8_a(0x00)
    a.ldh_a_a8(0x00)
    a.alu_d8("AND", 0x0F)


def memory_cart(ahead: int) -> bytes:
    rom = bytearray(0x8000)
    a = Asm(origin=PROGRAM_ORIGIN)
    a.ld_rr_d16("SP", 0xDFF0)
    a.label("loop")
    for k in range(24):
        a.ld_a_a16(0xC000 + k)
        a.push("BC")
        a.call("sub")
        a.pop("DE")
        a.ld_a16_a(0xC101 + k)
        a.ldh_a8_a(0x80 + k)
    if ahead:
        _joypad(a)
        a.alu_d8("CP", 0x0F)
        a.jr("same", "Z")
        for k in range(16):
            for _ in range(ahead):
                a.inc_r("B")
            a.ld_a16_a(0xC200 + k)
        a.label("same")
    a.jp("loop")
    a.label("sub")
    a.push("AF")
    a.pop("BC")
    a.ret()
    code = a.resolve()
    rom[PROGRAM_ORIGIN : PROGRAM_ORIGIN + len(code)] = code
    return finalize_rom(rom, "GBXAMD MEM", 0x00, 0x00, 0x00)


@pytest.mark.parametrize("ahead", [0, 1, 2, 3, 4])
def test_memory_only_programs(bootstub, ahead):
    require_gpu()
    _check(memory_cart(ahead), bootstub, 70, 4, 2, f"memory only, {ahead} ahead")
