"""Programs whose wavefronts take the step kernel's short ways, against the
oracle: loads, stores, calls and stack operations only (no register-only
instruction for a pass to run ahead), and the same with a register-only
instruction or four of them on one joypad-keyed path, so that some lanes of a
wavefront have what the others lack; and short loops that halt, whose lanes
hold at HALT for each other."""

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


def halt_cart(kind: int, ie: int, work: int, seed: int) -> bytes:
    """A main loop that halts after `work` stores and adds (more on one
    joypad-keyed path), with IME set on one path and clear on the other."""
    rng = np.random.default_rng(seed)
    rom = bytearray(0x8000)
    h = Asm(origin=0x0068)
    for name, counter in (("vbl", 0xDF00), ("stat", 0xDF01), ("timer", 0xDF02)):
        h.label(name)
        h.push("HL")
        h.ld_rr_d16("HL", counter)
        h.emit(0x34)  # INC (HL)
        if name == "stat":  # LYC on by a prime below 154
            h.push("AF")
            h.ldh_a_a8(0x45)
            h.alu_d8("ADD", 37)
            h.alu_d8("CP", 154)
            h.jr("lyc_ok", "C")
            h.alu_d8("SUB", 154)
            h.label("lyc_ok")
            h.ldh_a8_a(0x45)
            h.pop("AF")
        h.pop("HL")
        h.reti()
    code = h.resolve()
    rom[0x68 : 0x68 + len(code)] = code
    for vec, name in ((0x40, "vbl"), (0x48, "stat"), (0x50, "timer")):
        rom[vec : vec + 3] = bytes([0xC3, h.labels[name] & 0xFF, h.labels[name] >> 8])
    a = Asm(origin=PROGRAM_ORIGIN)
    a.ld_rr_d16("SP", 0xDFF0)
    for reg, v in ((0x06, int(rng.integers(0, 200))), (0x07, 0x05), (0x45, 10), (0x41, 0x40), (0x0F, 0), (0xFF, ie)):
        a.ld_r_d8("A", v)
        a.ldh_a8_a(reg)
    a.ei()
    a.label("loop")
    _joypad(a)
    a.ld_r_r("B", "A")
    for k in range(work):
        a.ld_a_a16(0xC000 + k)
        a.alu_d8("ADD", k + 1)
        a.ld_a16_a(0xC000 + k)
    a.ld_r_r("A", "B")
    a.alu_d8("CP", 0x0F)
    a.jp("ime_off", "NZ")
    a.ei()
    a.halt()
    a.nop()
    a.jp("loop")
    a.label("ime_off")
    a.di()
    a.ld_a16_a(0xC080)
    a.halt()
    a.nop()  # the IME=0 wake skips this byte
    a.inc_r("C")
    a.ei()
    a.jp("loop")
    code = a.resolve()
    rom[PROGRAM_ORIGIN : PROGRAM_ORIGIN + len(code)] = code
    return finalize_rom(rom, "GBXAMD HALT", kind, 0x00, 0x02 if kind == 0x13 else 0x00)


# VBlank, VBlank and STAT, all three; loops well below, about and above the
# 96 instructions within which a lane holds at HALT
@pytest.mark.parametrize("kind", [0x00, 0x01, 0x13])
@pytest.mark.parametrize("ie", [0x01, 0x03, 0x07])
@pytest.mark.parametrize("work", [0, 8, 26, 60])
def test_halt_loops(bootstub, kind, ie, work):
    require_gpu()
    mem = _check(halt_cart(kind, ie, work, 5), bootstub, 70, 3, 2, f"halt {kind} {ie} {work}")
    # every env got its interrupts, and both ways to halt were taken
    assert (mem[:, 0xDF00] > 0).all() and (mem[:, 0xC080] != 0).any()
