"""The boot image over every bank that the window at 0000 can hold, against
the oracle.

An MBC1 cart of 2 MiB in banking mode 1 maps bank 0, 32, 64 or 96 at 0000;
with the boot image still mapped (an imported state), addresses below 0100
read the boot image and the rest of the window that bank.  The program reads
on both sides of 0100 (a 16-bit read across it too), calls code in the
window, runs from the boot image across 0100 into the bank, and unmaps the
boot image from there, after which the bank's own first 256 bytes are read
and run.  Envs cover the four banks in both modes.
"""

from __future__ import annotations

import numpy as np
import pytest

from gbxcule_amd.abi import CART_STATE_INDEX
from gbxcule_amd.carts.asm import Asm
from gbxcule_amd.carts.synth import finalize_rom, seeded_actions
from oracle.ref import RefMachine

from ._parity import assert_same_state
from .conftest import require_gpu

pytestmark = pytest.mark.gpu

READS = (0x0000, 0x0050, 0x00FE, 0x00FF, 0x0100, 0x0101, 0x1234, 0x3FFF)


def _cart(seed: int) -> bytes:
    rng = np.random.default_rng(seed)
    rom = bytearray(rng.integers(0, 256, 2 << 20, dtype=np.uint8).tobytes())
    for k in range(4):
        low, high = k * 32 * 0x4000, (k * 32 + 1) * 0x4000
        rom[low + 0x100 : low + 0x104] = bytes([0x00, 0xC3, 0x50, 0x01])  # NOP; JP 0150
        a = Asm(origin=0x0060)  # the bank's own bytes under the boot image
        a.ld_r_d8("A", 0x31 + k)
        a.ld_a16_a(0xC022)
        a.ld_a_a16(0x0050)
        a.ld_a16_a(0xC023)
        a.label("end")
        a.jr("end")
        code = a.resolve()
        rom[low + 0x60 : low + 0x60 + len(code)] = code
        a = Asm(origin=0x0150)
        a.ld_r_r("A", "B")  # as the boot image's INC B left it
        a.ld_a16_a(0xC021)
        a.ld_r_d8("A", 0x01)
        a.ldh_a8_a(0x50)  # unmap the boot image
        a.jp(0x0060)
        code = a.resolve()
        rom[low + 0x150 : low + 0x150 + len(code)] = code
        a = Asm(origin=0x0200)
        a.ld_r_d8("A", 0x11 * (k + 1))
        a.alu_d8("ADD", 0x07)
        a.ld_a16_a(0xC020)
        a.ret()
        code = a.resolve()
        rom[low + 0x200 : low + 0x200 + len(code)] = code
        a = Asm(origin=0x4000)
        for i, addr in enumerate(READS):
            a.ld_a_a16(addr)
            a.ld_a16_a(0xC000 + i)
        a.ld_rr_d16("SP", 0x00FF)
        a.pop("BC")
        a.ld_r_r("A", "B")
        a.ld_a16_a(0xC010)
        a.ld_r_r("A", "C")
        a.ld_a16_a(0xC011)
        a.ld_rr_d16("SP", 0xDFF0)
        a.call(0x0200)
        a.ld_r_d8("B", 0x40)
        a.jp(0x00F8)
        code = a.resolve()
        rom[high : high + len(code)] = code
    return finalize_rom(rom, "GBXAMD BOOT", 0x01, 0x06, 0x00)


def test_boot_image_over_every_low_bank():
    require_gpu()
    from gbxcule_amd.backend import HipVecBackend

    rom = _cart(41)
    boot = bytearray(np.random.default_rng(42).integers(0, 256, 256, dtype=np.uint8).tobytes())
    boot[0xF8:0x100] = bytes([0x04] * 8)  # INC B up to and across 0100
    boot = bytes(boot)
    n = 70
    dut = HipVecBackend(rom, num_envs=n, frames_per_step=1, release_after_frames=1, stage="emulate_only", bootrom=boot)
    ref = RefMachine(n, rom, boot)
    try:
        dut.reset(seed=0)
        ref.step(None, 0, 0, "emulate_only")
        e = np.arange(n)
        cs = dut.export_cart_state()
        cs[:, CART_STATE_INDEX["rom_bank_lo"]] = 1
        cs[:, CART_STATE_INDEX["rom_bank_hi"]] = e % 4
        cs[:, CART_STATE_INDEX["bank_mode"]] = (e // 4) % 2
        assert (cs[:, CART_STATE_INDEX["bootrom_enabled"]] == 1).all()
        dut.import_cart_state(cs)
        ref.cart_state[:] = cs
        pc = np.full(n, 0x4000, np.int64)
        dut.import_field("pc", pc)
        ref.field("pc")[:] = pc
        for k in range(2):
            act = seeded_actions(41, k, n)
            dut.step(act)
            ref.step(act, 1, 1, "emulate_only", threads=4)
            assert_same_state(dut, ref, step=k, tag="boot window")
        assert int(ref.field("trap_flag").sum()) == 0
        mem = ref.mem.reshape(n, -1)
        assert (mem[:, 0xC021] == 0x48).all()
        mode1 = (e // 4) % 2 == 1
        assert (mem[mode1, 0xC022] == 0x31 + (e % 4)[mode1]).all() and (mem[~mode1, 0xC022] == 0x31).all()
    finally:
        dut.close()
        ref.close()
