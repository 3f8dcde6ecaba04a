"""ROMs larger than their windows reach, against the oracle: a cart without a
bank controller maps its first 32 KiB whatever its size, and a controller's
bank number has seven bits, 2 MiB.  Device memory follows what is reachable.

The programs jump with JP a16 between the two windows with register-only
instructions on both sides of the jump (one fused run), and hop through banks
reading and running each."""

from __future__ import annotations

import numpy as np
import pytest

from gbxcule_amd.carts.asm import Asm
from gbxcule_amd.carts.synth import PROGRAM_ORIGIN, finalize_rom

from .conftest import require_gpu
from .test_gpu_light_loops import _check, _joypad

pytestmark = pytest.mark.gpu


def rom_only_cart(code: int) -> bytes:
    """Of 32 KiB << code bytes, jumping between the windows."""
    rom = bytearray(np.random.default_rng(code).integers(0, 256, 0x8000 << code, dtype=np.uint8).tobytes())
    rom[0:0x100] = bytes(0x100)
    a = Asm(origin=PROGRAM_ORIGIN)
    a.ld_rr_d16("SP", 0xDFF0)
    a.label("loop")
    _joypad(a)
    a.ld_r_r("B", "A")
    a.inc_r("C")
    a.jp(0x4100)
    lo = a.resolve()
    rom[PROGRAM_ORIGIN : PROGRAM_ORIGIN + len(lo)] = lo
    b = Asm(origin=0x4100)
    b.alu_r("ADD", "C")
    b.ld_a16_a(0xC000)
    b.alu_d8("XOR", 0x3C)
    b.inc_r("D")
    b.jp(0x0400)
    hi = b.resolve()
    rom[0x4100 : 0x4100 + len(hi)] = hi
    c = Asm(origin=0x0400)
    c.alu_r("ADC", "D")
    c.jp(0x7F00)
    mid = c.resolve()
    rom[0x0400 : 0x0400 + len(mid)] = mid
    d = Asm(origin=0x7F00)
    d.ld_r_r("E", "A")
    d.ld_a16_a(0xC001)
    d.ld_a_a16(0x7FFF)
    d.ld_a16_a(0xC002)
    d.ld_a16_a(0x2000)  # no bank controller: without effect
    d.ld_a_a16(0x4000)
    d.ld_a16_a(0xC003)
    d.inc_r("B")
    d.jp(a.labels["loop"])
    end = d.resolve()
    rom[0x7F00 : 0x7F00 + len(end)] = end
    return finalize_rom(rom, "GBXAMD WIDE", 0x00, code, 0x00)


def banked_cart(kind: int, code: int) -> bytes:
    """Of 32 KiB << code bytes: every bank number, read and run in turn."""
    banks = 2 << code
    rom = bytearray(banks * 0x4000)
    for k in range(1, banks):
        b = Asm(origin=0x4000)
        b.ld_r_d8("A", (k * 37) & 0xFF)
        b.alu_d8("XOR", k >> 8)
        b.alu_r("ADD", "E")
        b.ld_r_r("E", "A")
        b.ret()
        run = b.resolve()
        rom[k * 0x4000 : k * 0x4000 + len(run)] = run
        rom[k * 0x4000 + 0x3FFF] = k & 0xFF
    a = Asm(origin=PROGRAM_ORIGIN)
    a.ld_rr_d16("SP", 0xDFF0)
    a.ld_r_d8("D", 0x00)
    a.label("loop")
    a.ld_r_r("A", "D")
    a.ld_a16_a(0x2000)  # low bits, or all seven on MBC3
    if kind == 0x01:
        a.ld_r_r("A", "D")
        for _ in range(5):
            a.cb(0x3F)  # SRL A
        a.ld_a16_a(0x4000)  # bits 5-6
    a.call(0x4000)
    a.ld_a_a16(0x7FFF)
    a.ld_rr_d16("HL", 0xC100)
    a.ld_r_r("L", "D")
    a.emit(0x77)  # LD (HL),A
    a.ld_r_r("A", "E")
    a.ld_a16_a(0xC000)
    a.inc_r("D")
    a.jp("loop")
    main = a.resolve()
    rom[PROGRAM_ORIGIN : PROGRAM_ORIGIN + len(main)] = main
    return finalize_rom(rom, "GBXAMD BANKS", kind, code, 0x00)


def _create_cost(rom, boot):
    """Device memory (MiB) that a one-env context takes."""
    import torch

    from gbxcule_amd.backend import HipVecBackend

    torch.cuda.synchronize()
    free0 = torch.cuda.mem_get_info()[0]
    be = HipVecBackend(rom, num_envs=1, frames_per_step=1, stage="emulate_only", bootrom=boot)
    be.reset(seed=0)
    free1 = torch.cuda.mem_get_info()[0]
    be.close()
    return (free0 - free1) / 2**20


@pytest.mark.parametrize("code", [0, 1, 8])
def test_rom_only(bootstub, code):
    require_gpu()
    rom = rom_only_cart(code)
    mem = _check(rom, bootstub, 66, 3, 2, f"rom only {code}")
    assert (mem[:, 0xC002] == rom[0x7FFF]).all() and (mem[:, 0xC003] == rom[0x4000]).all()
    # 320 bytes of records a byte of 64 KiB buffer, and the env's own blocks
    assert _create_cost(rom, bootstub) < 100


# 2 MiB, and 4 and 8 MiB of which 2 are reached
@pytest.mark.parametrize(("kind", "code"), [(0x01, 6), (0x01, 7), (0x11, 6), (0x11, 8)])
def test_banked(bootstub, kind, code):
    require_gpu()
    rom = banked_cart(kind, code)
    mem = _check(rom, bootstub, 66, 3, 2, f"banked {kind} {code}")
    want = np.arange(128) if kind == 0x11 else np.where(np.arange(128) % 32 == 0, np.arange(128) + 1, np.arange(128))
    assert (mem[:, 0xC100 + 1 : 0xC100 + 128] == want[1:].astype(np.uint8)).all()
    assert _create_cost(rom, bootstub) < 900
