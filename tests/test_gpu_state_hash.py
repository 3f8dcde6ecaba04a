"""The state hash against its definition, at env counts that fill, miss and
pass a 64-env memory block and that split a block's addresses over many or
few workgroups."""

from __future__ import annotations

import numpy as np
import pytest

from gbxcule_amd._lib import FIELDS

from .conftest import require_gpu

pytestmark = pytest.mark.gpu


def _weights(lo: int, count: int) -> np.ndarray:
    """splitmix64 of lo .. lo + count - 1."""
    z = (np.arange(lo, lo + count, dtype=np.uint64) + np.uint64(1)) * np.uint64(0x9E3779B97F4A7C15)
    z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
    z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
    return z ^ (z >> np.uint64(31))


@pytest.mark.parametrize("n", [1, 63, 64, 65, 2100])
def test_state_hash_matches_definition(carts, bootstub, n):
    require_gpu()
    import torch

    from gbxcule_amd.backend import HipVecBackend

    dut = HipVecBackend(carts["c4m3"], num_envs=n, frames_per_step=1, stage="emulate_only", bootrom=bootstub)
    try:
        dut.reset(seed=0)
        rng = np.random.default_rng(n)
        dut.step_torch(torch.from_numpy(rng.integers(0, 8, n, dtype=np.int32)).cuda())
        rows = min(n, 70)  # envs with every byte value at random, 0x00 and 0xFF runs among them
        mem = rng.integers(0, 256, (rows, 65536), dtype=np.uint8)
        mem[:, 0x8000:0x9000], mem[:, 0x9000:0xA000] = 0xFF, 0x00
        dut.memory_torch()[:rows] = torch.from_numpy(mem).cuda()
        got = [dut.state_hash_torch() for _ in range(2)]
        picks = sorted({0, n // 2, n - 1})
        cs = dut.export_cart_state()
        fields = {f: dut.export_field(f) for f in FIELDS}
        for e in picks:
            parts = [(dut.export_memory(e, e + 1)[0].astype(np.uint64) * _weights(0, 65536)).sum(dtype=np.uint64)]
            v = np.array([int(fields[f][e]) for f in FIELDS], dtype=np.int64)
            narrow = np.array([f not in ("instr_count", "cycle_count") for f in FIELDS])
            v = np.where(narrow, v & 0xFFFFFFFF, v).astype(np.uint64)
            parts.append((v * _weights(65536, len(FIELDS))).sum(dtype=np.uint64))
            c = (cs[e].astype(np.int64) & 0xFFFFFFFF).astype(np.uint64)
            parts.append((c * _weights(65536 + 64, c.size)).sum(dtype=np.uint64))
            want = sum(int(p) for p in parts) % 2**64
            for h in got:
                assert int(h[e].item()) & (2**64 - 1) == want, e
    finally:
        dut.close()
