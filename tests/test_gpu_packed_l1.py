"""The goal-distance kernel against the torch form of the same function: on
the GPU the same bits (the same sums of whole numbers, then a multiplication
by the 32-bit reciprocal, as torch divides by a number there); on the CPU,
which divides, a relative difference of at most 2 units in the last place,
2.4e-7.  Forms: one goal and
one per env, frame widths that allow 16-, 4- and 1-byte loads, views at odd
offsets and with gaps between frames, and forms that stay with torch."""

from __future__ import annotations

import pytest
import torch

from gbxcule_amd.rl import packed_l1_distance

from .conftest import require_gpu

pytestmark = pytest.mark.gpu


def _check(obs, goal):
    from gbxcule_amd.rl import packed

    want = packed_l1_distance(obs.cpu(), goal.cpu())
    got = packed_l1_distance(obs, goal)
    with pytest.MonkeyPatch.context() as mp:
        mp.setattr(packed, "_l1_kernel_operands", lambda *_: None)
        assert torch.equal(got, packed_l1_distance(obs, goal))
    assert got.dtype is torch.float32 and got.shape == want.shape and got.device == obs.device
    torch.testing.assert_close(got.cpu(), want, rtol=2.4e-7, atol=0)
    if obs.shape[1] == 1:
        assert int(torch.count_nonzero(packed_l1_distance(obs, obs))) == 0


@pytest.mark.parametrize("n", [1, 3, 4, 5, 130])
@pytest.mark.parametrize("hw", [(72, 20), (9, 20), (7, 19), (1, 1), (1, 300)])
def test_matches_torch(n, hw):
    require_gpu()
    from gbxcule_amd.rl import packed

    gen = torch.Generator(device="cuda").manual_seed(n * 1000 + hw[1])
    rnd = lambda *s: torch.randint(0, 256, s, dtype=torch.uint8, device="cuda", generator=gen)  # noqa: E731
    obs, goals = rnd(n, 1, *hw), rnd(n, 1, *hw)
    _check(obs, goals)
    _check(obs, goals[:1])
    _check(obs, goals[0])
    # a slot of a [T, N, ...] buffer, frames with gaps, an odd offset, a shared frame
    wide = rnd(n, 3, *hw)
    buf = rnd(n * hw[0] * hw[1] + 5)
    for view in (rnd(2, n, 1, *hw)[1], wide[:, 1:2], buf[3 : 3 + n * hw[0] * hw[1]].view(n, 1, *hw),
                 obs[:1].expand(n, 1, *hw)):  # fmt: skip
        assert packed._l1_kernel_operands(view, goals) is not None
        _check(view, goals)
    # forms the kernel leaves to torch
    for view in (rnd(n, 1, hw[0], hw[1] * 2)[..., ::2], rnd(n, 1, hw[1], hw[0]).transpose(2, 3), wide):
        if view.is_contiguous() and view.shape[1] == 1:
            continue  # one column or row: contiguous after all
        _check(view, goals[:1])


def test_all_shade_pairs_and_capture():
    require_gpu()
    a = torch.arange(256, dtype=torch.uint8, device="cuda")
    obs = a.view(1, 1, 1, 256).expand(256, 1, 1, 256).contiguous()
    goals = a.view(256, 1, 1, 1).expand(256, 1, 1, 256).contiguous()
    _check(obs, goals)
    out = torch.empty(256, device="cuda")
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out.copy_(packed_l1_distance(obs, goals))
    for k in range(3):
        obs.copy_(obs.roll(k + 1, dims=3))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, packed_l1_distance(obs, goals))


def test_more_frames_than_a_grid_has_wavefronts():
    """2^26 + 3 one-byte frames: one wavefront each would be a grid of more
    than 2^32 threads.  A frame's distance is that of its byte."""
    require_gpu()
    n = (1 << 26) + 3
    gen = torch.Generator(device="cuda").manual_seed(9)
    obs = torch.randint(0, 256, (n, 1, 1, 1), dtype=torch.uint8, device="cuda", generator=gen)
    goal = torch.tensor([0xB4], dtype=torch.uint8, device="cuda").view(1, 1, 1, 1)
    by_byte = packed_l1_distance(torch.arange(256, dtype=torch.uint8).view(256, 1, 1, 1), goal.cpu())
    got = packed_l1_distance(obs, goal)
    want = by_byte.cuda()[obs.view(-1).long()]
    torch.testing.assert_close(got, want, rtol=2.4e-7, atol=0)


def test_vmap_sees_torch_calls():
    require_gpu()
    gen = torch.Generator(device="cuda").manual_seed(5)
    obs = torch.randint(0, 256, (3, 4, 1, 9, 20), dtype=torch.uint8, device="cuda", generator=gen)
    goal = torch.randint(0, 256, (1, 9, 20), dtype=torch.uint8, device="cuda", generator=gen)
    want = torch.stack([packed_l1_distance(o, goal) for o in obs])
    got = torch.vmap(lambda o: packed_l1_distance(o, goal))(obs)
    torch.testing.assert_close(got, want, rtol=2.4e-7, atol=0)


def test_one_env_scalars_match_fields(carts, bootstub):
    """get_cpu_state reads one env's scalars in one call: the values of the
    per-field exports, at both ends of a 64-env block and in a partial one."""
    require_gpu()
    import numpy as np

    from gbxcule_amd import _lib
    from gbxcule_amd.backend import HipVecBackend
    from gbxcule_amd.carts.synth import seeded_actions

    n = 70
    dut = HipVecBackend(carts["c2"], num_envs=n, frames_per_step=1, bootrom=bootstub)
    try:
        dut.reset(seed=0)
        for k in range(3):
            dut.step(seeded_actions(2, k, n))
        fields = {f: dut.export_field(f) for f in _lib.FIELDS}
        for e in (0, 1, 63, 64, 69):
            got = np.empty(len(_lib.FIELDS), dtype=np.int64)
            dut._call("gbx_export_scalars", dut.ctx, e, got.ctypes.data)
            assert {f: int(v) for f, v in zip(_lib.FIELDS, got)} == {f: int(fields[f][e]) for f in _lib.FIELDS}
            assert dut.get_cpu_state(e)["instr_count"] == int(fields["instr_count"][e])
        for bad in (-1, n):
            with pytest.raises(ValueError):
                dut._call("gbx_export_scalars", dut.ctx, bad, got.ctypes.data)
    finally:
        dut.close()
