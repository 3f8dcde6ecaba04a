"""The work this framework is used for, as timed cases.

A case is one pass of a user's loop over the public API: a step of all envs,
an RL step with render, reward, senses and masked reset, a memory readout, a
lockstep verification step.  The carts are the repository's own synthetic ones
(``gbxcule_amd.carts.synth``), as are the workloads the sizes come from.

Everything an emulator returns is a whole number (memory bytes, shades,
registers), or one 32-bit rounding of one (observations, goal distances), so
outputs have to be the same.  Plain torch or numpy has no Game Boy to compute
them with in 64 bits: ``exact`` has no values.
"""

from __future__ import annotations

from functools import lru_cache

import numpy as np
import torch

from gbxcule_amd.backend import HipVecBackend
from gbxcule_amd.carts.bootstub import build_bootstub
from gbxcule_amd.carts.synth import CARTS, seeded_actions
from gbxcule_amd.reset_cache import ResetCache
from gbxcule_amd.rl import PackedPixelEnv, packed_l1_distance

STATE_BYTES = 922  # registers, counters, cartridge state and the IO page of one env
CYCLES_PER_FRAME = 17556  # machine cycles of one emulated frame
PACKED, UNPACKED = 72 * 20, 72 * 80  # bytes of one downsampled frame
TRACE = 16  # steps of the action trace and of the reset masks a state holds
SENSES = 32


def _step(name, cart, envs, frames, stage="emulate_only", cart_seed=0):
    return {"name": name, "kind": "step", "cart": cart, "cart_seed": cart_seed, "envs": envs, "frames": frames,
            "stage": stage}  # fmt: skip


def listed():
    return [
        # a handful of envs stepped a few frames at a time: a unit test, a
        # notebook, one player; launch and single-wavefront latency
        _step("smoke_64", "c1", 64, 4, "full_step", 0),
        # the CPU-step workload, 16,384 envs at frameskip 24
        _step("cpu_step_16384", "c2", 16_384, 24, "emulate_only", 1),
        # the same program at a ragged env count and a short frameskip
        _step("cpu_step_20011", "c2", 20_011, 4, "obs_only", 1),
        # banked cart with timer, STAT and VBlank interrupts, one frame a step
        _step("bank_131072_fs1", "c4", 131_072, 1, "emulate_only", 3),
        # banked cart with cartridge RAM and clock, a whole agent step
        _step("rtc_65536_fs24", "c4m3", 65_536, 24, "emulate_only", 4),
        # step and packed observation of a PPU-heavy cart
        {"name": "ppu_16384", "kind": "rollout", "cart_seed": 2, "envs": 16_384, "frames": 24, "packed": True,
         "senses": 0, "reset": 0.0},
        # the RL rollout shape: step, unpacked observation, ~1% masked resets,
        # RAM senses
        {"name": "rollout_131072", "kind": "rollout", "cart_seed": 2, "envs": 131_072, "frames": 24,
         "packed": False, "senses": SENSES, "reset": 0.01},
        # the packed RL env with a goal-distance reward, few envs (launches
        # and host calls count) and a ragged mid-size batch
        {"name": "env_64", "kind": "env", "cart_seed": 2, "envs": 64, "frames": 24, "reset": 0.02},
        {"name": "env_5003", "kind": "env", "cart_seed": 2, "envs": 5_003, "frames": 24, "reset": 0.01},
        # the numpy API: host actions in, host observations out, frames
        # rendered on each step
        {"name": "host_step_1000", "kind": "host", "cart_seed": 2, "envs": 1_000, "frames": 24},
        # RAM detectors reading slices of emulated memory of every env, and
        # one poke
        {"name": "readout_16384", "kind": "readout", "cart_seed": 1, "envs": 16_384, "span": 360},
        # lockstep verification: one frame, a state hash of every env, one
        # env's registers and work RAM read back
        {"name": "verify_4096", "kind": "verify", "cart": "c4", "cart_seed": 3, "envs": 4_096},
    ]  # fmt: skip


def _log_int(rng, lo, hi):
    """A whole number spread over the logarithm of [lo, hi]."""
    return max(lo, min(hi, int(round(lo * (hi / lo) ** rng.random()))))


def draw(rng):
    kind = rng.choice(["step", "step", "step", "rollout", "rollout", "env", "env", "host", "readout", "verify"])
    seed = rng.randrange(1, 1000)
    if kind == "step":
        cart = rng.choice(["c1", "c2", "c2", "c4", "c4m3"])
        frames = rng.choice([1, 2, 4, 8, 24])
        # no more env-frames than the largest listed step of its kind
        most = 16_384 * 24 if cart in ("c1", "c2") else 65_536 * 24
        envs = _log_int(rng, 32, min(131_072, most // frames))
        stage = rng.choice(["emulate_only", "obs_only", "reward_only", "full_step"])
        return {"kind": kind, "cart": cart, "cart_seed": seed, "envs": envs, "frames": frames, "stage": stage}
    if kind == "rollout":
        return {"kind": kind, "cart_seed": seed, "envs": _log_int(rng, 64, 131_072),
                "frames": rng.choice([4, 24]), "packed": rng.random() < 0.5,
                "senses": rng.choice([0, 3, 16, SENSES]), "reset": rng.choice([0.0, 0.005, 0.01, 0.05])}  # fmt: skip
    if kind == "env":
        return {"kind": kind, "cart_seed": seed, "envs": _log_int(rng, 16, 32_768), "frames": rng.choice([4, 24]),
                "reset": rng.choice([0.01, 0.02])}  # fmt: skip
    if kind == "host":
        return {"kind": kind, "cart_seed": seed, "envs": _log_int(rng, 16, 8_192), "frames": rng.choice([1, 24])}
    if kind == "readout":
        return {"kind": kind, "cart_seed": seed, "envs": _log_int(rng, 64, 32_768), "span": rng.randrange(17, 1025)}
    return {"kind": kind, "cart": rng.choice(["c2", "c4", "c4m3"]), "cart_seed": seed,
            "envs": _log_int(rng, 16, 8_192)}  # fmt: skip


@lru_cache(maxsize=32)
def _rom(cart, seed):
    return CARTS[cart](seed)


def _trace(seed, envs):
    """TRACE steps of seeded 8-way actions on the device."""
    return torch.from_numpy(np.stack([seeded_actions(seed, k, envs) for k in range(TRACE)])).cuda()


def _masks(seed, envs, prob):
    rng = np.random.default_rng(seed + 1000)
    return torch.from_numpy((rng.random((TRACE, envs)) < prob).astype(np.uint8)).cuda()


def _addrs(seed, count):
    rng = np.random.default_rng(seed + 2000)
    return np.sort(rng.choice(np.arange(0xC000, 0xE000), count, replace=False))


def _backend(cart, case, **options):
    options = {"stage": "emulate_only", "render_on_step": False, **options}
    be = HipVecBackend(_rom(cart, case["cart_seed"]), num_envs=case["envs"], frames_per_step=case.get("frames", 1),
                       bootrom=build_bootstub(), **options)  # fmt: skip
    be.reset(seed=0)
    return be


def _scatter(be, seed, kind):
    """Envs that have lived apart: seeded work RAM, or the PPU cart's frame
    counter, from which it takes its scroll position."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    lo, hi = (0xC000, 0xD000) if kind == "wram" else (0xC000, 0xC001)
    be.memory_torch()[:, lo:hi] = torch.randint(0, 256, (be.num_envs, hi - lo), dtype=torch.uint8, device="cuda",
                                                generator=gen)  # fmt: skip


def _settle(case):
    """Steps past the boot image and the cart's setup code: 48 frames."""
    return 48 // case.get("frames", 1)


def prepare(case, seed):
    n, kind = case["envs"], case["kind"]
    s = {"kind": kind, "k": 0}
    if kind == "env":
        return _prepare_env(case, seed, s)
    acts = s["actions"] = _trace(seed, n)
    if kind == "step":
        be = s["be"] = _backend(case["cart"], case, stage=case["stage"])
        s["obs"] = torch.empty((n, 32), device="cuda") if case["stage"] in ("obs_only", "full_step") else None
        s["reward"] = torch.empty((n,), device="cuda") if case["stage"] in ("reward_only", "full_step") else None
        s["addrs"] = _addrs(seed, SENSES)
        s["senses"] = torch.empty((n, SENSES), dtype=torch.uint8, device="cuda")
    elif kind == "rollout":
        be = s["be"] = _backend("c3", case, render_pixels=not case["packed"], render_pixels_packed=case["packed"])
        s["pixels"] = torch.empty((n, 72, 20), dtype=torch.uint8, device="cuda") if case["packed"] else None
        s["masks"] = s["cache"] = s["senses"] = None
        if case["reset"] > 0:
            s["cache"] = ResetCache.from_backend(be, env_idx=0)
            s["masks"] = _masks(seed, n, case["reset"])
        if case["senses"]:
            s["addrs"] = _addrs(seed, case["senses"])
            s["senses"] = torch.empty((n, case["senses"]), dtype=torch.uint8, device="cuda")
    elif kind == "host":
        be = s["be"] = _backend("c3", case, stage="full_step", render_pixels=True, render_on_step=True)
        s["host_actions"] = acts.cpu().numpy()
    elif kind == "readout":
        be = s["be"] = _backend("c2", {**case, "frames": 4})
        rng = np.random.default_rng(seed + 3000)
        s["span"] = case["span"]
        s["lo"] = int(rng.integers(0xC000, 0xE000 - case["span"]))
        s["at"] = [int(a) for a in rng.choice(np.arange(0xC000, 0xE000), 3, replace=False)]
        s["value"] = torch.from_numpy(rng.integers(0, 256, (n, 2), dtype=np.uint8)).cuda()
    else:
        be = s["be"] = _backend(case["cart"], case)
    if kind not in ("rollout", "host"):
        _scatter(be, seed, "wram")
    # a rollout some way in: its restored envs run out of phase with the others
    steps = 96 if kind == "rollout" and case["reset"] > 0 else 12 if kind == "readout" else _settle(case)
    for k in range(steps):
        be.step_torch(acts[k % TRACE])
        if s.get("cache") is not None:
            s["cache"].apply_mask_torch(s["masks"][k % TRACE])
    if kind in ("rollout", "host"):
        _scatter(be, seed, "counter")
    return s


def _prepare_env(case, seed, s):
    n = case["envs"]
    rng = np.random.default_rng(seed + 4000)
    goal = torch.from_numpy(rng.integers(0, 256, (1, 72, 20), dtype=np.uint8)).cuda()

    def reward(env, pixels, senses):
        # progress towards the goal frame; an env on its goal frame ends
        d = packed_l1_distance(pixels, goal)
        return 1.0 - d, d == 0

    env = s["env"] = PackedPixelEnv(
        _rom("c3", case["cart_seed"]), num_envs=n, frames_per_step=case["frames"],
        sense_addrs=[int(a) for a in _addrs(seed, 5)], reward_fn=reward, bootrom=build_bootstub(),
    )  # fmt: skip
    env.reset(seed=seed)
    s["actions"] = _trace(seed, n)
    s["ends"] = _masks(seed, n, case["reset"]).bool()  # episodes ended from outside
    s["slots"] = torch.empty((TRACE, n, 1, 72, 20), dtype=torch.uint8, device="cuda")
    for _ in range(_settle(case)):
        run(s)
    _scatter(env.backend, seed, "counter")
    return s


def run(s):
    k = s["k"] = (s["k"] + 1) % TRACE
    kind = s["kind"]
    if kind == "env":
        env, slot = s["env"], s["slots"][k]
        _, reward, terminated, truncated, _ = env.step(s["actions"][k], pixels_out=slot)
        done = terminated | truncated | s["ends"][k]
        env.reset_mask(done, pixels=slot)
        return {"pixels": slot, "senses": env.obs["senses"], "reward": reward, "done": done}
    be = s["be"]
    if kind == "step":
        be.step_torch(s["actions"][k])
        if s["obs"] is not None:
            s["obs"].copy_(be.obs_torch())
        if s["reward"] is not None:
            s["reward"].copy_(be.reward_torch())
        return [be.ram_senses_torch(s["addrs"], out=s["senses"]), s["obs"], s["reward"]]
    if kind == "rollout":
        be.step_torch(s["actions"][k])
        if s["pixels"] is not None:
            pixels = s["pixels"]
            be.render_pixels_snapshot_packed_to_torch(pixels, 0)
        else:
            be.render_pixels_snapshot()
            pixels = _kept(be, be.pixels_torch())
        if s["cache"] is not None:
            s["cache"].apply_mask_torch(s["masks"][k])
        if s["senses"] is not None:
            be.ram_senses_torch(s["addrs"], out=s["senses"])
        return [pixels, s["senses"]]
    if kind == "host":
        obs, reward, done, trunc, _ = be.step(s["host_actions"][k])
        return [obs, reward, done, trunc, _kept(be, be.pixels_torch())]
    if kind == "readout":
        mem, lo = be.memory_torch(), s["lo"]
        a, b, c = s["at"]
        out = [mem[:, lo : lo + s["span"]], mem[:, a], mem[:, b], mem[:, c : c + 2]]
        mem[:, 0xDFF0:0xDFF2] = s["value"]
        return out
    be.step_torch(s["actions"][k])
    regs = be.get_cpu_state(0)
    return [be.state_hash_torch(), regs, np.frombuffer(be.read_memory(0, 0xC000, 0xE000), dtype=np.uint8)]


def work(case):
    """Bytes: per-env state and memory a pass reads and writes at least once,
    inputs and outputs.  Operations: one per emulated machine cycle."""
    n, kind = case["envs"], case["kind"]
    frames = {"readout": 0, "verify": 1}.get(kind, case.get("frames", 1))
    b = n * (2 * STATE_BYTES + 4) if frames else 0
    if kind == "step":
        b += n * (SENSES * 2 + {"emulate_only": 0, "obs_only": 128, "reward_only": 4, "full_step": 132}[case["stage"]])
    elif kind == "rollout":
        # a render reads a frame's tiles, maps and sprites once
        b += n * (8364 + (PACKED if case["packed"] else UNPACKED) + 2 * case["senses"])
        b += int(n * case["reset"]) * (0x4200 + 1024)
    elif kind == "env":
        b += n * (8364 + 2 * PACKED + 16) + int(n * case["reset"]) * (0x4200 + 1024 + PACKED)
    elif kind == "host":
        b += n * (8364 + UNPACKED + 128)
    elif kind == "readout":
        b += 2 * n * (case["span"] + 4) + 2 * n * 2
    elif kind == "verify":
        b += n * (65536 + 8) + 2 * 8192
    return {"bytes": b, "flops": n * frames * CYCLES_PER_FRAME}


def tolerance(case):
    # one 32-bit division and one subtraction of whole numbers
    return {"rel": 3e-7} if case["kind"] == "env" else "exact"


def exact(case, seed):
    return None


def _kept(be, buf):
    """The backend's own buffer as an output that keeps the backend alive."""
    out = buf.view(buf.shape)
    out.owner = be
    return out
