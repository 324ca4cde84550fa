"""The numbers behind the exchange tags (mhc_pre_internal.h: LaunchTag), modelled on the CPU."""
from __future__ import annotations

import random
import re
from pathlib import Path

SRC = (Path(__file__).resolve().parents[1] / "mhcpre-review_amd" / "csrc" / "mhc_pre_internal.h").read_text()


def _const(name):
    return int(re.search(rf"{name} = (0x[0-9A-Fa-f]+|\d+)", SRC).group(1), 0)


CAPTURED, BITS, FILLED = _const("kCapturedNumbers"), _const("kReplayBits"), _const("kFilledNumbers")


def _mix32(v):
    v ^= v >> 16
    v = v * 0x85EBCA6B & 0xFFFFFFFF
    v ^= v >> 13
    v = v * 0xC2B2AE35 & 0xFFFFFFFF
    return v ^ v >> 16


def test_kinds_of_launches_share_no_number():
    """Eager launches, replays of captured ones and filled words each have a
    part of the 32-bit numbers, and the hash keeps numbers apart."""
    rng = random.Random(1)
    eager = {i & ~CAPTURED & 0xFFFFFFFF for i in (0, 1, CAPTURED - 1, CAPTURED, 0xFFFFFFFF)}
    eager |= {rng.getrandbits(32) & ~CAPTURED & 0xFFFFFFFF for _ in range(20000)}
    nodes = [0, 1, 2, (1 << 19) - 1, 1 << 19] + [rng.getrandbits(19) for _ in range(40)]
    seeds = {CAPTURED | (c << BITS & 0xFFFFFFFF & ~FILLED) for c in nodes}
    replays = {s | r & (1 << BITS) - 1 for s in seeds for r in range(1 << BITS)}
    assert len(replays) == len(seeds) << BITS  # a launch's replays keep clear of the other launches'
    filled = {FILLED | i for i in (0, 1, 2, FILLED ^ 0xFFFFFFFF)} | {FILLED | rng.getrandbits(30) for _ in range(20000)}
    assert all(n < CAPTURED for n in eager)
    assert all(CAPTURED <= n < FILLED for n in replays)
    assert all(n >= FILLED for n in filled)
    every = eager | replays | filled
    assert len({_mix32(n) for n in every}) == len(every)


def test_neighbouring_replays_differ():
    """What a replay finds at its own places is the previous replay's: their
    numbers differ, also where the count wraps."""
    for r in (0, 1, (1 << BITS) - 1, (1 << 31) - 2):
        now, then = (r + 1) & 0x7FFFFFFF, r
        assert now & (1 << BITS) - 1 != then & (1 << BITS) - 1
