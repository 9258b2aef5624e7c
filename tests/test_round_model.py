"""CPU model of the one-round scan's protocol (gpuprefixsums_amd/csrc/device_common.hpp:
one-round scans; scan_u32.hip: csdl_round_u32), in place, under random
interleavings. No GPU.

Every access to shared memory is one step. Workgroups start in any order, at
most `resident` at a time, so a tile may wait for one that cannot start
before it has ended: only the waiters' own summing of the missing tile ends
such a wait. Several launches reuse the status slots and the ticket word.
"""
import random
from collections import Counter

import pytest

from tests.test_protocol_model import AGG, MASK32, flag_of, make_status

TILE = 3      # elements of a tile
WAVES = 4     # waves of a workgroup: windows are dealt to them in turn
GROUP = 16    # kRoundGroup


class Memory:
    def __init__(self, tiles):
        self.status = [0] * tiles
        self.count = [0] * tiles
        self.ticket = 1 << 32
        self.data = []


def rearm(mem, epoch):
    mem.ticket = (epoch + 1) << 32


def window(mem, top, epoch, patience, stats):
    """One wave: the sum of the aggregates of tiles top, top - 1, ..., at most 64."""
    tiles = list(range(top, max(top - 64, -1), -1))
    value, polls = {}, 0
    while True:
        for j in tiles:
            if j in value:
                continue
            w = mem.status[j]
            yield
            if flag_of(w, epoch):
                value[j] = w & MASK32
        missing = [j for j in tiles if j not in value]
        if not missing:
            return sum(value.values())
        polls += 1
        if polls < patience:
            continue
        j, own = missing[0], 0
        for i in range(j * TILE, (j + 1) * TILE):
            own += mem.data[i]
            yield
        w = mem.status[j]
        yield
        stats["helped" if not flag_of(w, epoch) else "help_overtaken"] += 1
        value[j] = w & MASK32 if flag_of(w, epoch) else own


def tile_scan(mem, t, num_tiles, direct, patience, stats):
    old = mem.ticket
    if num_tiles <= direct:
        mem.ticket += 1
    yield
    epoch = old >> 32
    if num_tiles <= direct and old & MASK32 == num_tiles - 1:
        rearm(mem, epoch)
        yield
    x = mem.data[t * TILE:(t + 1) * TILE]
    yield
    mem.status[t] = make_status(sum(x), AGG, epoch)
    yield
    waves = [window(mem, top, epoch, patience, stats) for top in range(t - 1, -1, -64)]
    prefix, live = 0, list(waves)
    while live:  # the waves of one workgroup, interleaved
        for w in list(live):
            try:
                next(w)
                yield
            except StopIteration as end:
                prefix += end.value
                live.remove(w)
    if num_tiles > direct:  # its last wave counts the workgroup off
        first = t // GROUP * GROUP
        size = min(GROUP, num_tiles - first)
        mem.count[first] = (mem.count[first] + 1) % size
        full = mem.count[first] == 0
        yield
        if full:
            old = mem.ticket
            mem.ticket += 1
            yield
            if old & MASK32 == (num_tiles - 1) // GROUP:
                rearm(mem, old >> 32)
                yield
    for i, v in enumerate(x):  # in place, only after the word above is performed
        prefix += v
        mem.data[t * TILE + i] = prefix & MASK32
        yield


def launch(mem, num_tiles, resident, order, direct, patience, rng, stats):
    waiting = list(range(num_tiles))
    if order == "reversed":
        waiting.reverse()
    elif order == "shuffled":
        rng.shuffle(waiting)
    running = []
    while waiting or running:
        while waiting and len(running) < resident:
            running.append(tile_scan(mem, waiting.pop(0), num_tiles, direct, patience, stats))
        k = rng.randrange(len(running))
        for _ in range(rng.choice([1, 1, 2, 8, 64])):
            try:
                next(running[k])
            except StopIteration:
                running.pop(k)
                break


@pytest.mark.parametrize("order", ["ascending", "reversed", "shuffled"])
@pytest.mark.parametrize("direct", [0, 64], ids=["counted", "ticketed"])
def test_every_start_order_and_residency(order, direct):
    stats = Counter()
    for seed in range(6):
        rng = random.Random(seed)
        mem = Memory(140)
        for k, num_tiles in enumerate([2, 15, 16, 17, 64, 65, 66, 33, 130]):
            x = [rng.getrandbits(32) for _ in range(num_tiles * TILE)]
            mem.data = list(x)
            launch(mem, num_tiles, rng.choice([1, 2, 5, 200]), order, direct, rng.choice([1, 2, 6]), rng, stats)
            total, want = 0, []
            for v in x:
                total = (total + v) & MASK32
                want.append(total)
            assert mem.data == want, (seed, num_tiles)
            assert mem.ticket == (k + 2) << 32 and not any(mem.count), (seed, num_tiles)
    if order != "ascending":
        assert stats["helped"] > 0
    if order == "shuffled":
        assert stats["help_overtaken"] > 0
