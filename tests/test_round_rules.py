"""Which calls may run the one-round scans (gpuprefixsums_amd/csrc/round_rules.hpp):
the host rules, compiled with the host compiler, and a model of what they keep
apart. No GPU."""
import random
import shutil
import subprocess
from collections import Counter
from pathlib import Path

import pytest

from tests.test_protocol_model import AGG, MASK32, make_status
from tests.test_round_model import TILE, Memory, window

CSRC = Path(__file__).resolve().parents[1] / "gpuprefixsums_amd" / "csrc"


def holds(tmp_path, *conditions):
    """Compiles and evaluates conditions on the rules; `at(k)` is byte k of a buffer."""
    cxx = shutil.which("g++") or shutil.which("c++")
    assert cxx, "no host C++ compiler"
    src, exe = tmp_path / "rules.cpp", tmp_path / "rules"
    checks = "\n".join(f"    if (!({c})) return {k + 1};" for k, c in enumerate(conditions))
    src.write_text('#include "round_rules.hpp"\nusing namespace gps;\n'
                   "[[maybe_unused]] static const uint32_t* at(uint64_t k) { return reinterpret_cast<const uint32_t*>(4096 + k); }\n"
                   f"int main() {{\n{checks}\n    return 0;\n}}\n")
    subprocess.run([cxx, "-std=c++17", "-Wall", "-Werror", f"-I{CSRC}", str(src), "-o", str(exe)], check=True)
    k = subprocess.run([str(exe)]).returncode
    assert k == 0, conditions[k - 1]


def test_buffers(tmp_path):
    holds(tmp_path,
          "round_buffers(at(0), 400, at(0), 400)",                 # in place
          "round_buffers(at(0), 400, at(400), 400)",               # back to back, either way round
          "round_buffers(at(400), 400, at(0), 400)",
          "!round_buffers(at(4), 400, at(0), 400)",                # shifted by one element, either way
          "!round_buffers(at(0), 400, at(4), 400)",
          "!round_buffers(at(396), 400, at(0), 400)",              # by all but one
          "!round_buffers(at(0), 200, at(0), 400)",                # a BF16 input at the start of its output
          "!round_buffers(at(200), 200, at(0), 400)")


def test_carry_words(tmp_path):
    holds(tmp_path,
          "round_carries(nullptr, nullptr, at(0), at(0), 400)",
          "round_carries(at(800), at(804), at(0), at(400), 400)",
          "round_carries(at(0), nullptr, at(0), at(400), 400)",    # read only: anywhere but the output
          "round_carries(at(396), at(800), at(0), at(400), 400)",  # the word before the output: a chunk's last result
          "!round_carries(at(800), at(800), at(0), at(400), 400)",
          "!round_carries(at(400), nullptr, at(0), at(400), 400)",
          "!round_carries(at(796), at(900), at(0), at(400), 400)",
          "!round_carries(nullptr, at(0), at(0), at(400), 400)",   # written: anywhere but input and output
          "!round_carries(nullptr, at(796), at(0), at(400), 400)")


def test_patience(tmp_path):
    """Spin limits as they were given before the one-round scans, and as a
    handle reports them (4 by default), leave the patience at 64 polls; only a
    tile-schedule handle asks for less."""
    holds(tmp_path,
          "kRoundPatience == 64",
          *(f"round_patience(false, {s}) == 64" for s in (1, 2, 3, 4, 32, 65536)),
          *(f"round_patience(true, {s}) == {p}" for s, p in ((1, 1), (2, 4), (3, 16), (4, 64), (5, 64), (65536, 64))))


def shifted_tile(mem, t, epoch, patience, stats):
    """A workgroup of a one-round scan whose output begins one element before
    its input (tests/test_round_model.py's tile_scan without the epoch's part)."""
    x = mem.data[t * TILE:(t + 1) * TILE]
    yield
    mem.status[t] = make_status(sum(x), AGG, epoch)
    yield
    prefix = 0
    for top in range(t - 1, -1, -64):
        prefix += yield from window(mem, top, epoch, patience, stats)
    for i, v in enumerate(x, t * TILE):
        prefix += v
        if i:
            mem.data[i - 1] = prefix & MASK32
        else:
            mem.before = prefix & MASK32
        yield


@pytest.mark.parametrize("order,right", [("ascending", True), ("reversed", False)])
def test_a_shifted_output_needs_the_tiles_in_order(order, right):
    """With one workgroup at a time: in ticket order (each starts after the
    ones before it have loaded) the sums are right; out of it a wave sums tiles
    that have not started, and its workgroup's output replaces their input."""
    rng = random.Random(1)
    tiles = 12
    x = [rng.getrandbits(32) for _ in range(tiles * TILE)]
    mem, stats = Memory(tiles), Counter()
    mem.data = list(x)
    for t in (range(tiles) if order == "ascending" else reversed(range(tiles))):
        for _ in shifted_tile(mem, t, 1, 2, stats):
            pass
    want, total = [], 0
    for v in x:
        total = (total + v) & MASK32
        want.append(total)
    assert ([mem.before, *mem.data[:-1]] == want) is right
    assert (stats["helped"] == 0) is right
