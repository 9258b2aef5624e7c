"""Scans of buffers that start at any element: the tiles move 16-byte (BF16
input: 8-byte) vectors from element-aligned addresses, and in a partial tile
only the lane that straddles n moves single elements. Every pair of input and
output offsets, at remainders 0..5 around a tile edge, with guards on both
sides of the output; integer-valued floats keep every sum exact."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

import gpuprefixsums_amd as gps  # noqa: E402
from tests.gpu_util import first_mismatch, to_dev  # noqa: E402

TILE = 4096  # 256 threads x 4 vectors
GUARD = 16
HANDLES = {
    "csdl_tile": dict(algo=gps.ALGO_CSDL, schedule=gps.SCHEDULE_TILE),
    "csdl_persistent": dict(algo=gps.ALGO_CSDL, schedule=gps.SCHEDULE_PERSISTENT),
    "csdl_control": dict(algo=gps.ALGO_CSDL, schedule=gps.SCHEDULE_CONTROL),
    "csdldf": dict(algo=gps.ALGO_CSDLDF),
    "csdldf_stall2": dict(algo=gps.ALGO_CSDLDF, stall_period=2),
    "csdldf_persistent_stall7": dict(algo=gps.ALGO_CSDLDF, schedule=gps.SCHEDULE_PERSISTENT, stall_period=7),
    "rts": dict(algo=gps.ALGO_RTS),
}
SIZES = [1, 2, 3, 4, 5] + [t * TILE + r for t in (1, 3) for r in range(6)]


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if not torch.cuda.is_available():
        pytest.fail("GPU tests need a ROCm device")


def shifted(x: torch.Tensor, shift: int) -> torch.Tensor:
    """x at `shift` elements into an aligned buffer of its own."""
    b = torch.full((x.numel() + shift,), -7, dtype=x.dtype, device="cuda")
    b[shift:] = x
    return b[shift:]


def guarded(n: int, shift: int, dtype) -> tuple:
    b = torch.full((GUARD + shift + n + GUARD,), -7, dtype=dtype, device="cuda")
    return b, b[GUARD + shift:]


def check_guards(b: torch.Tensor, n: int, shift: int) -> None:
    assert bool((b[:GUARD + shift] == -7).all()) and bool((b[GUARD + shift + n:] == -7).all()), "wrote outside"


@pytest.mark.parametrize("name", HANDLES)
@pytest.mark.parametrize("shift_in", range(4))
@pytest.mark.parametrize("shift_out", range(4))
def test_u32_at_every_offset(name, shift_in, shift_out):
    with gps.ScanHandle(max_n=max(SIZES), block_threads=256, vec_per_thread=4, **HANDLES[name]) as h:
        for k, n in enumerate(SIZES):
            x = oracle.gen_u32(100 + k, n, 32)
            buf, out = guarded(n, shift_out, torch.int32)
            h.scan(shifted(to_dev(x), shift_in), out, n, k % 2 == 0)
            torch.cuda.synchronize()
            got, want = out[:n].cpu().numpy().view(np.uint32), oracle.scan_u32(x, k % 2 == 0)
            assert np.array_equal(got, want), (n, first_mismatch(got, want))
            check_guards(buf, n, shift_out)
        assert h.device_error() == 0


@pytest.mark.parametrize("schedule", [gps.SCHEDULE_TILE, gps.SCHEDULE_PERSISTENT], ids=["tile", "persistent"])
@pytest.mark.parametrize("comp", [gps.FP_PAIR, gps.FP_PLAIN], ids=["pair", "plain"])
@pytest.mark.parametrize("bf16", [False, True], ids=["f32", "bf16"])
@pytest.mark.parametrize("segmented", [False, True], ids=["whole", "segmented"])
def test_fp_at_every_offset(schedule, comp, bf16, segmented):
    rng = np.random.default_rng(5)
    with gps.ScanHandle(gps.ALGO_CSDL, max(SIZES), block_threads=256, vec_per_thread=4, schedule=schedule) as h:
        for k, n in enumerate(SIZES):
            x = torch.from_numpy(rng.integers(-8, 9, n)).to(torch.bfloat16 if bf16 else torch.float32).cuda()
            cuts = sorted({0, n, *(int(c) for c in rng.integers(0, n + 1, 5))}) if segmented else [0, n]
            want = torch.cat([torch.cumsum(x[a:b].double(), 0) for a, b in zip(cuts, cuts[1:])])
            off = torch.tensor(cuts, dtype=torch.int64, device="cuda")
            for shift_in in range(4):
                for shift_out in range(4):
                    src = shifted(x, shift_in)
                    buf, out = guarded(n, shift_out, torch.float32)
                    if segmented:
                        h.segmented_fp(src, out, off, len(cuts) - 1, n, bf16, comp)
                    elif bf16:
                        h.inclusive_bf16_f32(src, out, n, comp)
                    else:
                        h.inclusive_f32(src, out, n, comp)
                    torch.cuda.synchronize()
                    assert torch.equal(out[:n].double(), want), (n, shift_in, shift_out)
                    check_guards(buf, n, shift_out)
        assert h.device_error() == 0


@pytest.mark.parametrize("schedule", [gps.SCHEDULE_TILE, gps.SCHEDULE_PERSISTENT], ids=["tile", "persistent"])
@pytest.mark.parametrize("inclusive", [False, True], ids=["excl", "incl"])
def test_segmented_u32_at_every_offset(schedule, inclusive):
    rng = np.random.default_rng(6)
    with gps.ScanHandle(gps.ALGO_CSDL, max(SIZES), block_threads=256, vec_per_thread=4, schedule=schedule) as h:
        for k, n in enumerate(SIZES):
            x = oracle.gen_u32(200 + k, n, 32)
            off = np.array(sorted({0, n, *(int(c) for c in rng.integers(0, n + 1, 5))}), dtype=np.uint64)
            want = oracle.segmented_scan_u32(x, off, inclusive)
            for shift_in in range(4):
                for shift_out in range(4):
                    buf, out = guarded(n, shift_out, torch.int32)
                    h.segmented(shifted(to_dev(x), shift_in), out, to_dev(off), off.size - 1, n, inclusive)
                    torch.cuda.synchronize()
                    got = out[:n].cpu().numpy().view(np.uint32)
                    assert np.array_equal(got, want), (n, shift_in, shift_out, first_mismatch(got, want))
                    check_guards(buf, n, shift_out)
        assert h.device_error() == 0


@pytest.mark.parametrize("inclusive", [False, True], ids=["excl", "incl"])
@pytest.mark.parametrize("block,vec", [(256, 2), (512, 2), (1024, 8)])
def test_rts_with_and_without_the_spine(block, vec, inclusive):
    """Tile counts around the last one whose rescan adds up the tile sums by
    itself (16384), and around the spine's rounds of 32768 sums."""
    tile = block * vec * 4
    counts = [1, 2, 511, 513, 16384, 16385] + ([32768, 32769] if tile <= 4096 else [])
    n_max = max(counts) * tile
    x = torch.empty(n_max + 1, dtype=torch.int32, device="cuda")
    gps.fill_random_u32(x, n_max + 1, seed=9)
    out = torch.empty(n_max, dtype=torch.int32, device="cuda")
    with gps.ScanHandle(gps.ALGO_RTS, n_max, block_threads=block, vec_per_thread=vec) as h:
        for c in counts:
            for n in (c * tile - 3, c * tile):
                h.scan(x[1:], out, n, inclusive)
                assert gps.validate_scan_u32(x[1:], out, n, inclusive) == 0, (c, n)
