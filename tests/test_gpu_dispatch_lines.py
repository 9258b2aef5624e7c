"""Explicit handles on both sides of the lines where a scan changes its kernel."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

import gpuprefixsums_amd as gps  # noqa: E402


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if not torch.cuda.is_available():
        pytest.fail("GPU tests need a ROCm device")


@pytest.fixture(scope="module")
def words():
    """Random words, and a place for the result."""
    n = (1 << 25) + (1 << 16)
    x = torch.empty(n, dtype=torch.int32, device="cuda")
    gps.fill_random_u32(x, n, seed=11)
    return x, torch.empty_like(x)


def scan_and_validate(h, words, n, inclusive):
    x, out = words
    h.scan(x, out, n, inclusive)
    assert gps.validate_scan_u32(x, out, n, inclusive) == 0, n
    assert h.device_error() == 0


@pytest.mark.parametrize("inclusive", [False, True], ids=["excl", "incl"])
def test_rts_small_tiles(words, inclusive):
    """256 x 2: the rescan adds up the sums of up to 8192 tiles."""
    tile = 2048
    with gps.ScanHandle(gps.ALGO_RTS, 8193 * tile, block_threads=256, vec_per_thread=2) as h:
        for n in (8192 * tile, 8192 * tile + 1, 8193 * tile):
            scan_and_validate(h, words, n, inclusive)


@pytest.mark.parametrize("block", [256, 512, 1024])
@pytest.mark.parametrize("schedule", [gps.SCHEDULE_TILE, gps.SCHEDULE_PERSISTENT], ids=["tile", "persistent"])
@pytest.mark.parametrize("period", [0, 7])
def test_fallback_vec4(words, block, schedule, period):
    """VEC 4 at 2^25 elements: vectors per fallback round, workgroups per CU."""
    n = 1 << 25
    with gps.ScanHandle(gps.ALGO_CSDLDF, n + 5, block_threads=block, vec_per_thread=4, schedule=schedule,
                        stall_period=period) as h:
        for k, m in enumerate((n, n + 1, n + 5)):
            scan_and_validate(h, words, m, k % 2 == 0)


@pytest.mark.parametrize("block,vec", [(1024, 4), (1024, 8)])
@pytest.mark.parametrize("bf16", [False, True], ids=["f32", "bf16"])
@pytest.mark.parametrize("comp", [gps.FP_PAIR, gps.FP_PLAIN], ids=["pair", "plain"])
def test_fp_round_tiles(block, vec, bf16, comp):
    """1024 threads: pairs take one round up to 256 tiles, plain ones up to 640 or
    1024. Sums of -1, 0 and 1 are exact in any order."""
    tile = block * vec * 4
    lines = [256] if comp == gps.FP_PAIR else [640 if vec == 8 else 1024]
    x = torch.randint(-1, 2, ((lines[-1] + 1) * tile,), device="cuda").to(torch.bfloat16 if bf16 else torch.float32)
    want, out = torch.cumsum(x.double(), 0), torch.empty(x.numel(), device="cuda")
    with gps.ScanHandle(gps.ALGO_CSDL, x.numel(), block_threads=block, vec_per_thread=vec,
                        schedule=gps.SCHEDULE_TILE) as h:
        for k in lines:
            for n in (k * tile, k * tile + 1, (k + 1) * tile - 3):
                out.fill_(-7)
                (h.inclusive_bf16_f32 if bf16 else h.inclusive_f32)(x, out, n, comp)
                assert torch.equal(out[:n].double(), want[:n]), n
        assert h.device_error() == 0


@pytest.mark.parametrize("block,vec", [(512, 8), (1024, 4), (1024, 8)])
@pytest.mark.parametrize("inclusive", [False, True], ids=["excl", "incl"])
def test_struct_round(words, block, vec, inclusive):
    """Structs take one round up to 2^22 of them."""
    x, out = words
    with gps.ScanHandle(gps.ALGO_CSDL, (1 << 22) + 5, block_threads=block, vec_per_thread=vec,
                        schedule=gps.SCHEDULE_TILE) as h:
        for n in (1 << 22, (1 << 22) + 1, (1 << 22) + 5):
            v = x[:4 * n].view(n, 4).long() & 0xFFFFFFFF
            want = torch.cumsum(v, 0)
            if not inclusive:
                want -= v
            out.fill_(-7)
            h.scan_u32x4(x, out, n, inclusive)
            assert torch.equal(out[:4 * n].view(n, 4).long() & 0xFFFFFFFF, want & 0xFFFFFFFF), n
            assert bool((out[4 * n:4 * n + 64] == -7).all())
        assert h.device_error() == 0


@pytest.mark.parametrize("block,vec,line", [(256, 4, 257), (512, 4, 513), (1024, 2, 1024), (1024, 4, 1024), (1024, 8, 256)])
@pytest.mark.parametrize("segments", [1, 3000])
def test_segmented_round_tiles(words, block, vec, line, segments):
    """Segmented scans take one round up to `line` tiles."""
    x, out = words
    tile = block * vec * 4
    with gps.ScanHandle(gps.ALGO_CSDL, (line + 1) * tile, block_threads=block, vec_per_thread=vec,
                        schedule=gps.SCHEDULE_TILE) as h:
        for k, n in enumerate((line * tile, line * tile + 1, (line + 1) * tile - 3)):
            cuts = np.linspace(0, n, segments + 1).astype(np.uint64)
            off = torch.from_numpy(cuts.view(np.int64)).cuda()
            out.fill_(-7)
            h.segmented(x, out, off, segments, n, k % 2 == 0)
            want = oracle.segmented_scan_u32(x[:n].cpu().numpy().view(np.uint32), cuts, k % 2 == 0)
            assert np.array_equal(out[:n].cpu().numpy().view(np.uint32), want), n
        assert h.device_error() == 0


@pytest.mark.parametrize("block,vec,line", [(256, 4, 257), (512, 8, 513), (1024, 4, 512), (1024, 8, 1024)])
@pytest.mark.parametrize("bf16", [False, True], ids=["f32", "bf16"])
def test_segmented_fp_round_tiles(block, vec, line, bf16):
    """Segmented pair scans take one round up to `line` tiles."""
    tile, segments = block * vec * 4, 3000
    x = torch.randint(-1, 2, ((line + 1) * tile,), device="cuda").to(torch.bfloat16 if bf16 else torch.float32)
    c, out = torch.cumsum(x.double(), 0), torch.empty(x.numel(), device="cuda")
    with gps.ScanHandle(gps.ALGO_CSDL, x.numel(), block_threads=block, vec_per_thread=vec,
                        schedule=gps.SCHEDULE_TILE) as h:
        for n in (line * tile, line * tile + 1, (line + 1) * tile - 3):
            off = torch.linspace(0, n, segments + 1, dtype=torch.float64, device="cuda").long()
            before = torch.where(off[:-1] > 0, c[(off[:-1] - 1).clamp(min=0)], torch.zeros_like(c[:segments]))
            want = c[:n] - torch.repeat_interleave(before, off.diff())
            out.fill_(-7)
            h.segmented_fp(x, out, off, segments, n, bf16=bf16, compensated=True)
            assert torch.equal(out[:n].double(), want), n
        assert h.device_error() == 0
