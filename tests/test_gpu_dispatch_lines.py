"""Explicit handles on both sides of the lines where a scan changes its kernel."""
import pytest

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
