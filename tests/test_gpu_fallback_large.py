"""Decoupled fallback under emulated deadlock above 3 * 2^25 elements, where
half of each tile waits in LDS for its prefix: both sides of the line, both
scans, in place and at an offset, and the fallback counters."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

import gpuprefixsums_amd as gps  # noqa: E402
from tests.gpu_util import first_mismatch, to_dev  # noqa: E402

LINE = 3 << 25
TILE = 32768


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if not torch.cuda.is_available():
        pytest.fail("GPU tests need a ROCm device")


@pytest.mark.parametrize("n,period,inclusive,in_place,shift", [
    (LINE, 7, True, False, 0),
    (LINE + 1, 7, True, False, 0),
    (LINE + 1, 7, False, True, 0),
    (LINE + TILE - 3, 8, True, False, 1),
    (LINE + TILE + 5, 2, False, False, 3),
])
def test_stalled_tiles(n, period, inclusive, in_place, shift):
    x = oracle.gen_u32(period, n + shift, 32)
    d_in = to_dev(x)[shift:]
    out = d_in if in_place else torch.full_like(d_in, -7)
    with gps.ScanHandle(gps.ALGO_CSDLDF, n, stall_period=period) as h:
        h.reset_counters()
        h.scan(d_in, out, n, inclusive)
        torch.cuda.synchronize()
        got, want = out.cpu().numpy().view(np.uint32), oracle.scan_u32(x[shift:], inclusive)
        assert np.array_equal(got, want), first_mismatch(got, want)
        assert h.device_error() == 0
        tiles = (n + TILE - 1) // TILE
        stalled = (tiles - 1 + period - 1) // period  # the last tile never stalls
        c = h.counters()
        assert stalled <= c["insertions"] <= c["fallbacks"] and c["polls"] >= tiles - 1 and c["stall_timeouts"] == 0
