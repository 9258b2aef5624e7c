"""Persistent segmented uint32 scans on both sides of the line at which
segments count as long (8192 elements on average): even segments, heads at the
edges of a wave's run and of a tile, and units crowded into one place."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

import gpuprefixsums_amd as gps  # noqa: E402
from tests.gpu_util import first_mismatch, to_dev  # noqa: E402

N = (1 << 23) + 32768 + 5
RUN, TILE = 2048, 32768


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if not torch.cuda.is_available():
        pytest.fail("GPU tests need a ROCm device")


def cuts(kind, segments):
    if kind == "even":
        inner = np.linspace(0, N, segments + 1)[1:-1]
    elif kind == "edges":  # before, at and after run and tile edges
        at = np.r_[np.arange(RUN, N, RUN * 37), np.arange(TILE, N, TILE * 11)]
        inner = np.r_[at - 1, at, at + 1][:segments - 1]
        inner = np.r_[inner, np.full(segments - 1 - inner.size, N)]  # empty segments at the end
    else:  # units, all inside one tile, and a last one at the end
        inner = np.r_[5 * TILE + 100 + np.arange(segments - 2), [N - 1]][:segments - 1]
    return np.r_[0, np.sort(inner.astype(np.int64)), N].astype(np.uint64)


@pytest.mark.parametrize("kind", ["even", "edges", "crowded"])
@pytest.mark.parametrize("segments", [2, N // 8192, N // 8192 + 1])
@pytest.mark.parametrize("inclusive,in_place", [(True, False), (False, False), (False, True)])
def test_both_sides_of_the_line(kind, segments, inclusive, in_place):
    x, off = oracle.gen_u32(segments, N, 32), cuts(kind, segments)
    assert off.size == segments + 1
    d_in = to_dev(x)
    out = d_in if in_place else torch.full_like(d_in, -7)
    d_off = torch.from_numpy(off.view(np.int64)).cuda()
    with gps.ScanHandle(gps.ALGO_CSDL, N) as h:
        h.segmented(d_in, out, d_off, segments, N, inclusive)
        torch.cuda.synchronize()
        got, want = out.cpu().numpy().view(np.uint32), oracle.segmented_scan_u32(x, off, inclusive)
        assert np.array_equal(got, want), first_mismatch(got, want)
        assert h.device_error() == 0
