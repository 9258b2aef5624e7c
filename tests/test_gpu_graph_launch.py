"""gps_graph_launch into a stream that is being captured, and with an error of
an earlier HIP call pending: one graph per kernel that a replay can launch (a
single tile, one round, persistent)."""
import ctypes

import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

import gpuprefixsums_amd as gps  # noqa: E402
from tests.gpu_util import to_dev  # noqa: E402

SIZES = [777, (1 << 20) + 1, (1 << 23) + 5]
SEGMENTS = 37


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if not torch.cuda.is_available():
        pytest.fail("GPU tests need a ROCm device")


class Replay:
    def __init__(self, n):
        cuts = np.linspace(0, n, SEGMENTS + 1).astype(np.uint64)
        x = oracle.gen_u32(n, n, 32)
        self.want = torch.from_numpy(oracle.segmented_scan_u32(x, cuts, False).view(np.int32)).cuda()
        self.x, self.off = to_dev(x), torch.from_numpy(cuts.view(np.int64)).cuda()
        self.out = torch.empty(n, dtype=torch.int32, device="cuda")
        self.h = gps.ScanHandle(gps.ALGO_CSDL, n)
        self.g = self.h.segmented_graph(self.x, self.out, self.off, SEGMENTS, n, False)
        torch.cuda.synchronize()

    def right(self):
        torch.cuda.synchronize()
        return torch.equal(self.out, self.want)

    def close(self):
        torch.cuda.synchronize()
        self.g.close()
        assert self.h.device_error() == 0
        self.h.close()


@pytest.mark.parametrize("n", SIZES)
def test_replay_recorded_by_a_capture(n):
    r = Replay(n)
    s = torch.cuda.Stream()
    outer = torch.cuda.CUDAGraph()
    with torch.cuda.graph(outer, stream=s):
        r.out.fill_(-7)
        r.g.launch(s)
    for _ in range(4):
        outer.replay()
        assert r.right()
        r.out.fill_(-7)
        torch.cuda.synchronize()
        r.g.launch(s)  # between the replays, on its own
        assert r.right()
    del outer
    r.close()


@pytest.mark.parametrize("n", SIZES)
def test_replay_with_an_error_pending(n):
    hip = ctypes.CDLL("libamdhip64.so")
    r = Replay(n)
    for _ in range(3):
        r.out.fill_(-7)
        torch.cuda.synchronize()
        assert hip.hipSetDevice(999) != 0  # no such device: the host refuses it
        pending = hip.hipPeekAtLastError()
        assert pending != 0
        r.g.launch()
        assert hip.hipGetLastError() == pending  # still the caller's
        assert r.right()
    r.close()


def test_capture_with_an_error_pending_is_refused():
    """hipGraphLaunch would record nothing and report success."""
    hip = ctypes.CDLL("libamdhip64.so")
    r = Replay(SIZES[0])
    s = torch.cuda.Stream()
    outer = torch.cuda.CUDAGraph()
    with torch.cuda.graph(outer, stream=s):
        r.out.fill_(-7)
        assert hip.hipSetDevice(999) != 0
        pending = hip.hipPeekAtLastError()
        with pytest.raises(gps.GpsError, match="pending"):
            r.g.launch(s)
        assert hip.hipGetLastError() == pending
        r.g.launch(s)
    outer.replay()
    assert r.right()
    del outer
    r.close()
