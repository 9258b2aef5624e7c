"""Scans whose output begins one element before the input and overlaps it, and
carry words inside the output: with one tile, with as many as a one-round scan
takes (where a wave may sum a missing tile at once: a spin limit of one poll),
and on a default handle. Sums are of integers, exact in any order."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

import gpuprefixsums_amd as gps  # noqa: E402
from tests.gpu_util import first_mismatch, to_dev  # noqa: E402

TILE = 4096
SIZES = [5, TILE, 2 * TILE + 3, 65 * TILE, 300 * TILE - 1]
HANDLES = {"default": {}, "tile": dict(block_threads=256, vec_per_thread=4, schedule=gps.SCHEDULE_TILE, spin_limit=1)}


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if not torch.cuda.is_available():
        pytest.fail("GPU tests need a ROCm device")


def u32(t) -> np.ndarray:
    torch.cuda.synchronize()
    return t.cpu().numpy().view(np.uint32)


@pytest.mark.parametrize("name", HANDLES)
def test_shifted_u32(name):
    with gps.ScanHandle(gps.ALGO_CSDL, max(SIZES), **HANDLES[name]) as h:
        for k, n in enumerate(SIZES):
            x, inclusive = oracle.gen_u32(k, n, 32), k % 2 == 0
            buf = to_dev(np.r_[np.zeros(1, np.uint32), x])
            h.scan(buf[1:], buf[:-1], n, inclusive)
            got, want = u32(buf[:-1]), oracle.scan_u32(x, inclusive)
            assert np.array_equal(got, want), (n, first_mismatch(got, want))
        assert h.device_error() == 0


@pytest.mark.parametrize("name", HANDLES)
@pytest.mark.parametrize("comp", [gps.FP_PAIR, gps.FP_PLAIN], ids=["pair", "plain"])
def test_shifted_f32(name, comp):
    with gps.ScanHandle(gps.ALGO_CSDL, max(SIZES), **HANDLES[name]) as h:
        for k, n in enumerate(SIZES):
            x = np.random.default_rng(k).integers(-1, 2, n).astype(np.float32)
            buf = to_dev(np.r_[np.zeros(1, np.float32), x])
            h.inclusive_f32(buf[1:], buf[:-1], n, comp)
            torch.cuda.synchronize()
            assert np.array_equal(buf[:-1].cpu().numpy(), np.cumsum(x, dtype=np.float64)), n
        assert h.device_error() == 0


@pytest.mark.parametrize("schedule", [gps.SCHEDULE_DEFAULT, gps.SCHEDULE_TILE], ids=["default", "tile"])
def test_shifted_structs(schedule):
    shape = dict(block_threads=512, vec_per_thread=8) if schedule else {}
    with gps.ScanHandle(gps.ALGO_CSDL, max(SIZES), schedule=schedule, spin_limit=1, **shape) as h:
        for k, n in enumerate(SIZES):
            x = oracle.gen_u32(k, 4 * n, 32)
            buf = to_dev(np.r_[np.zeros(4, np.uint32), x])
            h.scan_u32x4(buf[4:], buf[:-4], n, True)
            want = np.cumsum(x.reshape(n, 4), axis=0, dtype=np.uint32).ravel()
            assert np.array_equal(u32(buf[:-4]), want), n
        assert h.device_error() == 0


@pytest.mark.parametrize("name", HANDLES)
@pytest.mark.parametrize("place", ["first", "last"])
def test_carry_in_inside_the_output(name, place):
    with gps.ScanHandle(gps.ALGO_CSDL, max(SIZES), **HANDLES[name]) as h:
        for k, n in enumerate(SIZES):
            x, first = oracle.gen_u32(k, n, 32), 0x9E3779B9
            out = to_dev(np.full(n, first, np.uint32))
            after = torch.zeros(1, dtype=torch.int32, device="cuda")
            word = out[:1] if place == "first" else out[-1:]
            h.scan_carry(to_dev(x), out, n, True, word, after)
            want = oracle.scan_u32(x, True) + np.uint32(first)
            got = u32(out)
            assert np.array_equal(got, want), (n, first_mismatch(got, want))
            assert int(after.item()) & 0xFFFFFFFF == int(want[-1])
        assert h.device_error() == 0


def cuts_of(n):
    """Segments none of which begins where a tile does, so that every tile
    waits for the one before it."""
    return np.array([0, *(c for c in (3, 5000, 8191, 100001, 700001) if c < n), n], dtype=np.uint64)


@pytest.mark.parametrize("name", HANDLES)
@pytest.mark.parametrize("whole", [True, False], ids=["one", "several"])
def test_shifted_segmented_u32(name, whole):
    with gps.ScanHandle(gps.ALGO_CSDL, max(SIZES), **HANDLES[name]) as h:
        for k, n in enumerate(SIZES):
            x, inclusive = oracle.gen_u32(k, n, 32), k % 2 == 0
            off = np.array([0, n], np.uint64) if whole else cuts_of(n)
            buf = to_dev(np.r_[np.zeros(1, np.uint32), x])
            h.segmented(buf[1:], buf[:-1], to_dev(off), off.size - 1, n, inclusive)
            got, want = u32(buf[:-1]), oracle.segmented_scan_u32(x, off, inclusive)
            assert np.array_equal(got, want), (n, first_mismatch(got, want))
        assert h.device_error() == 0


@pytest.mark.parametrize("name", HANDLES)
@pytest.mark.parametrize("comp", [gps.FP_PAIR, gps.FP_PLAIN], ids=["pair", "plain"])
def test_shifted_segmented_f32(name, comp):
    with gps.ScanHandle(gps.ALGO_CSDL, max(SIZES), **HANDLES[name]) as h:
        for k, n in enumerate(SIZES):
            x, off = np.random.default_rng(k).integers(-1, 2, n).astype(np.float32), cuts_of(n)
            buf = to_dev(np.r_[np.zeros(1, np.float32), x])
            h.segmented_fp(buf[1:], buf[:-1], to_dev(off), off.size - 1, n, False, comp)
            torch.cuda.synchronize()
            want = np.concatenate([np.cumsum(x[int(a):int(b)], dtype=np.float64) for a, b in zip(off, off[1:])])
            assert np.array_equal(buf[:-1].cpu().numpy(), want), n
        assert h.device_error() == 0
