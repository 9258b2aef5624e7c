"""The spin limit that a chained-scan handle reports is the one it was given, 4
by default, and makes another handle that reports the same."""
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

import gpuprefixsums_amd as gps  # noqa: E402


@pytest.mark.parametrize("schedule", [gps.SCHEDULE_DEFAULT, gps.SCHEDULE_TILE, gps.SCHEDULE_PERSISTENT])
@pytest.mark.parametrize("spin", [0, 1, 4, 9])
def test_reported_spin_limit(schedule, spin):
    if not torch.cuda.is_available():
        pytest.fail("GPU tests need a ROCm device")
    with gps.ScanHandle(gps.ALGO_CSDL, 1 << 20, schedule=schedule, spin_limit=spin) as h:
        assert h.spin_limit == (spin or 4)
        with gps.ScanHandle(gps.ALGO_CSDL, 1 << 20, block_threads=h.block_threads, vec_per_thread=h.vec_per_thread,
                            schedule=h.schedule, spin_limit=h.spin_limit) as same:
            assert same.spin_limit == h.spin_limit
