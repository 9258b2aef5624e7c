"""One-round scans (one workgroup per tile, up to 1024 tiles): tile counts at
the edges of a window of 64, of the ticketed launches and of the kernel's
range, the default handle's kernels on both sides of each size rule, and
workgroups that sum a missing tile by themselves (a spin limit of one poll).
Sums are of integers below 2^24, so every FP result is exact in any order."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

import gpuprefixsums_amd as gps  # noqa: E402
from tests.gpu_util import first_mismatch, to_dev  # noqa: E402

TILE = 4096  # 256 threads x 4 vectors
TILES = [1, 2, 16, 17, 63, 64, 65, 66, 80, 81, 129, 256, 257, 258]
RULES = [1, 2048, 4096, 8192, 16384, 1 << 18, 1 << 19, 1 << 20, 9 << 18, 1 << 21, 3 << 20, 1 << 22, 1 << 23]
SPINS = {"default": 0, "help": 1}


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if not torch.cuda.is_available():
        pytest.fail("GPU tests need a ROCm device")


def check_u32(h, n, seed, inclusive, in_place):
    x = oracle.gen_u32(seed, n, 32)
    d_in = to_dev(x)
    out = d_in if in_place else torch.full_like(d_in, -7)
    h.scan(d_in, out, n, inclusive)
    torch.cuda.synchronize()
    got, want = out.cpu().numpy().view(np.uint32), oracle.scan_u32(x, inclusive)
    assert np.array_equal(got, want), (n, first_mismatch(got, want))


def check_struct(h, n, seed, inclusive, in_place):
    x = oracle.gen_u32(seed, 4 * n, 32)
    d_in = to_dev(x)
    out = d_in if in_place else torch.full_like(d_in, -7)
    h.scan_u32x4(d_in, out, n, inclusive)
    torch.cuda.synchronize()
    got, x = out.cpu().numpy().view(np.uint32).reshape(n, 4), x.reshape(n, 4)
    want = np.cumsum(x, axis=0, dtype=np.uint32)
    if not inclusive:
        want -= x
    assert np.array_equal(got, want), (n, np.flatnonzero((got != want).any(axis=1))[0])


def check_segmented(h, n, seed, inclusive, segments, in_place):
    rng = np.random.default_rng(seed)
    x = oracle.gen_u32(seed, n, 32)
    cuts = np.r_[0, np.sort(rng.integers(0, n + 1, segments - 1)), n].astype(np.uint64)  # some of them empty
    d_in = to_dev(x)
    out = d_in if in_place else torch.full_like(d_in, -7)
    off = torch.from_numpy(cuts.view(np.int64)).cuda()
    h.segmented(d_in, out, off, segments, n, inclusive)
    torch.cuda.synchronize()
    got, want = out.cpu().numpy().view(np.uint32), oracle.segmented_scan_u32(x, cuts, inclusive)
    assert np.array_equal(got, want), (n, first_mismatch(got, want))


def check_fp(h, n, seed, bf16, comp, segments, in_place):
    rng = np.random.default_rng(seed)
    x = torch.from_numpy(rng.integers(-1, 2, n)).to(torch.bfloat16 if bf16 else torch.float32).cuda()
    cuts = np.unique(np.r_[0, rng.integers(0, n + 1, segments - 1), n]) if segments else np.array([0, n])
    c = torch.cumsum(x.double(), 0)
    starts = torch.from_numpy(cuts[:-1]).cuda()
    before = torch.where(starts > 0, c[(starts - 1).clamp(min=0)], torch.zeros_like(c[starts]))
    want = c - torch.repeat_interleave(before, torch.from_numpy(np.diff(cuts)).cuda())
    out = x if in_place else torch.full((n,), -7.0, dtype=torch.float32, device="cuda")
    if segments:
        off = torch.from_numpy(cuts.astype(np.int64)).cuda()
        h.segmented_fp(x, out, off, cuts.size - 1, n, bf16=bf16, compensated=comp)
    elif bf16:
        h.inclusive_bf16_f32(x, out, n, comp)
    else:
        h.inclusive_f32(x, out, n, comp)
    torch.cuda.synchronize()
    bad = torch.nonzero(out.double() != want)
    assert bad.numel() == 0, (n, int(bad[0]), bad.numel())


@pytest.mark.parametrize("in_place", [False, True], ids=["apart", "in_place"])
@pytest.mark.parametrize("spin", SPINS)
def test_u32_tile_counts(spin, in_place):
    with gps.ScanHandle(gps.ALGO_CSDL, 1025 * TILE, block_threads=256, vec_per_thread=4,
                        schedule=gps.SCHEDULE_TILE, spin_limit=SPINS[spin]) as h:
        for k, tiles in enumerate([*TILES, 1023, 1024, 1025]):
            for n in (tiles * TILE, tiles * TILE - 5):
                check_u32(h, n, k, k % 2 == 0, in_place)
        assert h.device_error() == 0


@pytest.mark.parametrize("same_word", [False, True], ids=["two_words", "one_word"])
@pytest.mark.parametrize("spin", SPINS)
def test_u32_carries(spin, same_word):
    with gps.ScanHandle(gps.ALGO_CSDL, 257 * TILE, block_threads=256, vec_per_thread=4,
                        schedule=gps.SCHEDULE_TILE, spin_limit=SPINS[spin]) as h:
        for k, tiles in enumerate([1, 2, 64, 65, 66, 257]):
            n, first = tiles * TILE - 3, 0x9E3779B9
            x = oracle.gen_u32(k, n, 32)
            want = oracle.scan_u32(x, True) + np.uint32(first)
            word = torch.tensor([first - (1 << 32)], dtype=torch.int32, device="cuda")
            after = word if same_word else torch.zeros_like(word)
            d_in = to_dev(x)
            h.scan_carry(d_in, d_in, n, True, word, after)
            torch.cuda.synchronize()
            assert np.array_equal(d_in.cpu().numpy().view(np.uint32), want), tiles
            assert int(after.item()) & 0xFFFFFFFF == int(want[-1])
        assert h.device_error() == 0


@pytest.mark.parametrize("spin", SPINS)
@pytest.mark.parametrize("comp", [gps.FP_PAIR, gps.FP_PLAIN], ids=["pair", "plain"])
@pytest.mark.parametrize("bf16", [False, True], ids=["f32", "bf16"])
@pytest.mark.parametrize("segments", [0, 5, 3000])
def test_fp_tile_counts(spin, comp, bf16, segments):
    with gps.ScanHandle(gps.ALGO_CSDL, 1025 * TILE, block_threads=256, vec_per_thread=4,
                        schedule=gps.SCHEDULE_TILE, spin_limit=SPINS[spin]) as h:
        for k, tiles in enumerate([*TILES, 1024, 1025]):
            for n in (tiles * TILE, tiles * TILE - 5):
                check_fp(h, n, k, bf16, comp, segments, in_place=not bf16 and k % 2 == 1)
        assert h.device_error() == 0


@pytest.mark.parametrize("in_place", [False, True], ids=["apart", "in_place"])
@pytest.mark.parametrize("spin", SPINS)
@pytest.mark.parametrize("segments", [1, 5, 3000])
def test_segmented_u32_tile_counts(spin, in_place, segments):
    with gps.ScanHandle(gps.ALGO_CSDL, 1025 * TILE, block_threads=256, vec_per_thread=4,
                        schedule=gps.SCHEDULE_TILE, spin_limit=SPINS[spin]) as h:
        for k, tiles in enumerate([*TILES, 1025]):
            for n in (tiles * TILE, tiles * TILE - 5):
                check_segmented(h, n, k, k % 2 == 0, segments, in_place)
        assert h.device_error() == 0


@pytest.mark.parametrize("in_place", [False, True], ids=["apart", "in_place"])
@pytest.mark.parametrize("spin", SPINS)
@pytest.mark.parametrize("shape", [(512, 8), (1024, 4)])
def test_struct_tile_counts(spin, in_place, shape):
    with gps.ScanHandle(gps.ALGO_CSDL, 1025 * TILE, block_threads=shape[0], vec_per_thread=shape[1],
                        schedule=gps.SCHEDULE_TILE, spin_limit=SPINS[spin]) as h:
        for k, tiles in enumerate([1, 2, 16, 17, 32, 33, 64, 65, 128, 129, 256, 257, 1024, 1025]):
            for n in (tiles * TILE, tiles * TILE - 5):
                check_struct(h, n, k, k % 2 == 0, in_place)
        assert h.device_error() == 0


def test_default_handle_on_both_sides_of_each_size_rule():
    with gps.ScanHandle(gps.ALGO_CSDL, (1 << 23) + 1) as h:
        for k, edge in enumerate(RULES):
            for n in (edge, edge + 1):
                check_u32(h, n, k, k % 2 == 0, False)
                check_segmented(h, n, k, k % 2 == 1, 2000, k % 2 == 0)
                for bf16 in (False, True):
                    check_fp(h, n, k, bf16, gps.FP_PAIR, 0, False)
                    check_fp(h, n, k, bf16, gps.FP_PLAIN, 2000, False)
                check_fp(h, n, k, False, gps.FP_PAIR, 7, True)
                if n <= (1 << 22) + 1:
                    check_struct(h, n, k, k % 2 == 0, False)
        assert h.device_error() == 0


def test_segment_heads_with_more_offsets_in_a_tile_than_a_workgroup_reads_at_once():
    n = 3 * TILE + 17  # units and empty segments: 8 offsets per element of the second tile
    starts = np.r_[0, np.repeat(np.arange(TILE, 2 * TILE), 8), 2 * TILE + 1, n].astype(np.int64)
    x = torch.from_numpy(np.random.default_rng(3).integers(-8, 9, n).astype(np.float32)).cuda()
    c = torch.cumsum(x.double(), 0).cpu().numpy()
    head = np.zeros(n, dtype=np.int64)
    head[starts[:-1]] = starts[:-1]
    head = np.maximum.accumulate(head)
    want = c - np.where(head > 0, c[head - 1], 0.0)
    out = torch.empty_like(x)
    with gps.ScanHandle(gps.ALGO_CSDL, n, block_threads=256, vec_per_thread=4, schedule=gps.SCHEDULE_TILE) as h:
        h.segmented_fp(x, out, torch.from_numpy(starts).cuda(), starts.size - 1, n, bf16=False, compensated=True)
        torch.cuda.synchronize()
        assert np.array_equal(out.cpu().numpy().astype(np.float64), want)
        assert h.device_error() == 0


@pytest.mark.parametrize("n", [1 << 16, 1 << 20, 1 << 22])
def test_replays_of_a_captured_scan(n):
    x = oracle.gen_u32(4, n, 32)
    d_in, out = to_dev(x), torch.empty(n, dtype=torch.int32, device="cuda")
    want = torch.from_numpy(oracle.scan_u32(x, True).view(np.int32)).cuda()
    with gps.ScanHandle(gps.ALGO_CSDL, n) as h:
        g = torch.cuda.CUDAGraph()
        h.scan(d_in, out, n, True)
        torch.cuda.synchronize()
        with torch.cuda.graph(g):
            h.scan(d_in, out, n, True)
        for _ in range(5):
            out.fill_(-7)
            g.replay()
            assert torch.equal(out, want)
            out.fill_(-7)
            h.scan(d_in, out, n, True)
            assert torch.equal(out, want)
        assert h.device_error() == 0


@pytest.mark.parametrize("n", [0, 5, 1 << 16, (1 << 20) + 1, (1 << 23) + 5])
@pytest.mark.parametrize("own_stream", [False, True], ids=["null_stream", "own_stream"])
def test_segmented_graph_replays(n, own_stream):
    segments = 37
    cuts = np.linspace(0, n, segments + 1).astype(np.uint64)
    x = oracle.gen_u32(n + 1, max(n, 1), 32)[:n]
    want = torch.from_numpy(oracle.segmented_scan_u32(x, cuts, False).view(np.int32)).cuda() if n else None
    d_in, out = to_dev(oracle.gen_u32(n + 1, max(n, 1), 32)), torch.empty(max(n, 1), dtype=torch.int32, device="cuda")
    off = torch.from_numpy(cuts.view(np.int64)).cuda()
    stream = torch.cuda.Stream() if own_stream else torch.cuda.current_stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream), gps.ScanHandle(gps.ALGO_CSDL, max(n, 1)) as h:
        with h.segmented_graph(d_in, out, off, segments, n, False) as g:
            for _ in range(4):
                out.fill_(-7)
                g.launch(stream)
                assert n == 0 or torch.equal(out[:n], want)
                out.fill_(-7)
                h.segmented(d_in, out, off, segments, n, False)
                assert n == 0 or torch.equal(out[:n], want)
        assert h.device_error() == 0
