"""Inputs above 64 MiB, which tiles load past the Infinity Cache, from and to
buffers that start at any element: FP32 and uint32 at 4-byte addresses, BF16 at
2-byte ones, with a partial last tile and guards on both sides of the output.
Floats are -1, 0 or 1, so every sum is exact in FP32."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

import gpuprefixsums_amd as gps  # noqa: E402
from tests.gpu_util import to_dev  # noqa: E402

LINE = 64 << 20  # bytes; larger inputs stream
GUARD = 16
SHIFTS = [(1, 0), (2, 1), (3, 3)]  # input, output
SHAPES = {
    "default": dict(),
    "tile_256x4": dict(block_threads=256, vec_per_thread=4, schedule=gps.SCHEDULE_TILE),
    "tile_1024x8": dict(block_threads=1024, vec_per_thread=8, schedule=gps.SCHEDULE_TILE),
    "persistent_512x8": dict(block_threads=512, vec_per_thread=8, schedule=gps.SCHEDULE_PERSISTENT),
    "persistent_1024x4": dict(block_threads=1024, vec_per_thread=4, schedule=gps.SCHEDULE_PERSISTENT),
}
CONTROL = dict(block_threads=512, vec_per_thread=4, schedule=gps.SCHEDULE_CONTROL)


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if not torch.cuda.is_available():
        pytest.fail("GPU tests need a ROCm device")


def sizes(width):
    n = LINE // width
    return [n + 1, n + 2 * 32768 - 3]


def check(launch, x, want, shift_in, shift_out):
    """launch(in, out) with both buffers at their shifts; want on the device."""
    src = torch.empty(x.numel() + shift_in, dtype=x.dtype, device="cuda")[shift_in:]
    src.copy_(x)
    lead = GUARD + shift_out
    buf = torch.full((lead + want.numel() + GUARD,), -7, dtype=want.dtype, device="cuda")
    out = buf[lead:lead + want.numel()]
    launch(src, out)
    torch.cuda.synchronize()
    bad = torch.nonzero(out != want)
    assert bad.numel() == 0, (shift_in, shift_out, bad.numel(), int(bad[0]))
    assert bool((buf[:lead] == -7).all()) and bool((buf[lead + want.numel():] == -7).all()), "wrote outside"


U32_HANDLES = {f"csdl_{k}": dict(algo=gps.ALGO_CSDL, **v) for k, v in {**SHAPES, "control": CONTROL}.items()}
U32_HANDLES |= {f"csdldf_{k}": dict(algo=gps.ALGO_CSDLDF, stall_period=s, **v)
                for k, s, v in [("default", 0, {}), ("tile_256x4", 7, SHAPES["tile_256x4"]),
                                ("persistent_1024x4", 7, SHAPES["persistent_1024x4"])]}
U32_HANDLES["rts"] = dict(algo=gps.ALGO_RTS)


@pytest.mark.parametrize("name", U32_HANDLES)
def test_u32(name):
    for k, n in enumerate(sizes(4)):
        host = oracle.gen_u32(300 + k, n, 32)
        x = to_dev(host)
        with gps.ScanHandle(max_n=n, **U32_HANDLES[name]) as h:
            for inclusive in (False, True):
                want = to_dev(oracle.scan_u32(host, inclusive))
                for shifts in SHIFTS:
                    check(lambda i, o: h.scan(i, o, n, inclusive), x, want, *shifts)
            assert h.device_error() == 0


def signs(n, bf16, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randint(-1, 2, (n,), dtype=torch.int32, device="cuda", generator=g)
    return x, x.to(torch.bfloat16 if bf16 else torch.float32)


@pytest.mark.parametrize("name", SHAPES)
@pytest.mark.parametrize("comp", [gps.FP_PAIR, gps.FP_PLAIN], ids=["pair", "plain"])
@pytest.mark.parametrize("bf16", [False, True], ids=["f32", "bf16"])
def test_fp(name, comp, bf16):
    for k, n in enumerate(sizes(2 if bf16 else 4)):
        ints, x = signs(n, bf16, 7 + k)
        want = torch.cumsum(ints, 0).float()
        with gps.ScanHandle(gps.ALGO_CSDL, n, **SHAPES[name]) as h:
            for shifts in SHIFTS:
                check(lambda i, o: (h.inclusive_bf16_f32 if bf16 else h.inclusive_f32)(i, o, n, comp), x, want, *shifts)
            assert h.device_error() == 0


def cuts_of(n):
    """Empty segments, ends on and beside tile edges, and long segments."""
    rng = np.random.default_rng(n)
    cuts = [0, 0, 1, 4096, 32768, 32769, 32769, n - 1, n, *(int(c) for c in rng.integers(0, n, 500))]
    return np.array(sorted(cuts), dtype=np.uint64)


@pytest.mark.parametrize("name", SHAPES)
@pytest.mark.parametrize("inclusive", [False, True], ids=["excl", "incl"])
def test_segmented_u32(name, inclusive):
    for k, n in enumerate(sizes(4)):
        host, off = oracle.gen_u32(400 + k, n, 32), cuts_of(n)
        x, d_off, want = to_dev(host), to_dev(off), to_dev(oracle.segmented_scan_u32(host, off, inclusive))
        with gps.ScanHandle(gps.ALGO_CSDL, n, **SHAPES[name]) as h:
            for shifts in SHIFTS:
                check(lambda i, o: h.segmented(i, o, d_off, off.size - 1, n, inclusive), x, want, *shifts)
            assert h.device_error() == 0


@pytest.mark.parametrize("name", SHAPES)
@pytest.mark.parametrize("comp", [gps.FP_PAIR, gps.FP_PLAIN], ids=["pair", "plain"])
@pytest.mark.parametrize("bf16", [False, True], ids=["f32", "bf16"])
def test_segmented_fp(name, comp, bf16):
    n = sizes(2 if bf16 else 4)[1]
    ints, x = signs(n, bf16, 17)
    off = to_dev(cuts_of(n))
    sums = torch.cat([torch.zeros(1, dtype=torch.int64, device="cuda"), torch.cumsum(ints, 0)])
    lengths = off[1:] - off[:-1]
    want = (sums[1:] - torch.repeat_interleave(sums[off[:-1]], lengths)).float()
    with gps.ScanHandle(gps.ALGO_CSDL, n, **SHAPES[name]) as h:
        for shifts in SHIFTS:
            check(lambda i, o: h.segmented_fp(i, o, off, off.numel() - 1, n, bf16, comp), x, want, *shifts)
        assert h.device_error() == 0
