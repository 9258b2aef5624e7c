"""torch.ops.gps.*: the device kernels (csrc/torch_ops.cpp) against the Python
implementations they stand in for, over every form of input, and the calls
that must still reach those: gradients, errors, other streams and threads."""
import threading

import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

import gpuprefixsums_amd.torch_ops as ops  # noqa: E402

DTYPES = [torch.int32, torch.uint32, torch.float32, torch.bfloat16]
FORMS = {
    "whole": lambda x: x,
    "offset": lambda x: x[3:],
    "strided": lambda x: x[::2],
    "one": lambda x: x[:1],
    "one_of_a_stride": lambda x: x[::100][:1],
    "expanded": lambda x: x[:1].expand(9),
    "empty": lambda x: x[:0],
}


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if not torch.cuda.is_available():
        pytest.fail("GPU tests need a ROCm device")


def values(dtype, n=5000):
    g = torch.Generator().manual_seed(n)
    x = torch.randint(-9, 10, (n,), generator=g, dtype=torch.int32)
    return (x.view(dtype) if dtype in (torch.int32, torch.uint32) else x.to(dtype)).cuda()


def cuts(n):
    return torch.tensor([0, n // 3, n // 3, n], device="cuda")


def same(a, b):
    assert (a.dtype, a.shape, a.stride(), a.device) == (b.dtype, b.shape, b.stride(), b.device)
    view = torch.int32 if a.dtype == torch.uint32 else a.dtype
    assert torch.equal(a.view(view), b.view(view))


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("form", FORMS)
def test_same_as_the_python_implementation(dtype, form):
    x = FORMS[form](values(dtype))
    offsets = cuts(x.numel())
    spread = torch.stack([offsets, offsets], 1)[:, 0]  # strided offsets
    for _ in range(2):  # the first call may make the stream's handle
        for inclusive in (True, False) if dtype in (torch.int32, torch.uint32) else (True,):
            for compensated in (True, False):
                same(torch.ops.gps.cumsum(x, inclusive, compensated), ops.cumsum._init_fn(x, inclusive, compensated))
                want = ops.segmented_cumsum._init_fn(x, offsets, inclusive, compensated)
                same(torch.ops.gps.segmented_cumsum(x, offsets, inclusive, compensated), want)
                same(torch.ops.gps.segmented_cumsum(x, spread, inclusive, compensated), want)


def test_what_was_refused_stays_refused():
    x, offsets = values(torch.float32), cuts(5000)
    torch.ops.gps.cumsum(x)  # a handle is in place
    for call, text in [
        (lambda: torch.ops.gps.cumsum(x.view(50, 100)), "1-D"),
        (lambda: torch.ops.gps.cumsum(x[0]), "1-D"),
        (lambda: torch.ops.gps.cumsum(x, False), "inclusive"),
        (lambda: torch.ops.gps.segmented_cumsum(x, offsets, False), "inclusive"),
        (lambda: torch.ops.gps.cumsum(x.double()), "unsupported dtype"),
        (lambda: torch.ops.gps.segmented_cumsum(x, offsets.int()), "int64"),
        (lambda: torch.ops.gps.segmented_cumsum(x, offsets.cpu()), "int64"),
        (lambda: torch.ops.gps.segmented_cumsum(x, offsets[None]), "int64"),
        (lambda: torch.ops.gps.segmented_cumsum(x, offsets[:0]), "at least one"),
        (lambda: torch.ops.gps.cumsum(x.cpu()), "ROCm device"),
    ]:
        with pytest.raises(RuntimeError, match=text):
            call()


def test_gradients_go_to_the_autograd_wrapper():
    x = values(torch.float32).requires_grad_()
    offsets = cuts(5000)
    for call in (lambda: torch.ops.gps.cumsum(x), lambda: torch.ops.gps.segmented_cumsum(x, offsets)):
        y = call()
        assert y.requires_grad
        with pytest.raises(RuntimeError, match="no autograd formula"):
            y.sum().backward()
        with torch.no_grad():
            same(call(), y.detach())
        with torch.inference_mode():
            assert torch.equal(call(), y.detach())


def test_tracing_modes_and_vmap_see_the_operator():
    from torch.utils._python_dispatch import TorchDispatchMode
    x = values(torch.float32)
    seen = []

    class Record(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen.append(str(func))
            return func(*args, **(kwargs or {}))

    with Record():
        torch.ops.gps.cumsum(x)
    assert seen[0] == "gps.cumsum.default"
    rows = x.view(5, 1000)
    assert torch.equal(torch.vmap(torch.ops.gps.cumsum)(rows), torch.stack([torch.ops.gps.cumsum(r) for r in rows]))
    traced = torch.compile(lambda v: torch.ops.gps.cumsum(v) + 1, backend="aot_eager", fullgraph=True)
    assert torch.equal(traced(x), torch.ops.gps.cumsum(x) + 1)


def test_threads_on_streams_of_their_own():
    xs = [values(torch.int32, 1000 + 7 * i) for i in range(4)]
    want = [ops.cumsum._init_fn(x) for x in xs]
    torch.cuda.synchronize()
    got = [None] * len(xs)

    def work(i):
        with torch.cuda.stream(torch.cuda.Stream()):
            got[i] = [torch.ops.gps.cumsum(xs[i]) for _ in range(40)]
            torch.cuda.current_stream().synchronize()

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(xs))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for ys, w in zip(got, want):
        assert all(torch.equal(y, w) for y in ys)


def test_a_grown_handle_replaces_the_smaller_one():
    with torch.cuda.stream(torch.cuda.Stream()):
        small = values(torch.int32, 1000)
        large = values(torch.int32, (1 << 20) + 3)  # above the first handle's size
        for x in (small, large, small, large):
            same(torch.ops.gps.cumsum(x), torch.cumsum(x, 0, dtype=torch.int32))
        torch.cuda.current_stream().synchronize()
