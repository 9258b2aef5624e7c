"""gpuprefixsums_amd.torch_ops without a usable libgps_torch.so: the operators are
there all the same, from their Python implementations."""
import subprocess
import sys
import textwrap

import pytest

torch = pytest.importorskip("torch")

# The library is looked for beside _lib.LIB_PATH, so libgps.so itself is loaded first.
HEAD = """
import pathlib, sys, warnings
import torch
from gpuprefixsums_amd import _lib
_lib.load()
_lib.LIB_PATH = pathlib.Path(sys.argv[1]) / "libgps.so"
with warnings.catch_warnings(record=True) as w:
    warnings.simplefilter("always")
    import gpuprefixsums_amd.torch_ops as ops
assert ops._kernels is None and any("through Python" in str(x.message) for x in w)
"""


def run(tmp_path, present, code):
    if present:
        (tmp_path / "libgps_torch.so").write_text("not a library")
    p = subprocess.run([sys.executable, "-c", HEAD + textwrap.dedent(code), str(tmp_path)], capture_output=True, text=True)
    assert p.returncode == 0, p.stderr


@pytest.mark.parametrize("present", [False, True], ids=["absent", "unloadable"])
def test_import(tmp_path, present):
    run(tmp_path, present, """
        y = torch.ops.gps.cumsum(torch.empty(9, dtype=torch.bfloat16, device="meta"))
        assert y.dtype == torch.float32 and y.shape == (9,)
        try:
            torch.ops.gps.cumsum(torch.zeros(4))
        except RuntimeError as e:
            assert "ROCm device" in str(e)
        else:
            raise AssertionError("a CPU tensor was taken")
    """)


@pytest.mark.gpu
def test_calls(tmp_path):
    if not torch.cuda.is_available():
        pytest.fail("GPU tests need a ROCm device")
    run(tmp_path, False, """
        x = torch.arange(-500, 1500, device="cuda", dtype=torch.int32)
        for _ in range(2):
            assert torch.equal(torch.ops.gps.cumsum(x).long(), x.long().cumsum(0))
            y = torch.ops.gps.segmented_cumsum(x.float(), torch.tensor([0, 700, 2000], device="cuda"))
            assert torch.equal(y[700:].double(), x[700:].double().cumsum(0))
    """)
