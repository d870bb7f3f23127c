"""The native packing of a call (g950_py.cpp) against the ctypes path it
stands before: the same kernel and bits for every scalar type and tensor form
either takes, and the same errors for what neither does."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from compiler_amd import operators as ops  # noqa: E402
from compiler_amd import runtime as rt  # noqa: E402

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.fixture
def ctypes_path(monkeypatch):
    """Calls made inside run on the ctypes path."""
    def use():
        monkeypatch.setattr(rt.module(), "_pack_launch", lambda *a: None)
    return use


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16, torch.float16])
def test_same_bits_on_both_paths(dt, ctypes_path):
    x = torch.randn(9, 70, device=DEV).to(dt)[1:, 3:67]      # strided view into a larger storage
    w = torch.nn.Parameter(torch.rand(64, device=DEV).to(dt))
    calls = [lambda: ops.rmsnorm(x, w, 1e-6, sync=True), lambda: (ops.softmax(x, sync=True),),
             lambda: (ops.matmul(x, x.t(), sync=True),),
             lambda: ops.attention(*[x.reshape(1, 1, 8, 64)] * 3, sync=True)]
    native = [(c(), rt.module().last_kernel) for c in calls]
    ctypes_path()
    for c, (want, kernel) in zip(calls, native):
        got = c()
        assert rt.module().last_kernel == kernel
        assert all(torch.equal(a, b) for a, b in zip(got, want))


@pytest.mark.parametrize("n", [64, np.int32(64), np.int64(64), np.uint8(64), rt.scalar(64), rt.scalar(64, "int16")])
def test_scalar_types(n):
    x = torch.randn(5, 64, device=DEV)
    y = torch.empty_like(x)
    ops.softmax_kernel(x, y, n, sync=True)
    assert torch.equal(y, ops.softmax(x, sync=True))


@pytest.mark.parametrize("native", [True, False])
def test_errors(native, ctypes_path):
    x = torch.randn(5, 64, device=DEV)
    if not native:
        ctypes_path()
    with pytest.raises(rt.G950Error, match="n_cols"):
        ops.softmax_kernel(x, torch.empty_like(x), 63)
    with pytest.raises(rt.G950Error, match="device"):
        ops.softmax_kernel(x.cpu(), torch.empty_like(x), 64)
    with pytest.raises(rt.G950Error, match="unsupported tensor dtype"):
        ops.softmax_kernel(x.to(torch.complex64), torch.empty_like(x), 64)
    with pytest.raises(rt.G950Error, match="unsupported scalar"):
        ops.softmax_kernel(x, torch.empty_like(x), "64")
    with pytest.raises(OverflowError):
        ops.softmax_kernel(x, torch.empty_like(x), 1 << 70)
    with pytest.raises(rt.G950Error, match="outside|stride|reach|contiguous"):
        ops.softmax_kernel(x.t(), torch.empty_like(x).t(), 5)


def test_streams_and_no_alloc():
    x = torch.randn(5, 64, device=DEV)
    want = ops.softmax(x, sync=True)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        a = ops.softmax(x, sync=True)
        with rt.no_alloc():
            b = ops.softmax(x, sync=True)
    c = ops.softmax(x, stream=s, sync=True)
    d = ops.softmax(x, stream=s.cuda_stream, sync=True)
    assert all(torch.equal(want, t) for t in (a, b, c, d))
