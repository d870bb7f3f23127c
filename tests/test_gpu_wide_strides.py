"""GPU results of GEMM calls whose rows lie too far apart for 32-bit byte
offsets (the last token of long sequences: hidden[:, -1, :]), against the CPU
oracle (bf16 2e-2 on y = a . (b * scale))."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from compiler_amd import operators as ops  # noqa: E402
from compiler_amd import runtime as rt  # noqa: E402
from oracle import reference as ref  # noqa: E402

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def strided_rows(rng, m, k, stride, dtype=torch.bfloat16):
    """m rows of k elements, `stride` elements apart in one allocation."""
    a = torch.empty((m - 1) * stride + k, dtype=dtype, device=DEV).as_strided((m, k), (stride, 1))
    a.copy_(torch.from_numpy(rng.standard_normal((m, k)).astype(np.float32) * 0.5))
    return a


# one row (whatever its stride), and rows past 4 GiB in each kernel
@pytest.mark.parametrize("row_major", [False, True])
@pytest.mark.parametrize("m,stride", [(1, 1 << 31), (16, 5 << 25), (31, 5 << 24), (64, 1 << 26), (100, 3 << 23),
                                      (300, 3 << 23)])
def test_w8a16_far_rows_of_a(m, stride, row_major):
    rng = np.random.default_rng(m)
    n, k = 272, 320
    a = strided_rows(rng, m, k, stride)
    w = rng.integers(-127, 128, (k, n)).astype(np.int8)
    # row-major rows padded by 16 bytes
    b = (torch.from_numpy(np.pad(w, ((0, 0), (0, 16)))).to(DEV)[:, :n] if row_major
         else torch.from_numpy(np.ascontiguousarray(w.T)).to(DEV).t())
    s = torch.from_numpy((rng.random(n) / 64).astype(np.float32)).to(DEV).to(torch.bfloat16)
    y = torch.full((m + 2, n), 7.0, dtype=torch.bfloat16, device=DEV)
    ops.dequant_matmul_kernel(a, b, s, y[:m], m, n, k, sync=True)
    assert ("skinny" if m == 1 else "_far") in rt.module().last_kernel
    expect = ref.matmul(a.float().cpu().numpy(), ref.dequantize(w, s.float().cpu().numpy()))
    ok, err = ref.isclose_verdict(y[:m].float().cpu().numpy(), expect, 2e-2, 2e-2)
    assert ok, err
    assert bool((y[m:] == 7.0).all())


@pytest.mark.parametrize("m", [3, 20, 33, 100])
def test_w8a16_far_rows_of_weights(m):
    """80 rows of Bt whose 64th lies past 4 GiB, K tail of a slab."""
    rng = np.random.default_rng(m)
    n, k, stride = 80, 400, 70_000_000
    bt = torch.empty((n - 1) * stride + k, dtype=torch.int8, device=DEV).as_strided((n, k), (stride, 1))
    w = rng.integers(-127, 128, (n, k)).astype(np.int8)
    bt.copy_(torch.from_numpy(w))
    a = torch.from_numpy(rng.standard_normal((m, k)).astype(np.float32) * 0.5).to(DEV).to(torch.float16)
    s = torch.from_numpy((rng.random(n) / 64).astype(np.float32)).to(DEV).to(torch.float16)
    y = ops.dequant_matmul(a, bt.t(), s, sync=True)
    assert "_far" in rt.module().last_kernel
    expect = ref.matmul(a.float().cpu().numpy(), ref.dequantize(w.T, s.float().cpu().numpy()))
    ok, err = ref.isclose_verdict(y.float().cpu().numpy(), expect, 2e-2, 2e-2)
    assert ok, err
