"""GPU parity of the few-row GEMM kernels (M <= 64, K-contiguous operands) in
every mode: bf16, fp16, fp32, int8 and int8 weights under 16-bit A.  Rows at
the edges of the row classes (4, 8, 16, 32, 64), column counts that reach
every number of column groups per workgroup, K below, at and past a round of
the waves' 128-byte units and with tails; guard rows and columns untouched;
against the CPU oracle (bf16 2e-2, fp16 1e-2, fp32 1e-5 with the sqrt(K)
absolute term, int8 exact)."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from compiler_amd import operators as ops  # noqa: E402
from compiler_amd import runtime as rt  # noqa: E402
from oracle import reference as ref  # noqa: E402

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
TD = {"float32": torch.float32, "bfloat16": torch.bfloat16, "float16": torch.float16}

# rows, columns, K in 16-byte chunks of an operand row
SHAPES = [(1, 1, 64), (4, 33, 65), (5, 47, 127), (8, 4097, 64), (9, 12300, 72), (16, 100, 300), (16, 6200, 70),
          (17, 70, 64), (32, 4100, 81), (31, 8200, 64), (33, 130, 90), (64, 4098, 64), (64, 8208, 73)]

# the widest column groups with one DMA instruction of A (8 rows; int8 weights: 4)
SHAPES_FEW = [(7, 12300, 72)]
SHAPES_W8 = [(3, 20, 1), (16, 14400, 9), (32, 12300, 20), (4, 6200, 70), (2, 10000, 33), (3, 14400, 9), (1, 8192, 130)]


@pytest.mark.parametrize("dt", ["bfloat16", "float16", "float32", "int8"])
@pytest.mark.parametrize("m,n,chunks", SHAPES + SHAPES_FEW)
def test_few_rows(m, n, chunks, dt):
    rng = np.random.default_rng(m + 3 * n + 7 * chunks)
    k = chunks * {"float32": 4, "int8": 16}.get(dt, 8)
    short = {"bfloat16": "bf16", "float16": "f16", "float32": "f32", "int8": "i8"}[dt]
    rows = 16 if m <= 16 else 32 if m <= 32 else 64
    if dt == "int8":
        a = rng.integers(-127, 127, (m, k), dtype=np.int8)
        bt = rng.integers(-127, 127, (n, k), dtype=np.int8)
        full = torch.full((m + 2, n + 5), -5, dtype=torch.int32, device=DEV)
        y = torch.as_strided(full, (m, n), (n + 5, 1), (n + 5) // 4 * 4)
        ops.matmul_i8_kernel(torch.from_numpy(a).to(DEV), torch.from_numpy(bt).to(DEV).t(), y, m, n, k, sync=True)
        assert rt.module().last_kernel == f"g950_gemm_skinny{rows}_i8"
        assert np.array_equal(y.cpu().numpy(), ref.matmul_i8(a, bt.T))
        y.fill_(-5)
        assert bool((full == -5).all())
        return
    a = torch.from_numpy(rng.standard_normal((m, k)).astype(np.float32) / np.float32(np.sqrt(k))).to(DEV).to(TD[dt])
    bt = torch.from_numpy(rng.standard_normal((n, k)).astype(np.float32)).to(DEV).to(TD[dt])
    full = torch.full((m + 2, n + 5), 7.0, dtype=TD[dt], device=DEV)
    y = torch.as_strided(full, (m, n), (n + 5, 1), (n + 5) // 8 * 8)
    ops.matmul_kernel(a, bt.t(), y, m, n, k, sync=True)
    assert rt.module().last_kernel == f"g950_gemm_skinny{rows}_{short}"
    bar = {"bfloat16": (2e-2, 2e-2), "float16": (1e-2, 1e-2), "float32": (1e-5, 1e-5)}[dt]
    expect = ref.matmul(a.float().cpu().numpy(), bt.float().cpu().numpy().T)
    ok, err = ref.isclose_verdict(y.float().cpu().numpy(), expect, *bar)
    assert ok, err
    y.fill_(7.0)
    assert bool((full == 7.0).all())


@pytest.mark.parametrize("dt", ["bfloat16", "float16"])
@pytest.mark.parametrize("m,n,chunks", SHAPES + SHAPES_W8)
def test_few_rows_int8_weights(m, n, chunks, dt):
    rng = np.random.default_rng(m + n + chunks)
    k = 16 * chunks
    a = torch.from_numpy(rng.standard_normal((m, k)).astype(np.float32) * 0.5).to(DEV).to(TD[dt])
    bt = rng.integers(-127, 128, (n, k)).astype(np.int8)
    s = torch.from_numpy((rng.random(n) / 64).astype(np.float32)).to(DEV).to(TD[dt])
    full = torch.full((m + 2, n + 5), 7.0, dtype=TD[dt], device=DEV)
    y = torch.as_strided(full, (m, n), (n + 5, 1), (n + 5) // 8 * 8)
    ops.dequant_matmul_kernel(a, torch.from_numpy(bt).to(DEV).t(), s, y, m, n, k, sync=True)
    assert rt.module().last_kernel.startswith("g950_gemm_w8a16_skinny")
    expect = ref.matmul(a.float().cpu().numpy(), ref.dequantize(bt.T, s.float().cpu().numpy()))
    ok, err = ref.isclose_verdict(y.float().cpu().numpy(), expect, 2e-2, 2e-2)
    assert ok, err
    y.fill_(7.0)
    assert bool((full == 7.0).all())


def test_few_rows_keep_nan_to_their_own_row():
    """A NaN in one row of A reaches that output row alone, also below the
    rows that a call with fewer than 9 rows brings in."""
    a = torch.randn(5, 1024, device=DEV).to(torch.bfloat16)
    a[2, 700] = float("nan")
    bt = torch.randn(40, 1024, device=DEV).to(torch.bfloat16)
    y = ops.matmul(a, bt.t(), sync=True)
    assert bool(y[2].isnan().all()) and not bool(y[[0, 1, 3, 4]].isnan().any())


@pytest.mark.parametrize("dt", ["bfloat16", "float16"])
@pytest.mark.parametrize("m,n,chunks", [(1, 16385, 1), (4, 16415, 9), (3, 20001, 69), (2, 16390, 64), (1, 16400, 127),
                                        (4, 33000, 17)])
def test_few_rows_int8_weights_past_one_round(m, n, chunks, dt):
    """Up to four rows of A against more columns than one round of the widest
    form holds: the two-workgroups-per-CU kernel, whose workgroups start at
    different units of K and wrap round (fewer units than waves, tails)."""
    rng = np.random.default_rng(m + n + chunks)
    k = 16 * chunks
    a = torch.from_numpy(rng.standard_normal((m, k)).astype(np.float32) * 0.5).to(DEV).to(TD[dt])
    bt = rng.integers(-127, 128, (n, k)).astype(np.int8)
    s = torch.from_numpy((rng.random(n) / 64).astype(np.float32)).to(DEV).to(TD[dt])
    full = torch.full((m + 2, n + 5), 7.0, dtype=TD[dt], device=DEV)
    y = torch.as_strided(full, (m, n), (n + 5, 1), (n + 5) // 8 * 8)
    ops.dequant_matmul_kernel(a, torch.from_numpy(bt).to(DEV).t(), s, y, m, n, k, sync=True)
    assert rt.module().last_kernel == f"g950_gemm_w8a16_few_{'bf16' if dt == 'bfloat16' else 'f16'}"
    expect = ref.matmul(a.float().cpu().numpy(), ref.dequantize(bt.T, s.float().cpu().numpy()))
    ok, err = ref.isclose_verdict(y.float().cpu().numpy(), expect, 2e-2, 2e-2)
    assert ok, err
    y.fill_(7.0)
    assert bool((full == 7.0).all())
