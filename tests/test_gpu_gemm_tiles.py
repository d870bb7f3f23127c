"""GPU parity of the smaller workgroup tiles of the whole-slab MFMA GEMM
(64x64, 64x128, 128x128): every element of shapes at the tiles' edges, one to
many K slabs (fewer and more than the ring's stages), guard rows and columns
untouched, against the CPU oracle (bf16 2e-2, fp16 1e-2, fp32 1e-5 with the
sqrt(K) absolute term for sums in another order, int8 exact)."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from compiler_amd import operators as ops  # noqa: E402
from compiler_amd import runtime as rt  # noqa: E402
from oracle import reference as ref  # noqa: E402

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
TD = {"float32": torch.float32, "bfloat16": torch.bfloat16, "float16": torch.float16}

# 64 x 64 tiles, then 264 or 272 of them (64 x 128), then 160 128 x 128 tiles,
# and past those; (63, 130, 576) is the few-row kernels'
SHAPES = [(1, 3, 64), (64, 64, 128), (65, 129, 448), (63, 130, 576), (100, 1000, 2048),
          (500, 2100, 128), (513, 1900, 704), (1000, 2500, 128), (1023, 2401, 640), (70, 130, 576), (2049, 4097, 128)]


def check_form(m, n):
    """The tile that ran is the one the shape is listed for."""
    want = ("64x16" if m == 63 else "64x64" if m * n <= 300_000 else
            "64x128" if m < 600 else "128x128" if m < 2000 else "256x256")
    assert rt.load_library().g950_last_form().decode() == want


@pytest.mark.parametrize("dt", ["bfloat16", "float16", "float32", "int8"])
@pytest.mark.parametrize("m,n,k", SHAPES)
def test_gemm_tiles(m, n, k, dt):
    rng = np.random.default_rng(m + 3 * n + 7 * k)
    if dt == "int8":
        k *= 2  # whole 128-byte slabs
        a = rng.integers(-127, 128, (m, k), dtype=np.int8)
        bt = rng.integers(-127, 128, (n, k), dtype=np.int8)
        full = torch.full((m + 2, n + 5), -5, dtype=torch.int32, device=DEV)
        y = torch.as_strided(full, (m, n), (n + 5, 1), (n + 5) // 4 * 4)  # 16-byte aligned start
        ops.matmul_i8_kernel(torch.from_numpy(a).to(DEV), torch.from_numpy(bt).to(DEV).t(), y, m, n, k, sync=True)
        check_form(m, n)
        assert np.array_equal(y.cpu().numpy(), ref.matmul_i8(a, bt.T))
        y.fill_(-5)
        assert bool((full == -5).all())
        return
    a = torch.from_numpy(rng.standard_normal((m, k)).astype(np.float32) / np.float32(np.sqrt(k))).to(DEV).to(TD[dt])
    bt = torch.from_numpy(rng.standard_normal((n, k)).astype(np.float32)).to(DEV).to(TD[dt])
    full = torch.full((m + 2, n + 5), 7.0, dtype=TD[dt], device=DEV)
    y = torch.as_strided(full, (m, n), (n + 5, 1), (n + 5) // 8 * 8)
    ops.matmul_kernel(a, bt.t(), y, m, n, k, sync=True)
    check_form(m, n)
    bar = {"bfloat16": (2e-2, 2e-2), "float16": (1e-2, 1e-2), "float32": (1e-5, 1e-5)}[dt]
    expect = ref.matmul(a.float().cpu().numpy(), bt.float().cpu().numpy().T)
    ok, err = ref.isclose_verdict(y.float().cpu().numpy(), expect, *bar)
    assert ok, err
    y.fill_(7.0)
    assert bool((full == 7.0).all())


@pytest.mark.parametrize("dt", ["bfloat16", "float16"])
@pytest.mark.parametrize("m,n,k", [(65, 3, 128), (65, 129, 16), (100, 1000, 2064), (500, 2100, 112), (513, 1900, 704),
                                   (1000, 2500, 144), (1023, 2401, 1280)])
def test_w8a16_tiles(m, n, k, dt):
    """int8 weights on the same tiles, slabs of 128 k with tails of every
    multiple of 16, against float64 a . (b * scale) on the rounded inputs."""
    rng = np.random.default_rng(m + 3 * n + 7 * k)
    a = torch.from_numpy(rng.standard_normal((m, k)).astype(np.float32) * 0.5).to(DEV).to(TD[dt])
    bt = rng.integers(-127, 128, (n, k)).astype(np.int8)
    s = torch.from_numpy((rng.random(n) / 64).astype(np.float32)).to(DEV).to(TD[dt])
    full = torch.full((m + 2, n + 5), 7.0, dtype=TD[dt], device=DEV)
    y = torch.as_strided(full, (m, n), (n + 5, 1), (n + 5) // 8 * 8)
    ops.dequant_matmul_kernel(a, torch.from_numpy(bt).to(DEV).t(), s, y, m, n, k, sync=True)
    check_form(m, n)
    expect = ref.matmul(a.float().cpu().numpy(), ref.dequantize(bt.T, s.float().cpu().numpy()))
    ok, err = ref.isclose_verdict(y.float().cpu().numpy(), expect, 2e-2, 2e-2)
    assert ok, err
    y.fill_(7.0)
    assert bool((full == 7.0).all())


@pytest.mark.parametrize("dt", ["bfloat16", "float16"])
@pytest.mark.parametrize("m,n,k", [(256, 256, 64), (257, 264, 576), (300, 1000, 448), (500, 2104, 128), (513, 1912, 704),
                                   (1000, 2504, 128), (1023, 2408, 640)])
def test_row_major_b_tiles(m, n, k, dt):
    """Row-major B on the smaller tiles: right-edge windows, every fragment of
    the transposing reads, and the column scale of row-major int8 weights."""
    rng = np.random.default_rng(m + 3 * n + 7 * k)
    a = torch.from_numpy(rng.standard_normal((m, k)).astype(np.float32) / np.float32(np.sqrt(k))).to(DEV).to(TD[dt])
    b = torch.from_numpy(rng.standard_normal((k, n + 8)).astype(np.float32)).to(DEV).to(TD[dt])[:, :n]
    full = torch.full((m + 2, n + 5), 7.0, dtype=TD[dt], device=DEV)
    y = torch.as_strided(full, (m, n), (n + 5, 1), (n + 5) // 8 * 8)
    ops.matmul_kernel(a, b, y, m, n, k, sync=True)
    check_form(m, n)
    bar = {"bfloat16": (2e-2, 2e-2), "float16": (1e-2, 1e-2)}[dt]
    ok, err = ref.isclose_verdict(y.float().cpu().numpy(), ref.matmul(a.float().cpu().numpy(), b.float().cpu().numpy()),
                                  *bar)
    assert ok, err
    y.fill_(7.0)
    assert bool((full == 7.0).all())
    n -= n % 16
    w = rng.integers(-127, 128, (k, n)).astype(np.int8)
    s = torch.from_numpy((rng.random(n) / 64).astype(np.float32)).to(DEV).to(TD[dt])
    got = ops.dequant_matmul(a, torch.from_numpy(w).to(DEV), s, sync=True)
    check_form(m, n)
    expect = ref.matmul(a.float().cpu().numpy(), ref.dequantize(w, s.float().cpu().numpy()))
    ok, err = ref.isclose_verdict(got.float().cpu().numpy(), expect, 2e-2, 2e-2)
    assert ok, err
