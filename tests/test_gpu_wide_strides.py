"""GPU results of GEMM calls whose rows lie too far apart for 32-bit byte
offsets (the last token of long sequences: hidden[:, -1, :]) or at negative
strides (through the C ABI: torch has none), against the CPU oracle (bf16 2e-2
on y = a . (b * scale))."""
import ctypes

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


def launch(op, tensors, strides, scalars):
    """g950_launch on views of `tensors` whose dimensions d with strides[i][d]
    < 0 run backwards (from the last element of d); the last is the output."""
    lib, mod = rt.load_library(), rt.module()
    packed = rt._ViewArray(tensors, [False] * (len(tensors) - 1) + [True])
    for v, t, sign in zip(packed.views, tensors, strides):
        for d, s in enumerate(sign):
            if s < 0:
                v.data += (t.shape[d] - 1) * v.strides[d]
                v.strides[d] = -v.strides[d]
    sc = (rt.Scalar * len(scalars))(*[rt.scalar(x) for x in scalars])
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    rc = lib.g950_launch(mod._handle, op, packed.views, len(tensors), sc, len(scalars), stream)
    assert rc == rt.OK, lib.g950_last_error().decode()
    torch.cuda.synchronize()
    return lib.g950_last_kernel().decode()


@pytest.mark.parametrize("rev", ["a", "b", "ab"])
@pytest.mark.parametrize("m,n,k,col_b", [(3, 70, 1040, True), (20, 70, 1024, True), (40, 300, 1040, True),
                                         (100, 300, 128, True), (300, 272, 128, True), (300, 272, 128, False),
                                         (40, 80, 528, False)])
@pytest.mark.parametrize("kind", ["bf16", "int8", "w8a16"])
def test_negative_row_strides(kind, m, n, k, col_b, rev):
    """Rows of A and of B (columns, K-contiguous; k-rows, row-major) backwards,
    in the kernels of few rows, tiles, K tails and row-major B."""
    if kind == "int8" and not col_b:
        pytest.skip("row-major int8 x int8 runs the general kernel")
    rng = np.random.default_rng(m + n + k)
    sa, sb = (-1, 1) if "a" in rev else (1, 1), ((1, -1) if col_b else (-1, 1)) if "b" in rev else (1, 1)

    def flip(x, s):
        return np.ascontiguousarray(x[:: s[0], :: s[1]])
    if kind == "bf16":
        a = torch.from_numpy(rng.standard_normal((m, k)).astype(np.float32) / np.float32(np.sqrt(k))).bfloat16()
        b = torch.from_numpy(rng.standard_normal((k, n)).astype(np.float32)).bfloat16()
    else:
        a = (torch.from_numpy(rng.integers(-127, 128, (m, k)).astype(np.int8)) if kind == "int8" else
             torch.from_numpy(rng.standard_normal((m, k)).astype(np.float32) * 0.5).bfloat16())
        b = torch.from_numpy(rng.integers(-127, 128, (k, n)).astype(np.int8))
    bd = b.t().contiguous().to(DEV).t() if col_b else b.to(DEV)
    s = torch.from_numpy((rng.random(n) / 64).astype(np.float32)).bfloat16()
    out = torch.int32 if kind == "int8" else torch.bfloat16
    full = torch.full((m + 2, n), 7, dtype=out, device=DEV)
    args, signs = [a.to(DEV), bd] + ([s.to(DEV)] if kind == "w8a16" else []) + [full[:m]], [sa, sb, (1, 1), (1, 1)]
    op = {"bf16": rt.OP_MATMUL, "int8": rt.OP_MATMUL_I8, "w8a16": rt.OP_DEQUANT_MATMUL}[kind]
    name = launch(op, args, signs, [k, m, n])
    assert "general" not in name
    got = full[:m].cpu()
    if kind == "int8":
        assert np.array_equal(got.numpy(), ref.matmul_i8(flip(a.numpy(), sa), flip(b.numpy(), sb)))
    else:
        bf = flip(b.float().numpy(), sb)
        if kind == "w8a16":
            bf = ref.dequantize(bf.astype(np.int8), s.float().numpy())
        ok, err = ref.isclose_verdict(got.float().numpy(), ref.matmul(flip(a.float().numpy(), sa), bf), 2e-2, 2e-2)
        assert ok, (name, err)
    assert bool((full[m:] == 7).all())
