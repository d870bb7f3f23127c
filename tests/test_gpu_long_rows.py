"""GPU parity of the one-workgroup-per-row masked kernels (g950_rl_*) and of
the masked chunks of the split kernels, for every row operator: row lengths
one element around each form's capacity, every 16-byte phase of the row
starts (odd row strides), gaps between rows untouched, special values in the
edge vectors' neighbours; against the CPU oracle (fp32 1e-5, 16-bit 1e-2)."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from compiler_amd import operators as ops  # noqa: E402
from compiler_amd import runtime as rt  # noqa: E402
from oracle import reference as ref  # noqa: E402

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
TD = {"float32": torch.float32, "bfloat16": torch.bfloat16, "float16": torch.float16}


def case(rows, cols, stride, dt, seed):
    """x as the cols first elements of rows `stride` apart, the gaps holding
    the largest finite values (they must never reach a reduction)."""
    rng = np.random.default_rng(seed)
    big = {"float32": 3e38, "bfloat16": 3e38, "float16": 6e4}[dt]
    full = torch.full((rows * stride + 16,), big, dtype=TD[dt], device=DEV)
    x = torch.as_strided(full, (rows, cols), (stride, 1), 3)
    x.copy_(torch.from_numpy((rng.standard_normal((rows, cols)) * 3).astype(np.float32)).to(DEV))
    w = torch.from_numpy(rng.uniform(0.5, 1.5, cols + 1).astype(np.float32)).to(DEV).to(TD[dt])[1:]
    b = torch.from_numpy((rng.standard_normal(cols + 1) * 0.1).astype(np.float32)).to(DEV).to(TD[dt])[1:]
    return x, w, b


def guarded(rows, cols, stride, dt):
    full = torch.full((rows * stride + 16,), -7.0, dtype=TD[dt], device=DEV)
    return full, torch.as_strided(full, (rows, cols), (stride, 1), 3)


def host(t):
    return t.float().cpu().numpy()


SHAPES = {  # rows, cols, extra stride, kernel prefix
    "float32": [(130, 2049, 1, "rl"), (140, 4089, 0, "rl"), (129, 4097, 3, "rl"), (128, 8191, 0, "rl"),
                (131, 32761, 2, "rl"), (3, 20001, 1, "rs"), (2, 70001, 0, "rs"), (101, 17001, 1, "rs"),
                (2, 800001, 0, "rs"), (262, 9001, 0, "rs"), (390, 8201, 1, "rl")],
    "bfloat16": [(5, 4097, 0, "rl"), (130, 8185, 1, "rl"), (128, 8193, 6, "rl"), (129, 16379, 0, "rl"),
                 (128, 50001, 0, "rl"), (128, 65521, 3, "rl"), (3, 40001, 1, "rs"), (2, 140001, 0, "rs"),
                 (61, 40001, 0, "rs"), (262, 17001, 1, "rs"), (2, 800001, 1, "rs"), (449, 16401, 0, "rl")],
}
SHAPES["float16"] = SHAPES["bfloat16"][1::2]


@pytest.mark.parametrize("dt,shape", [(d, s) for d in SHAPES for s in SHAPES[d]])
def test_long_odd_rows(dt, shape):
    rows, cols, extra, kind = shape
    stride = cols + extra
    x, w, b = case(rows, cols, stride, dt, rows + cols)
    xr, wr, br = host(x), host(w), host(b)
    bar = (1e-5, 1e-6) if dt == "float32" else (1e-2, 1e-2)

    def check(got, want, rtol, atol, kind=kind):
        ok, err = ref.isclose_verdict(got, want, rtol, atol)
        assert ok, (rt.module().last_kernel, err)
        name = rt.module().last_kernel
        assert name.startswith(f"g950_{kind}_") and "_v1" in name, name
        if kind == "rs":
            limit = 256 * (6 if "layernorm" in name else 4)
            many = rows * -(-cols // 1024) > limit
            assert rt.load_library().g950_last_form() == (b"vectors" if many else b"elements"), name

    full, y = guarded(rows, cols, stride, dt)
    ops.softmax_kernel(x, y, cols, sync=True)
    check(host(y), ref.softmax(xr), *bar)
    lse = torch.empty(rows, device=DEV)
    ops.logsumexp_kernel(x, lse, cols, sync=True)
    # logsumexp splits rows that reach past 2048 vectors at some phase
    v = 16 // x.element_size()
    check(lse.cpu().numpy(), ref.logsumexp(xr), 3e-5, 3e-6, "rs" if (cols + 2 * (v - 1)) // v > 2048 else kind)
    r = torch.empty(rows, device=DEV)
    ops.rms_layernorm_forward_kernel(y, stride, x, stride, w, 1, r, 1, cols, 1e-6, sync=True)
    ey, er = ref.rms_layernorm(xr, wr, 1e-6)
    check(host(y), ey, *bar)
    check(r.cpu().numpy(), er, 1e-5, 1e-6)
    mean, rstd = torch.empty(rows, device=DEV), torch.empty(rows, device=DEV)
    ops.layernorm_kernel(x, y, w, b, mean, rstd, stride, cols, 1e-5, sync=True)
    ey, em, es = ref.layernorm(xr, wr, br, 1e-5)
    check(host(y), ey, *(bar if dt != "float32" else (1e-5, 1e-5)))
    check(mean.cpu().numpy(), em, 1e-5, 1e-6)
    check(rstd.cpu().numpy(), es, 1e-5, 1e-6)
    y.fill_(-7.0)
    assert bool((full == -7.0).all())


# rows whose vectors fill their chunks exactly at some phases and reach one
# vector further at others (chunks of 1024 vectors): the last chunk is empty
# for part of the rows
@pytest.mark.parametrize("dt,cols,rows", [("bfloat16", 8186, 9), ("bfloat16", 8190, 9), ("bfloat16", 16383, 9),
                                          ("float16", 8192, 9), ("float32", 4095, 9), ("float32", 4094, 9),
                                          ("float32", 12287, 9), ("bfloat16", 16378, 126), ("bfloat16", 16383, 126),
                                          ("float16", 24575, 126), ("float32", 16381, 126), ("float32", 16383, 126)])
def test_split_rows_last_chunk_empty(dt, cols, rows):
    stride = cols + 1
    x, w, b = case(rows, cols, stride, dt, cols)
    _, y = guarded(rows, cols, stride, dt)
    xr, wr, br = host(x), host(w), host(b)
    bar = (1e-5, 1e-6) if dt == "float32" else (1e-2, 1e-2)
    mean, rstd = torch.empty(rows, device=DEV), torch.empty(rows, device=DEV)
    ops.layernorm_kernel(x, y, w, b, mean, rstd, stride, cols, 1e-5, sync=True)
    assert rt.module().last_kernel.startswith("g950_rs_final_layernorm") and "_v1" in rt.module().last_kernel
    # (few rows run by elements; only vectors can leave a chunk empty)
    assert rt.load_library().g950_last_form() == (b"elements" if rows == 9 else b"vectors")
    want = ref.layernorm(xr, wr, br, 1e-5)
    ln_bar = bar if dt != "float32" else (1e-5, 1e-5)
    for got, exp, (rtol, atol) in zip((host(y), mean.cpu().numpy(), rstd.cpu().numpy()), want,
                                      (ln_bar, (1e-5, 1e-6), (1e-5, 1e-6))):
        ok, err = ref.isclose_verdict(got, exp, rtol, atol)
        assert ok, err
    ops.softmax_kernel(x, y, cols, sync=True)
    ok, err = ref.isclose_verdict(host(y), ref.softmax(xr), *bar)
    assert ok, err
    r = torch.empty(rows, device=DEV)
    ops.rms_layernorm_forward_kernel(y, stride, x, stride, w, 1, r, 1, cols, 1e-6, sync=True)
    ok, err = ref.isclose_verdict(host(y), ref.rms_layernorm(xr, wr, 1e-6)[0], *bar)
    assert ok, err


@pytest.mark.parametrize("rows,cols", [(130, 131065), (129, 65537), (128, 131072)])
def test_long_rows_packed(rows, cols):
    """softmax and logsumexp rows past the widened forms: bf16 up to 131072
    elements in one workgroup, aligned ones too, and the special rows."""
    x = (torch.randn(rows, cols, device=DEV) * 3).to(torch.bfloat16)
    x[1, 5], x[2, cols - 1], x[3, :], x[4, 0] = float("inf"), float("nan"), float("-inf"), float("-inf")
    xr = host(x)
    y = ops.softmax(x, sync=True)
    assert rt.module().last_kernel == "g950_rl_softmax_bf16_v1_i16_b1024"
    got = host(y)
    with np.errstate(invalid="ignore"):
        want = ref.softmax(xr)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    keep = ~np.isnan(want)
    ok, err = ref.isclose_verdict(got[keep], want[keep], 1e-2, 1e-2)
    assert ok, err
    assert abs(got[5].astype(np.float64).sum() - 1) < 1e-2
    lse = ops.logsumexp(x, sync=True).cpu().numpy()
    want = ref.logsumexp(xr)
    assert np.array_equal(np.isnan(lse), np.isnan(want)) and np.isposinf(lse[1]) and np.isneginf(lse[3])
    ok, err = ref.isclose_verdict(lse[5:], want[5:], 3e-5, 3e-6)
    assert ok, err


# the most columns a row may have, and the most that vectors take (at two
# 16-byte phases; y one element off x's phase: elements)
@pytest.mark.parametrize("n,offset,y_offset", [(2**31 - 1, 3, 3), (2**31 - 16385, 0, 0), (2**31 - 16385, 3, 3),
                                               (2**31 - 16385, 0, 1), (2**31 - 9001, 0, 0)])
def test_split_rows_of_the_most_columns(n, offset, y_offset):
    """Columns up to 2^31 - 1: the last chunk counts (its values alone set the
    variance and the logsumexp) and no vector past the row is read.  Four
    buffers of 4.3 GB.  LayerNorm bf16: the statistics within 1e-4 (fp32 sums of 2^31
    terms in chunks), y within bf16 rounding."""
    pad, tail, big = 16, 4000, 1024.0
    vectors = n <= 2**31 - 16385 and offset == y_offset
    g = torch.Generator(device="cuda").manual_seed(1)
    xs = torch.empty(n + pad, dtype=torch.bfloat16, device="cuda")
    for c in xs.split(1 << 28):
        c.normal_(generator=g)
    x = xs[offset:offset + n].view(1, n)
    x[0, -tail:] = big
    mean = sum(c.double().sum().item() for c in x[0].split(1 << 27)) / n
    var = sum((c.double() - mean).square().sum().item() for c in x[0].split(1 << 27)) / n
    ys = torch.full((n + pad,), 7.0, dtype=torch.bfloat16, device="cuda")
    y = ys[y_offset:y_offset + n].view(1, n)
    w = torch.ones(n, dtype=torch.bfloat16, device="cuda")
    b = torch.zeros(n, dtype=torch.bfloat16, device="cuda")
    _, m, r = ops.layernorm(x, w, b, 1e-5, out=y, sync=True)
    assert rt.module().last_kernel == "g950_rs_final_layernorm_bf16_v1"
    assert rt.load_library().g950_last_form() == (b"vectors" if vectors else b"elements")
    rstd = (var + 1e-5) ** -0.5
    assert abs(m.item() - mean) < 1e-4 and abs(r.item() / rstd - 1) < 1e-4
    for xc, yc in zip(x[0].split(1 << 27), y[0].split(1 << 27)):
        want = (xc.float() - mean) * rstd
        assert bool(((want - yc.float()).abs() <= 2**-8 * want.abs() + 1e-3).all())
    assert bool((ys[:y_offset] == 7.0).all()) and bool((ys[y_offset + n:] == 7.0).all())
    if y_offset == offset:
        del y, ys
        x[0, -tail:] = 0.0
        x[0, -1] = 40.0
        lse = ops.logsumexp(x, sync=True)
        assert rt.module().last_kernel == "g950_rs_final_logsumexp_bf16_v1"
        assert abs(lse.item() - 40.0) < 1e-3  # log(e^40 + 2^31 e^0.5): 1.5e-8 past 40


def test_poorly_filled_rounds_under_capture():
    """262 rows run the split pair; captured on a stream that holds no
    workspace (nothing can be allocated there) one workgroup per row, on one
    that does the split pair again.  Every replay gives the eager result (fp32
    exponentials and sums in another order: 2e-5)."""
    x = torch.randn(262, 33000, device=DEV)
    want = torch.softmax(x, -1)
    y = torch.empty_like(x)
    torch.cuda.synchronize()
    for warm in (False, True):
        stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
        if warm:
            with torch.cuda.stream(stream):
                ops.softmax_kernel(x, y, 33000, sync=True)
            assert rt.module().last_kernel == "g950_rs_final_softmax_f32_v4"
        held = rt.module().workspace_bytes(stream)
        with torch.cuda.graph(graph, stream=stream):
            ops.softmax_kernel(x, y, 33000)
        if held:
            assert rt.module().last_kernel == "g950_rs_final_softmax_f32_v4"
        else:
            assert rt.module().last_kernel == "g950_rl_softmax_f32_v1_i16_b1024"
        assert rt.module().workspace_bytes(stream) == held
        for _ in range(3):
            y.fill_(7.0)
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.allclose(y, want, rtol=2e-5, atol=0)
