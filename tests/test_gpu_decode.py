"""GPU parity of the few-query attention kernels (g950_attn_dec_*): calls of
flash_varlen_fwd_kernel whose query rows of one KV head (seqlen_q x heads per
KV head) are at most 32, against the CPU oracle at the varlen bars (bf16 1e-2,
fp16 3e-2 on O and LSE: the probabilities and O round to 16 bits)."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from compiler_amd import operators as ops  # noqa: E402
from compiler_amd import runtime as rt  # noqa: E402
from oracle import inputs  # noqa: E402
from oracle import reference as ref  # noqa: E402

import test_gpu_varlen as tv  # noqa: E402

pytestmark = pytest.mark.gpu

# key counts at the edges of a tile (16), a round of the four waves (64), a
# key range (256) and beyond several ranges; 1, 2 and 32 rows per KV head
CASES = {
    "one_key": dict(batches=1, max_q=1, max_k=1, h=4, hk=4, d=128),
    "tile_edges": dict(batches=3, max_q=1, max_k=18, h=8, hk=2, d=128, var_q=False),
    "round_edges": dict(batches=3, max_q=1, max_k=66, h=8, hk=1, d=64, var_q=False),
    "ranges": dict(batches=2, max_q=1, max_k=1500, h=32, hk=8, d=128, var_q=False, causal=True, window_right=0),
    "ranges_d64": dict(batches=2, max_q=2, max_k=2051, h=16, hk=4, d=64, var_q=False, causal=True, window_right=0),
    "rows32": dict(batches=2, max_q=4, max_k=700, h=8, hk=1, d=128, causal=True, window_right=0),
    "rows17": dict(batches=1, max_q=17, max_k=513, h=2, hk=2, d=64, causal=True, window_right=0),
    "group3": dict(batches=2, max_q=5, max_k=300, h=6, hk=2, d=128, causal=True, window_right=0),
    "local": dict(batches=2, max_q=4, max_k=900, h=4, hk=2, d=128, local=True, window_left=100, window_right=0),
    "local_empty": dict(batches=2, max_q=4, max_k=300, h=4, hk=2, d=64, local=True, window_left=-40,
                        window_right=80),
    "paged16": dict(batches=3, max_q=1, max_k=777, h=8, hk=2, d=128, var_q=False, paged=True, block_size=16,
                    causal=True, window_right=0),
    "paged64": dict(batches=2, max_q=4, max_k=4500, h=8, hk=1, d=64, paged=True, block_size=64, causal=True,
                    window_right=0),
    "paged_rows32": dict(batches=2, max_q=4, max_k=1300, h=8, hk=1, d=128, paged=True, block_size=32, causal=True,
                         window_right=0),
    "paged48": dict(batches=2, max_q=1, max_k=400, h=4, hk=4, d=128, var_q=False, paged=True, block_size=48),
    "fewer_keys_than_queries": dict(batches=1, max_q=8, max_k=5, h=2, hk=1, d=64, causal=True, window_right=0),
    "seqused": dict(batches=3, max_q=1, max_k=520, h=8, hk=8, d=128, var_q=False, seqused_trim=37),
}


@pytest.mark.parametrize("dt", ["bfloat16", "float16"])
@pytest.mark.parametrize("case", sorted(CASES))
def test_decode_attention(case, dt):
    a, meta = inputs.varlen_case(**CASES[case])
    tv.check(a, meta, dt, f"g950_attn_dec_{'bf16' if dt == 'bfloat16' else 'f16'}_d{CASES[case]['d']}_")


def test_decode_attention_sequences_without_keys_or_queries():
    """A sequence with no keys (O = 0, LSE = +inf), one with no queries, and
    rows past cu_seqlens_q[-1] (untouched), with and without key ranges."""
    for max_k in (200, 3000):
        a, meta = inputs.varlen_case(batches=3, max_q=6, max_k=max_k, h=4, hk=2, d=128, seqused_trim=5)
        used, cu = a["seqused_k_ptr"].copy(), a["cu_seqlens_q_ptr"].copy()
        used[0] = 0
        cu[2] = cu[1]
        cu[3] = cu[2] + 2
        a = dict(a, seqused_k_ptr=used, cu_seqlens_q_ptr=cu)
        tv.check(a, meta, "bfloat16", "g950_attn_dec_")


def test_decode_attention_scores_climb():
    """Scores that grow with the key index by about 16 log2 units per 64 keys:
    every tile moves the reference maximum, and the key ranges' maxima lie far
    apart when they are joined."""
    a, meta = inputs.varlen_case(batches=2, max_q=1, max_k=2000, h=8, hk=2, d=128, var_q=False, var_k=False)
    q = a["q_ptr"].reshape(-1, 128)
    q[:, 0] = 4.0
    k = a["k_ptr"].reshape(2, 2000, 2, 128)
    k[..., 0] = np.arange(2000)[None, :, None] / 64 * 16 / 1.4427 / (meta["scale_softmax"] * 4.0)
    tv.check(dict(a, q_ptr=q.reshape(-1), k_ptr=k.reshape(-1)), meta, "bfloat16", "g950_attn_dec_")


@pytest.mark.parametrize("seqlen_q,d", [(1, 128), (2, 64), (5, 128)])
def test_decode_attention_longer_sequences_than_seqlen_q(seqlen_q, d):
    """cu_seqlens_q lives on the device, so a sequence may hold more queries
    than the scalar seqlen_q (1 and 2 queries: fewer rows than the kernel's
    tile holds): every query is computed, and the partial records of the other
    sequences and KV heads are left alone."""
    a, meta = inputs.varlen_case(batches=3, max_q=12, max_k=2500, h=8, hk=2, d=d, causal=True, window_right=0)
    tv.check(dict(a, seqlen_q=seqlen_q), meta, "bfloat16", "g950_attn_dec_")
    assert rt.module().last_kernel.endswith("_merge")


def device_args(a, dt=torch.bfloat16):
    t = {n: torch.from_numpy(np.ascontiguousarray(a[n]).view(np.int64) if a[n].dtype == np.uint64
                             else np.ascontiguousarray(a[n])).to("cuda") for n in ops._VARLEN_VIEWS}
    for n in ("q_ptr", "k_ptr", "v_ptr", "o_ptr"):
        t[n] = t[n].to(dt)
    return t


def test_decode_attention_without_workspace():
    """No-alloc calls and captured graphs keep to one workgroup per pair (no
    workspace) and give the same results; a graph replayed between other work
    gives its own result again."""
    a, meta = inputs.varlen_case(batches=2, max_q=1, max_k=3000, h=8, hk=2, d=128, var_q=False, var_k=False)
    t = device_args(a)
    scal = {n: {**a, **meta}[n] for n in ops._VARLEN_SCALARS}
    ops.flash_varlen_fwd_kernel(**t, **scal, sync=True)
    assert rt.module().last_kernel.endswith("_merge")
    split = t["o_ptr"].clone()
    with rt.no_alloc():
        ops.flash_varlen_fwd_kernel(**t, **scal, sync=True)
    assert rt.module().last_kernel == "g950_attn_dec_bf16_d128_r16"
    one = t["o_ptr"].clone()
    ok, err = ref.isclose_verdict(one.float().cpu().numpy(), split.float().cpu().numpy(), 1e-2, 1e-2)
    assert ok, err
    graph, stream = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    with torch.cuda.graph(graph, stream=stream):
        ops.flash_varlen_fwd_kernel(**t, **scal)
    for _ in range(3):
        t["o_ptr"].zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(t["o_ptr"], one)
        ops.flash_varlen_fwd_kernel(**t, **scal, sync=True)
        assert torch.equal(t["o_ptr"], split)


def test_decode_attention_leaves_captured_workspace_alone():
    """A graph may hold the address of its stream's workspace (split softmax
    rows): a decoding step's key ranges on that stream, which need more, leave
    it as it is."""
    stream = torch.cuda.Stream()
    a, meta = inputs.varlen_case(batches=4, max_q=1, max_k=4000, h=32, hk=8, d=128, var_q=False, var_k=False)
    t = device_args(a)
    scal = {n: {**a, **meta}[n] for n in ops._VARLEN_SCALARS}
    x = torch.randn(2, 60000, device="cuda")
    y = torch.zeros_like(x)
    torch.cuda.synchronize()
    with torch.cuda.stream(stream):
        ops.softmax_kernel(x, y, 60000, sync=True)
        assert rt.module().last_kernel.startswith("g950_rs_final_softmax")
        want = y.clone()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        ops.softmax_kernel(x, y, 60000)
    held = rt.module().workspace_bytes(stream)
    with torch.cuda.stream(stream):
        ops.flash_varlen_fwd_kernel(**t, **scal, sync=True)
        assert rt.module().last_kernel.endswith("_merge")
    # the key ranges came on top of what the softmax call holds
    recs = 4 * 32 * 16
    assert rt.module().workspace_bytes(stream) >= held + recs * (128 + 2) * 4
    for _ in range(3):
        y.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, want)


SAME_BITS = {n: CASES[n] for n in ("ranges", "ranges_d64", "rows32", "rows17", "local", "paged16", "paged64",
                                 "paged_rows32", "seqused")}
SAME_BITS["one_long"] = dict(batches=1, max_q=1, max_k=8000, h=8, hk=1, d=128, causal=True, window_right=0)


@pytest.mark.parametrize("case", sorted(SAME_BITS) + ["longer_than_seqlen_q", "climbing", "not_finite"])
def test_decode_attention_same_bits_without_workspace(case):
    """A call gives the same bits whether its key ranges run side by side (own
    workspace), under no_alloc or in a captured graph, on every replay: the
    ranges are joined by the same operations in the same order.  Also where
    sequences hold more queries than seqlen_q, where every range moves the
    maximum, and where keys are inf or NaN."""
    a, meta = inputs.varlen_case(**SAME_BITS.get(case, dict(batches=2, max_q=5, max_k=2500, h=8, hk=2, d=128, causal=True,
                                                            window_right=0)))
    scal = {n: {**a, **meta}[n] for n in ops._VARLEN_SCALARS}
    t = device_args(a)
    if case == "longer_than_seqlen_q":
        scal["seqlen_q"] = 2
    rows = t["k_ptr"].view(-1, 2, 128) if case in ("climbing", "not_finite") else None
    if case == "climbing":
        rows *= (torch.arange(rows.shape[0], device="cuda")[:, None, None] / 40).to(rows.dtype)
    if case == "not_finite":
        rows[700, 0], rows[900, 1] = float("inf"), float("nan")
    out = ("o_ptr", "softmax_lse_ptr")

    def result():
        torch.cuda.synchronize()
        return [t[n].view(torch.int16 if n == "o_ptr" else torch.int32).clone() for n in out]

    def poison():
        for n in out:
            t[n].fill_(7.0)

    poison()
    ops.flash_varlen_fwd_kernel(**t, **scal, sync=True)
    assert rt.module().last_kernel.endswith("_merge")
    want = result()
    graph, stream = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    with torch.cuda.graph(graph, stream=stream):
        ops.flash_varlen_fwd_kernel(**t, **scal)
    for _ in range(3):
        poison()
        graph.replay()
        assert all(torch.equal(g, w) for g, w in zip(result(), want))
        poison()
        ops.flash_varlen_fwd_kernel(**t, **scal)
        assert all(torch.equal(g, w) for g, w in zip(result(), want))
    poison()
    with rt.no_alloc():
        ops.flash_varlen_fwd_kernel(**t, **scal)
    assert not rt.module().last_kernel.endswith("_merge")
    assert all(torch.equal(g, w) for g, w in zip(result(), want))


def test_decode_attention_per_thread_streams_share_no_workspace():
    """hipStreamPerThread (handle 2) is one handle for a stream of every
    thread: calls on it take no workspace, and give the same bits, also from
    two threads at once."""
    import threading
    a, meta = inputs.varlen_case(batches=2, max_q=1, max_k=3000, h=8, hk=2, d=128, var_q=False, var_k=False)
    scal = {n: {**a, **meta}[n] for n in ops._VARLEN_SCALARS}
    t = [device_args(a) for _ in range(2)]
    ops.flash_varlen_fwd_kernel(**t[0], **scal, sync=True)
    want = t[0]["o_ptr"].clone()
    t[0]["o_ptr"].zero_()
    torch.cuda.synchronize()
    names, held = [], rt.module().workspace_bytes(2)

    def calls(args):
        for _ in range(20):
            ops.flash_varlen_fwd_kernel(**args, **scal, stream=2)
        rt.load_library().g950_sync(2)
        names.append(rt.load_library().g950_last_kernel().decode())
    threads = [threading.Thread(target=calls, args=(x,)) for x in t]
    for th in threads:
        th.start()
    for th in threads:
        th.join()
    torch.cuda.synchronize()
    assert names == ["g950_attn_dec_bf16_d128_r16"] * 2 and rt.module().workspace_bytes(2) == held == 0
    assert all(torch.equal(x["o_ptr"], want) for x in t)
