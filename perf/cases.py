"""The calls this library's speed is judged by: what an inference program that
uses these operators has them do, from one-token steps to full prefills.

Sizes are the repository's own (the benchmark's shapes, the tests' decode and
ragged shapes) or generic transformer sizes.  ``listed()`` names twelve cases;
``draw(rng)`` gives further ones of the same ranges.  ``prepare`` builds what a
program holds before the call, ``run`` makes one call through
``compiler_amd.operators``, ``exact`` is the same result in 64 bits from plain
torch.  Serving-loop cases keep a prepared call on fixed buffers, as such a
loop does; the others call the operator directly.
"""
import math

import torch

from compiler_amd import operators as ops

DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
SIZE = {"bf16": 2, "f16": 2, "f32": 4}


def listed():
    return [
        # one decoding step's norm over a small batch: launch latency and the
        # host's share of a call
        {"name": "rmsnorm_decode", "op": "rmsnorm", "rows": 16, "cols": 4096, "dtype": "bf16"},
        # a norm over a long prompt whose rows are no power of two
        {"name": "layernorm_ragged", "op": "layernorm", "rows": 8191, "cols": 3000, "dtype": "bf16"},
        # row softmax in fp32 (attention scores, router logits)
        {"name": "softmax_fp32", "op": "softmax", "rows": 4096, "cols": 4096, "dtype": "f32"},
        # sampling: probabilities over an odd-sized vocabulary for a batch
        {"name": "softmax_vocab", "op": "softmax", "rows": 256, "cols": 50001, "dtype": "bf16"},
        # a projection in a decoding step: 16 tokens against resident weights
        {"name": "matmul_decode", "op": "matmul", "m": 16, "n": 4096, "k": 4096, "dtype": "bf16",
         "layout": "nk", "prepared": True},
        # the same projection for a chunk of a prompt
        {"name": "matmul_chunk", "op": "matmul", "m": 512, "n": 4096, "k": 4096, "dtype": "bf16",
         "layout": "nk", "prepared": False},
        # a whole batch of prompts: the benchmark's square GEMM
        {"name": "matmul_large", "op": "matmul", "m": 8192, "n": 8192, "k": 8192, "dtype": "bf16",
         "layout": "nk", "prepared": False},
        # quantized inference: int8 x int8 with the dequantising epilogue
        {"name": "int8_dequant", "op": "int8", "m": 4096, "n": 8192, "k": 8192},
        # weight-only quantisation in a decoding step
        {"name": "w8a16_decode", "op": "w8a16", "m": 16, "n": 8192, "k": 8192, "dtype": "bf16",
         "prepared": True},
        # prefill attention of equal prompts: causal, grouped heads, with LSE
        {"name": "attention_prefill", "op": "attention", "z": 4, "h": 32, "hk": 8, "s": 4096, "d": 128,
         "dtype": "bf16", "causal": True},
        # prefill of prompts of different lengths, packed
        {"name": "varlen_prefill", "op": "varlen", "b": 8, "h": 32, "hk": 8, "d": 128, "dtype": "bf16",
         "q_max": 4096, "q_min": 2304, "k_max": 4096, "k_min": 2304, "page": 0, "prepared": False},
        # a decoding step of a batch at different positions on a paged cache
        {"name": "varlen_decode", "op": "varlen", "b": 32, "h": 32, "hk": 8, "d": 128, "dtype": "bf16",
         "q_max": 1, "q_min": 1, "k_max": 4096, "k_min": 300, "page": 64, "prepared": True},
    ]


# ------------------------------------------------------------------ drawing
def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _mult(rng, lo, hi, of):
    return max(of, _log(rng, lo, hi) // of * of)


def draw(rng):
    kind = rng.choice(["rmsnorm", "layernorm", "softmax", "vocab", "matmul", "matmul", "int8", "w8a16",
                       "attention", "varlen", "decode", "decode"])
    half = rng.choice(["bf16", "bf16", "f16"])
    if kind in ("rmsnorm", "layernorm", "softmax"):
        rows, cols = _log(rng, 1, 16384), _log(rng, 256, 8192)
        if rng.random() < 0.7:
            cols = max(8, cols // 8 * 8)
        return {"op": kind, "rows": rows, "cols": cols, "dtype": rng.choice([half, half, "f32"])}
    if kind == "vocab":
        return {"op": rng.choice(["softmax", "logsumexp"]), "rows": _log(rng, 1, 512),
                "cols": _log(rng, 30000, 160000), "dtype": rng.choice([half, "f32"])}
    if kind == "matmul":
        dtype = rng.choice([half, half, half, "f32"])
        m = _log(rng, 1, 8192) if dtype != "f32" else _log(rng, 16, 1024)
        top = 11008 if dtype != "f32" else 4096
        n, k = _mult(rng, 1024, top, 8), _mult(rng, 2048, top, 64)
        if m * n * k > 8192 ** 3:
            m = 8192 ** 3 // (n * k)
        return {"op": "matmul", "m": m, "n": n, "k": k, "dtype": dtype,
                "layout": rng.choice(["nk", "nk", "kn"]), "prepared": m <= 64}
    if kind == "int8":
        return {"op": "int8", "m": _log(rng, 16, 4096), "n": _mult(rng, 1024, 8192, 16),
                "k": _mult(rng, 1024, 8192, 128)}
    if kind == "w8a16":
        m = _log(rng, 1, 1024)
        return {"op": "w8a16", "m": m, "n": _mult(rng, 1024, 11008, 16), "k": _mult(rng, 1024, 11008, 64),
                "dtype": half, "prepared": m <= 64}
    heads = rng.choice([(32, 8), (32, 32), (16, 4), (8, 8), (8, 1)])
    d = rng.choice([128, 128, 64])
    if kind == "attention":
        s = _log(rng, 128, 4096)
        z = max(1, min(_log(rng, 1, 16), 4 * 32 * 4096 ** 2 // (heads[0] * s * s)))
        return {"op": "attention", "z": z, "h": heads[0], "hk": heads[1], "s": s, "d": d, "dtype": half,
                "causal": rng.random() < 0.8 or s > 2500}
    if kind == "varlen":
        b, q = _log(rng, 1, 8), _log(rng, 256, 4096)
        lo = max(1, int(q * rng.uniform(0.3, 1.0)))
        return {"op": "varlen", "b": b, "h": heads[0], "hk": heads[1], "d": d, "dtype": half, "q_max": q,
                "q_min": lo, "k_max": q, "k_min": lo, "page": rng.choice([0, 0, 64, 128]), "prepared": False}
    b, k = _log(rng, 1, 64), _log(rng, 256, 8192)
    q = rng.choice([1, 1, 1, 2, 4])
    return {"op": "varlen", "b": b, "h": heads[0], "hk": heads[1], "d": d, "dtype": half, "q_max": q,
            "q_min": q, "k_max": k, "k_min": max(q, int(k * rng.uniform(0.05, 1.0))),
            "page": rng.choice([0, 16, 64, 64, 128]), "prepared": True}


# ------------------------------------------------------------------- inputs
def _lengths(case):
    """Query and key lengths of a varlen case's sequences, longest first."""
    b = case["b"]
    step = lambda hi, lo, i: hi if b == 1 else hi - (hi - lo) * i // (b - 1)  # noqa: E731
    q = [step(case["q_max"], case["q_min"], i) for i in range(b)]
    k = [step(case["k_max"], case["k_min"], i) for i in range(b)]
    return q, k


def _inputs(case, seed):
    """The input tensors, from the seed alone."""
    g = torch.Generator(device="cuda").manual_seed(seed)

    def normal(shape, dtype, std=1.0, mean=0.0):
        x = torch.randn(shape, generator=g, device="cuda", dtype=torch.float32)
        return (x * std + mean).to(DTYPES[dtype])

    def uniform(shape, lo, hi, dtype="f32"):
        return (torch.rand(shape, generator=g, device="cuda") * (hi - lo) + lo).to(DTYPES[dtype])

    def int8(shape):
        return torch.randint(-127, 128, shape, generator=g, device="cuda", dtype=torch.int8)

    op = case["op"]
    if op in ("rmsnorm", "layernorm", "softmax", "logsumexp"):
        r, c, dt = case["rows"], case["cols"], case["dtype"]
        # vocabulary logits are spread wider than activations
        i = {"x": normal((r, c), dt, 3.0 if c >= 30000 or op == "layernorm" else 1.0)}
        if op in ("rmsnorm", "layernorm"):
            i["w"] = uniform((c,), 0.5, 1.5, dt)
        if op == "layernorm":
            i["b"] = normal((c,), dt, 0.1)
        return i
    if op == "matmul":
        m, n, k, dt = case["m"], case["n"], case["k"], case["dtype"]
        std = 1.0 / math.sqrt(k)
        a = normal((m, k), dt, std)
        b = normal((n, k), dt, std).t() if case["layout"] == "nk" else normal((k, n), dt, std)
        return {"a": a, "b": b}
    if op == "int8":
        m, n, k = case["m"], case["n"], case["k"]
        return {"a": int8((m, k)), "b": int8((n, k)).t(), "sa": uniform((m,), 0.001, 0.02),
                "sb": uniform((n,), 0.001, 0.02)}
    if op == "w8a16":
        m, n, k, dt = case["m"], case["n"], case["k"], case["dtype"]
        return {"a": normal((m, k), dt, 0.5), "b": int8((n, k)).t(), "scale": uniform((n,), 0.001, 0.02, dt)}
    if op == "attention":
        z, h, hk, s, d, dt = (case[n] for n in ("z", "h", "hk", "s", "d", "dtype"))
        return {"q": normal((z, h, s, d), dt), "k": normal((z, hk, s, d), dt), "v": normal((z, hk, s, d), dt)}
    # varlen: token-major tensors; a paged cache holds its pages in shuffled order
    h, hk, d, dt, page = (case[n] for n in ("h", "hk", "d", "dtype", "page"))
    ql, kl = _lengths(case)
    i = {"q": normal((sum(ql), h, d), dt)}
    if page:
        per = [(n + page - 1) // page for n in kl]
        order = torch.randperm(sum(per), generator=g, device="cuda").to(torch.int32)
        table = torch.zeros((case["b"], max(per)), dtype=torch.int32, device="cuda")
        at = 0
        for row, n in enumerate(per):
            table[row, :n] = order[at:at + n]
            at += n
        rows = sum(per) * page
        i["table"] = table
    else:
        rows = sum(kl)
    i["k"], i["v"] = normal((rows, hk, d), dt), normal((rows, hk, d), dt)
    return i


def _varlen_args(case, i, o, lse):
    h, hk, d, page = (case[n] for n in ("h", "hk", "d", "page"))
    ql, kl = _lengths(case)
    cu = lambda n: torch.tensor([sum(n[:j]) for j in range(len(n) + 1)], dtype=torch.int32, device="cuda")  # noqa: E731
    one = torch.zeros(1, dtype=torch.int32, device="cuda")
    scale = 1.0 / math.sqrt(d)
    return dict(
        q_ptr=i["q"], k_ptr=i["k"], v_ptr=i["v"], o_ptr=o, softmax_lse_ptr=lse, p_ptr=one.float(),
        cu_seqlens_q_ptr=cu(ql), cu_seqlens_k_ptr=cu(kl),
        seqused_k_ptr=torch.tensor(kl, dtype=torch.int32, device="cuda"), philox_args=one.to(torch.int64),
        alibi_slopes_ptr=one.float(), page_table_ptr=i["table"] if page else one,
        q_row_stride=h * d, k_row_stride=hk * d, v_row_stride=hk * d, o_row_stride=h * d, q_head_stride=d,
        k_head_stride=d, v_head_stride=d, o_head_stride=d, q_batch_stride=0, k_batch_stride=0, v_batch_stride=0,
        o_batch_stride=0, is_cu_seqlens_q=True, is_cu_seqlens_k=not page, is_seqused_k=bool(page), b=case["b"],
        bk=case["b"], h=h, hk=hk, h_hk_ratio=h // hk, seqlen_q=max(ql), seqlen_k=max(kl),
        seqlen_q_rounded=(max(ql) + 127) // 128 * 128, seqlen_k_rounded=(max(kl) + 31) // 32 * 32, d=d,
        is_softcap=False, softcap=0.0, scale_softmax=scale, scale_softmax_log2=scale * math.log2(math.e),
        is_dropout=False, p_dropout=1.0, rp_dropout=1.0, p_dropout_in_uint8_t=255, return_softmax=False,
        is_causal=True, is_local=False, window_size_left=-1, window_size_right=0, seqlenq_ngroups_swapped=False,
        is_paged=bool(page), is_alibi=False, alibi_slopes_batch_stride=0, total_q=sum(ql),
        page_table_batch_stride=i["table"].shape[1] if page else 0, block_size=page or 1,
        k_page_stride=page * hk * d)


def prepare(case, seed):
    i = _inputs(case, seed)
    state = {"case": dict(case), "i": i}
    if case["op"] == "int8":
        state["y"] = torch.empty((case["m"], case["n"]), dtype=torch.bfloat16, device="cuda")
    if case["op"] == "varlen":
        o = torch.zeros_like(i["q"])
        lse = torch.zeros((case["h"], i["q"].shape[0]), dtype=torch.float32, device="cuda")
        state["args"], state["out"] = _varlen_args(case, i, o, lse), {"o": o, "lse": lse}
    if case.get("prepared"):
        if case["op"] == "varlen":
            state["call"] = ops.flash_varlen_fwd_kernel(**state["args"], prepare=True)
        else:
            y = torch.empty((case["m"], case["n"]), dtype=i["a"].dtype, device="cuda")
            state["out"] = y
            if case["op"] == "matmul":
                state["call"] = ops.matmul_kernel(i["a"], i["b"], y, case["m"], case["n"], case["k"], prepare=True)
            else:
                state["call"] = ops.dequant_matmul_kernel(i["a"], i["b"], i["scale"], y, case["m"], case["n"],
                                                          case["k"], prepare=True)
    return state


def run(state):
    if "call" in state:
        state["call"]()
        return state["out"]
    case, i = state["case"], state["i"]
    op = case["op"]
    if op == "rmsnorm":
        y, r = ops.rmsnorm(i["x"], i["w"], 1e-6)
        return {"y": y, "r": r}
    if op == "layernorm":
        y, mean, rstd = ops.layernorm(i["x"], i["w"], i["b"], 1e-5)
        return {"y": y, "mean": mean, "rstd": rstd}
    if op == "softmax":
        return ops.softmax(i["x"])
    if op == "logsumexp":
        return ops.logsumexp(i["x"])
    if op == "matmul":
        return ops.matmul(i["a"], i["b"])
    if op == "int8":
        ops.matmul_i8_dequant_kernel(i["a"], i["b"], i["sa"], i["sb"], state["y"], case["m"], case["n"], case["k"])
        return state["y"]
    if op == "w8a16":
        return ops.dequant_matmul(i["a"], i["b"], i["scale"])
    if op == "attention":
        o, lse = ops.attention(i["q"], i["k"], i["v"], causal=case["causal"])
        return {"o": o, "lse": lse}
    ops.flash_varlen_fwd_kernel(**state["args"])
    return state["out"]


# --------------------------------------------------------------------- work
def work(case):
    op = case["op"]
    if op in ("rmsnorm", "layernorm", "softmax", "logsumexp"):
        r, c, e = case["rows"], case["cols"], SIZE[case["dtype"]]
        move = {"rmsnorm": 2 * r * c * e + c * e + 4 * r, "layernorm": 2 * r * c * e + 2 * c * e + 8 * r,
                "softmax": 2 * r * c * e, "logsumexp": r * c * e + 4 * r}[op]
        return {"bytes": move, "flops": 5 * r * c}
    if op in ("matmul", "int8", "w8a16"):
        m, n, k = case["m"], case["n"], case["k"]
        if op == "int8":
            move = m * k + n * k + 2 * m * n + 4 * (m + n)
        else:
            e = SIZE[case["dtype"]]
            move = m * k * e + n * k * (1 if op == "w8a16" else e) + m * n * e + (n * e if op == "w8a16" else 0)
        return {"bytes": move, "flops": 2 * m * n * k}
    h, hk, d, e = case["h"], case["hk"], case["d"], SIZE[case["dtype"]]
    if op == "attention":
        z, s = case["z"], case["s"]
        ql, kl = [s] * z, [s] * z
        causal = case["causal"]
    else:
        ql, kl = _lengths(case)
        causal = True
    pairs = sum(q * k - (q * (q - 1) // 2 if causal else 0) for q, k in zip(ql, kl))
    return {"bytes": 2 * sum(ql) * h * d * e + 2 * sum(kl) * hk * d * e + 4 * h * sum(ql),
            "flops": 4 * h * d * pairs}


# ---------------------------------------------------------------- tolerance
def tolerance(case):
    """Against 64 bits the paths measure 1.3e-3 to 1.7e-3 (bf16 outputs: their
    rounding), 2.1e-3 to 2.3e-3 (bf16 attention: the probabilities round as
    well), an eighth of those in f16, 1e-7 in f32 rows and up to 1.2e-6 in f32
    products; four times that, and for a single value a few last-place steps
    of the output type."""
    attn = case["op"] in ("attention", "varlen")
    dtype = case.get("dtype", "bf16")
    if dtype == "f32" or case["op"] == "logsumexp":
        return {"rel": 5e-6 if case["op"] == "matmul" else 1e-6, "max": 1e-4}
    if dtype == "f16":
        return {"rel": 1.2e-3 if attn else 9e-4, "max": 8e-3 if attn else 4e-3}
    return {"rel": 9e-3 if attn else 7e-3, "max": 5e-2 if attn else 2.5e-2}


# -------------------------------------------------------------------- exact
def _attend(q, k, v, scale, first):
    """Softmax attention of one head in 64 bits; query i sees keys <= i + first
    (None: all keys).  Returns the output rows and their logsumexp."""
    s = (q @ k.t()) * scale
    if first is not None:
        i = torch.arange(q.shape[0], device=q.device)[:, None]
        j = torch.arange(k.shape[0], device=q.device)[None, :]
        s.masked_fill_(j > i + first, -math.inf)
    lse = torch.logsumexp(s, -1)
    s.sub_(lse[:, None]).exp_()
    return s @ v, lse


def exact(case, seed):
    i = _inputs(case, seed)
    op = case["op"]
    if op in ("rmsnorm", "layernorm", "softmax", "logsumexp"):
        x = i["x"].double()
        if op == "softmax":
            return torch.softmax(x, -1)
        if op == "logsumexp":
            return torch.logsumexp(x, -1)
        if op == "rmsnorm":
            r = torch.rsqrt((x * x).mean(-1) + 1e-6)
            return {"y": x * r[:, None] * i["w"].double(), "r": r}
        mean = x.mean(-1)
        rstd = torch.rsqrt(((x - mean[:, None]) ** 2).mean(-1) + 1e-5)
        return {"y": (x - mean[:, None]) * rstd[:, None] * i["w"].double() + i["b"].double(), "mean": mean,
                "rstd": rstd}
    if op == "matmul":
        return i["a"].double() @ i["b"].double()
    if op == "int8":
        return (i["a"].double() @ i["b"].double()) * i["sa"].double()[:, None] * i["sb"].double()
    if op == "w8a16":
        return (i["a"].double() @ i["b"].double()) * i["scale"].double()
    h, hk, d = case["h"], case["hk"], case["d"]
    scale = 1.0 / math.sqrt(d)
    if op == "attention":
        o = torch.empty(i["q"].shape, dtype=torch.float64, device="cuda")
        lse = torch.empty(i["q"].shape[:3], dtype=torch.float64, device="cuda")
        for z in range(case["z"]):
            for n in range(h):
                c = n // (h // hk)
                o[z, n], lse[z, n] = _attend(i["q"][z, n].double(), i["k"][z, c].double(), i["v"][z, c].double(),
                                             scale, 0 if case["causal"] else None)
        return {"o": o, "lse": lse}
    ql, kl = _lengths(case)
    page = case["page"]
    o = torch.empty(i["q"].shape, dtype=torch.float64, device="cuda")
    lse = torch.empty((h, i["q"].shape[0]), dtype=torch.float64, device="cuda")
    qa = ka = 0
    for z, (nq, nk) in enumerate(zip(ql, kl)):
        if page:
            j = torch.arange(nk, device="cuda")
            rows = i["table"][z].long()[j // page] * page + j % page
        else:
            rows = torch.arange(ka, ka + nk, device="cuda")
        for n in range(h):
            c = n // (h // hk)
            on, ln = _attend(i["q"][qa:qa + nq, n].double(), i["k"][rows, c].double(), i["v"][rows, c].double(),
                             scale, nk - nq)
            o[qa:qa + nq, n], lse[n, qa:qa + nq] = on, ln
        qa, ka = qa + nq, ka + nk
    return {"o": o, "lse": lse}
