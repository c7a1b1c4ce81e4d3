"""The measured cases of the paged-attention library: decode, prefill, mixed
batches and the KV-cache write, through the package's public entry points.

Every case is one call a serving loop makes for one layer, over a paged pool
whose pages are scattered (a random permutation as block table).  Calls with
the reference operators' types (fp32 q, fp32 output) and the short ones go
through torch.ops.gb10_attn.*, calls that pick the output type through the
Python functions with the output (and scratch) tensors the program keeps.
K, V and q are N(0, 1); FP8 caches hold the values divided by 1/16.

Ranges.  Heads are GPT-2 style (12 x 64), GQA groups of 4 and 8 at head_dim
128 and 64 and their tensor-parallel shares; pages of 16 tokens mostly, of 8
and 32 now and then; batches of 1 to 256 sequences, contexts of 1 to 32768
tokens, uniform or ragged; prefill chunks of 1 to 4096 rows, whole prompts or
behind a cached prefix; caches of fp16, bf16 and FP8 (E4M3).
"""
import math
import random

import numpy as np
import torch

import __graft_entry__

DT = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16, "fp8": torch.float8_e4m3fn}
SIZE = {"f32": 4, "f16": 2, "bf16": 2, "fp8": 1}
FP8_SCALE = 1.0 / 16

MAX_BYTES = 2.2e9    # the most KV bytes a drawn case touches (the ragged GQA decode below)
MAX_FLOPS = 2.7e11   # the most matrix work of a drawn prefill (the long-prompt prefill below)
MAX_FLOPS32 = 1.1e10  # of a drawn fp32-arithmetic prefill


def listed():
    gpt2 = dict(H=12, HKV=12, D=64, BS=16)
    llama = dict(H=32, HKV=8, D=128, BS=16)
    ref = dict(q="f32", out="f32", api="op")  # the reference operators' types
    return [
        # One user's next token at a short context: launch latency, a few work-groups.
        dict(name="decode_b1_c512", kind="decode", B=1, ctx=512, ragged=False, kv="f16", splits=0, **gpt2, **ref),
        # A small batch as the reference's own harness calls v3: its fp32 q and its chosen split count.
        dict(name="decode_b16_c2048_split", kind="decode", B=16, ctx=2048, ragged=False, kv="f16", splits=-1, **gpt2,
             **ref),
        # A full decode batch of a GPT-2 size model: the library's headline workload.
        dict(name="decode_b64_c2048", kind="decode", B=64, ctx=2048, ragged=False, kv="f16", splits=0, q="f16",
             out="f16", api="py", **gpt2),
        # Grouped-query decode over a ragged batch of long contexts, bf16 model.
        dict(name="decode_gqa4_ragged", kind="decode", B=32, ctx=32768, ragged=True, kv="bf16", splits=0, q="bf16",
             out="bf16", api="py", **llama),
        # The same batch over a quantised cache.
        dict(name="decode_gqa4_ragged_fp8", kind="decode", B=32, ctx=32768, ragged=True, kv="fp8", splits=0, q="bf16",
             out="bf16", api="py", **llama),
        # Groups of eight query heads (a larger model), long uniform contexts.
        dict(name="decode_gqa8_c8192", kind="decode", B=32, ctx=8192, ragged=False, kv="bf16", splits=0, q="bf16",
             out="bf16", api="py", H=64, HKV=8, D=128, BS=16),
        # Prompts of a batch, head_dim 64: many short causal blocks.
        dict(name="prefill_b8_s1024", kind="prefill", B=8, S=1024, ctx=1024, kv="f16", q="f16", out="f32", api="op",
             **gpt2),
        # Long prompts, head_dim 128: the largest matrix work.
        dict(name="prefill_b2_s4096", kind="prefill", B=2, S=4096, ctx=4096, kv="bf16", q="bf16", out="bf16",
             api="py", H=32, HKV=32, D=128, BS=16),
        # Chunked prefill behind a cached prefix, the reference harness's shape and types.
        dict(name="prefill_chunk_c2048", kind="prefill", B=4, S=512, ctx=2048, kv="f16", **gpt2, **ref),
        # The same chunk through the fp32-arithmetic prefill operator.
        dict(name="prefill32_chunk_c2048", kind="prefill32", B=4, S=512, ctx=2048, kv="f16", **gpt2, **ref),
        # A continuous-batching step: decoding sequences and prompt chunks in one packed call.
        dict(name="mixed_64x1_4x256", kind="mixed", nd=64, npf=4, S=256, ctx=2048, ragged=False, kv="f16", q="f16",
             out="f32", api="op", **gpt2),
        # The prompt's new K/V rows quantised into the paged FP8 cache.
        dict(name="write_t8192_fp8", kind="write", T=8192, src="bf16", kv="fp8", HKV=32, D=128, BS=16),
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["decode"] * 4 + ["prefill"] * 3 + ["prefill32", "mixed", "mixed", "write"])
    H, HKV, D = rng.choice([(12, 12, 64), (12, 12, 64), (32, 8, 128), (32, 8, 128), (64, 8, 128), (8, 2, 128),
                            (8, 1, 128), (16, 16, 128), (16, 4, 64)])
    BS = rng.choice([16, 16, 16, 16, 32, 8])
    kv = rng.choice(["f16", "f16", "bf16", "bf16", "fp8"])
    c = dict(kind=kind, HKV=HKV, D=D, BS=BS, kv=kv)
    row = 2 * HKV * D * SIZE[kv]  # K and V bytes of one token
    if kind == "write":
        c.update(T=_log(rng, 1, 8192), src=rng.choice(["f16", "bf16", "f32"]))
        if kv != "fp8" and c["src"] != "f32":
            c["src"] = kv
        return c
    # The model's activations: fp32 (the reference's operators) or the cache's 16-bit type.
    q = rng.choice(["f32", "act"])
    q = {"f16": "f16", "bf16": "bf16", "fp8": rng.choice(["f16", "bf16"])}[kv] if q == "act" else "f32"
    c.update(H=H, q=q, api="op", out="f32")
    if q != "f32" and rng.random() < 0.5:
        c.update(api="py", out=q)
    if kind == "decode":
        B = _log(rng, 1, 256)
        ctx = _log(rng, 32, max(32, min(32768, int(MAX_BYTES / (row * B)))))
        c.update(B=B, ctx=ctx, ragged=rng.random() < 0.5, splits=rng.choice([0, 0, -1]))
        return c
    if kind == "mixed":
        nd, npf = _log(rng, 1, 96), rng.randint(1, 6)
        c.update(nd=nd, npf=npf, S=_log(rng, 16, 1024), ragged=rng.random() < 0.5)
        c["ctx"] = max(c["S"], _log(rng, 64, 8192))
        while work(c)["flops"] > MAX_FLOPS or row * (nd + npf) * c["ctx"] > MAX_BYTES:
            c["ctx"] = max(c["S"], c["ctx"] // 2)
            c["nd"] = nd = max(1, nd // 2)
        return c
    B = rng.choice([1, 1, 2, 3, 4, 8])
    S = _log(rng, 16, 4096) if kind == "prefill" else _log(rng, 8, 1024)
    prefix = rng.choice([0, _log(rng, 1, 16384 if kind == "prefill" else 4096)])
    c.update(B=B, S=S, ctx=S + prefix)
    if kind == "prefill32":
        # (The scaled FP8 form exists for the matrix-core prefill only.)
        c["kv"] = kv = "f16" if kv == "fp8" else kv
        c["q"] = "f32" if q not in ("f32", kv) else q
        c.update(api="op", out="f32")
    top = MAX_FLOPS if kind == "prefill" else MAX_FLOPS32
    while work(c)["flops"] > top:
        c["B"] = max(1, c["B"] // 2)
        c["S"] = max(8, c["S"] * 3 // 4)
        c["ctx"] = max(c["S"], c["ctx"] * 3 // 4)
    return c


# ------------------------------------------------------------------ inputs --

def _lens(c):
    """Context lengths of the case (the same for every seed): all `ctx`, or ragged over [ctx / 32, ctx]."""
    n = c["nd"] + c["npf"] if c["kind"] == "mixed" else c["B"]
    if not c.get("ragged"):
        return [c["ctx"]] * n
    r = np.random.default_rng(3)
    lens = [int(x) for x in r.integers(max(1, c["ctx"] // 32), c["ctx"] + 1, n)]
    return [max(x, y) for x, y in zip(lens, _rows(c))]


def _rows(c):
    """New query rows of each sequence."""
    if c["kind"] == "decode":
        return [1] * c["B"]
    if c["kind"] != "mixed":
        return [c["S"]] * c["B"]
    if not c["ragged"]:
        return [1] * c["nd"] + [c["S"]] * c["npf"]
    r = np.random.default_rng(4)
    return [1] * c["nd"] + [int(x) for x in r.integers(max(2, c["S"] // 4), c["S"] + 1, c["npf"])]


def _randn(shape, g, dtype, mul=1.0):
    if dtype == "fp8":
        x = torch.empty(shape, dtype=torch.float8_e4m3fn, device="cuda")
        flat, step = x.view(-1), 1 << 28
        for i in range(0, flat.numel(), step):
            n = min(step, flat.numel() - i)
            flat[i:i + n] = (torch.randn(n, generator=g, device="cuda", dtype=torch.float16) * mul).to(x.dtype)
        return x
    return torch.randn(shape, generator=g, device="cuda", dtype=DT[dtype])


def _inputs(c, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed * 7919 + 11)
    rng = np.random.default_rng(seed)
    HKV, D, BS, s = c["HKV"], c["D"], c["BS"], {}
    if c["kind"] == "write":
        T = c["T"]
        nb = -(-T // BS) + 3
        s["key"] = _randn((T, HKV, D), g, c["src"])
        s["value"] = _randn((T, HKV, D), g, c["src"])
        s["k"] = torch.zeros((nb, BS, HKV, D), device="cuda", dtype=DT[c["kv"]])
        s["v"] = torch.zeros((nb, BS, HKV, D), device="cuda", dtype=DT[c["kv"]])
        pages, t = rng.permutation(nb), np.arange(T)
        s["slots"] = torch.from_numpy(pages[t // BS] * BS + t % BS).cuda()
        return s
    lens, rows = _lens(c), _rows(c)
    pages = [-(-n // BS) for n in lens]
    nb, mb = sum(pages), max(pages)
    s["k"] = _randn((nb, BS, HKV, D), g, c["kv"], 1 / FP8_SCALE)
    s["v"] = _randn((nb, BS, HKV, D), g, c["kv"], 1 / FP8_SCALE)
    perm, bt, at = rng.permutation(nb).astype(np.int32), np.zeros((len(lens), mb), np.int32), 0
    for i, n in enumerate(pages):
        bt[i, :n] = perm[at:at + n]
        at += n
    s["bt"] = torch.from_numpy(bt).cuda()
    s["ctx"] = torch.tensor(lens, dtype=torch.int32, device="cuda")
    shape = {"decode": (len(lens), c["H"], D), "mixed": (sum(rows), c["H"], D)}.get(
        c["kind"], (len(lens), c.get("S"), c["H"], D))
    s["q"] = _randn(shape, g, c["q"])
    if c["kind"] == "mixed":
        s["cu"] = torch.tensor(np.concatenate([[0], np.cumsum(rows)]), dtype=torch.int32, device="cuda")
    return s


def prepare(case, seed):
    pa = __graft_entry__.load_package()
    s = _inputs(case, seed)
    s["pa"], s["ops"], s["case"] = pa, pa.torch_ops(), case
    s["scale"] = 1.0 / math.sqrt(case["D"])
    s["kvs"] = FP8_SCALE if case["kv"] == "fp8" else 1.0
    if case["kind"] == "mixed":
        s["max_q"] = max(_rows(case))
    if case["kind"] == "decode":
        s["splits"] = case["splits"]
        if case["splits"] < 0:  # the reference's harness asks its chooser for the count
            s["splits"] = pa.choose_num_splits(case["B"], case["H"], max(_lens(case)))
    if case.get("api") == "py":
        s["out"] = torch.empty(s["q"].shape, dtype=DT[case["out"]], device="cuda")
        if case["kind"] == "decode":
            n = pa.workspace_size(s["q"], s["k"], s["bt"], s["splits"])
            s["ws"] = torch.empty(max(n, 256), dtype=torch.uint8, device="cuda")
    return s


# --------------------------------------------------------------------- run --

def run(s):
    c, f8 = s["case"], s["kvs"]
    if c["kind"] == "write":
        s["ops"].write_kv_scaled(s["k"], s["v"], s["key"], s["value"], s["slots"], f8, f8)
        if c["kv"] == "fp8":
            return s["k"].view(torch.uint8), s["v"].view(torch.uint8)
        return s["k"], s["v"]
    a = (s["q"], s["k"], s["v"], s["bt"], s["ctx"])
    if c["kind"] == "prefill32":
        return s["ops"].paged_attention_prefill(*a, s["scale"])
    if c["api"] == "py":
        kw = dict(out=s["out"], k_scale=f8, v_scale=f8)
        if c["kind"] == "decode":
            return s["pa"].paged_attention_v3(*a, s["scale"], s["splits"], workspace=s["ws"], **kw)
        if c["kind"] == "prefill":
            return s["pa"].paged_attention_prefill_wmma(*a, s["scale"], **kw)
        return s["pa"].paged_attention_prefill_varlen(*a, s["cu"], s["max_q"], s["scale"], **kw)
    ops = s["ops"]
    if c["kind"] == "decode":
        if f8 == 1.0:
            return ops.paged_attention_v3(*a, s["scale"], s["splits"])
        return ops.paged_attention_v3_scaled(*a, s["scale"], s["splits"], f8, f8)
    if c["kind"] == "prefill":
        if f8 == 1.0:
            return ops.paged_attention_prefill_wmma(*a, s["scale"])
        return ops.paged_attention_prefill_wmma_scaled(*a, s["scale"], f8, f8)
    if f8 == 1.0:
        return ops.paged_attention_prefill_varlen(*a, s["cu"], s["max_q"], s["scale"])
    return ops.paged_attention_prefill_varlen_scaled(*a, s["cu"], s["max_q"], s["scale"], f8, f8)


# ------------------------------------------------------------- work, exact --

def work(case):
    c = case
    if c["kind"] == "write":
        n = 2 * c["T"] * c["HKV"] * c["D"]
        return {"bytes": n * (SIZE[c["src"]] + SIZE[c["kv"]]) + 8 * c["T"], "flops": 0}
    lens, rows = _lens(c), _rows(c)
    row = 2 * c["HKV"] * c["D"] * SIZE[c["kv"]]
    heads = c["H"] * c["D"]
    # Row r of a sequence's n new rows attends ctx - n + r + 1 keys.
    seen = sum(n * (t - n) + n * (n + 1) // 2 for t, n in zip(lens, rows))
    io = sum(rows) * heads * (SIZE[c["q"]] + SIZE[c["out"]])
    tables = sum(-(-t // c["BS"]) for t in lens) * 4 + 4 * len(lens)
    return {"bytes": row * sum(lens) + io + tables, "flops": 4 * heads * seen}


def tolerance(case):
    # About four times the error measured against exact().
    if case["kind"] == "write":
        return "exact"  # bytes
    if case["kind"] == "prefill32" or (case["kind"] == "decode" and case["H"] == case["HKV"] and case["out"] == "f32"):
        return {"rel": 1e-5, "max": 1e-4}  # fp32 sums (measured 1e-7 to 4e-7)
    if case["out"] == "bf16":
        return {"rel": 7e-3, "max": 4e-2}  # the output's rounding (measured 1.7e-3)
    # fp16 outputs, or the weights' rounding to 16 bits in P.V on the matrix cores and in the packed dot
    # products of grouped fp16 and FP8 decode (measured 1.5e-4 to 2.1e-4).
    return {"rel": 1e-3, "max": 1e-2}


def exact(case, seed):
    c = case
    if c["kind"] == "write":
        return None  # whole bytes: compared exactly
    s = _inputs(c, seed)
    lens, rows, BS, HKV, D = _lens(c), _rows(c), c["BS"], c["HKV"], c["D"]
    G = c["H"] // HKV
    kvs = FP8_SCALE if c["kv"] == "fp8" else 1.0
    q = s["q"].reshape(-1, c["H"], D).double()
    out, at = torch.empty_like(q), 0
    for b, (t, n) in enumerate(zip(lens, rows)):
        pg = s["bt"][b, :-(-t // BS)].long()
        byte = torch.uint8 if c["kv"] == "fp8" else s["k"].dtype

        def seq(x):  # [HKV, t, D] in 64 bits
            y = x.view(byte)[pg].view(x.dtype).reshape(-1, HKV, D)[:t].double() * kvs
            return y.permute(1, 0, 2).contiguous()

        k, v = seq(s["k"]), seq(s["v"])
        key = torch.arange(t, device="cuda")
        for h in range(HKV):
            kt, vh = k[h].t().contiguous(), v[h]
            for r0 in range(0, n, 1024):
                m = min(1024, n - r0)
                qh = q[at + r0:at + r0 + m, h * G:(h + 1) * G].reshape(m * G, D)
                sc = (qh @ kt) / math.sqrt(D)
                pos = torch.arange(r0, r0 + m, device="cuda").repeat_interleave(G) + (t - n)
                sc.masked_fill_(key[None, :] > pos[:, None], float("-inf"))
                out[at + r0:at + r0 + m, h * G:(h + 1) * G] = (torch.softmax(sc, -1) @ vh).reshape(m, G, D)
        at += n
    return out.reshape(s["q"].shape)
