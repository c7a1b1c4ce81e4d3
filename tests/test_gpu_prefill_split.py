"""Context split of the prefill (paged_attention_prefill_split, which the
Python functions and the torch operators call): partitions of whole key tiles
merged by a second launch, against the CPU oracle, at contexts around the
partition and tile edges, in the 16-bit-weight, variable-length and
fp32-precision kernels; poisoned and padded rows; the workspace checks."""
import ctypes as C

import numpy as np
import pytest
import torch

import oracle
from _helpers import close, to_dev, to_host
from test_gpu_prefill import dev_args, prefill_case, want_of

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D", [32, 64, 128, 256])
@pytest.mark.parametrize("kv,qt", [("f16", "f32"), ("bf16", "bf16")])
@pytest.mark.parametrize("entry", ["paged_attention_prefill_wmma", "paged_attention_prefill"])
def test_prefill_split(pa, dev, D, kv, qt, entry):
    """Contexts of one partition, of its edges and of many; a chunk longer than
    its context (rows before it) and an empty one, in one batch."""
    if D == 256 and entry == "paged_attention_prefill":
        pytest.skip("the fp32-precision matrix kernel is off at D = 256: wrong rows and a memory fault, cause not found")
    for S, BS, ctx in ((70, 16, [1537, 1024, 1023, 300, 64, 40, 0]), (65, 5, [2500])):
        print("split", D, kv, entry, S, flush=True)
        # (Groups over fp16 caches run the fp32-precision form on the decode kernel.)
        HKV = 2 if kv == "f16" and entry == "paged_attention_prefill" else 1
        inp = prefill_case(len(ctx), S, 2, HKV, D, BS, ctx, seed=D + S, kv=kv, qt=qt)
        got = to_host(getattr(pa, entry)(*dev_args(inp, dev), 0.2))
        assert "prefill_reduce_kernel" in pa.last_launch(), pa.last_launch()
        close(got, want_of(inp, 0.2))


def test_prefill_split_fp8_and_poison(pa, dev):
    """An invalid block id reaches the rows that read its page whichever
    partition holds it; a context beyond the table poisons its sequence."""
    from test_gpu_prefill import _fp8, fp8_prefill_case
    B, S, H, D, ctx = 3, 40, 2, 64, [2000, 1500, 1990]
    inp, k8, v8, kf, vf = fp8_prefill_case(B, S, H, 2, D, 16, ctx, seed=4, qt="bf16", k_scale=0.05, v_scale=0.02)
    bt, c = inp["bt"].copy(), inp["ctx"].copy()
    bt[1, 92] = -3   # keys 1472..1487: rows from 1472 - 1460 on
    bt[2, 0] = 10 ** 6
    c[0] = bt.shape[1] * 16 + 1
    print("split fp8 poison", flush=True)
    got = to_host(pa.paged_attention_prefill_wmma(
        to_dev(inp["q"], "bf16", dev), _fp8(k8, dev), _fp8(v8, dev), torch.from_numpy(bt).to(dev),
        torch.from_numpy(c).to(dev), 0.125, k_scale=0.05, v_scale=0.02))
    assert "prefill_reduce_kernel" in pa.last_launch(), pa.last_launch()
    want = oracle.prefill(inp["q_f32"], kf, vf, inp["bt"], inp["ctx"], 0.125, "f32")
    assert np.isnan(got[0]).all() and np.isnan(got[2]).all() and np.isnan(got[1, 12:]).all()
    close(got[1, :12], want[1, :12])


def test_varlen_split(pa, dev):
    G, HKV, D = 3, 2, 64
    lens, ctx = [13, 1, 0, 26, 70, 1], [1300, 30, 9, 2400, 900, 2000]
    inp = oracle.paged_inputs(len(lens), 1, HKV, D, 16, ctx, seed=8, kv_dtype="bf16")
    q = np.random.default_rng(8).standard_normal((sum(lens), G * HKV, D), dtype=np.float32)
    cu = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    print("split varlen", flush=True)
    got = to_host(pa.paged_attention_prefill_varlen(
        to_dev(q, "f32", dev), to_dev(inp["k"], "bf16", dev), to_dev(inp["v"], "bf16", dev),
        torch.from_numpy(inp["bt"]).to(dev), torch.from_numpy(inp["ctx"]).to(dev), torch.from_numpy(cu).to(dev),
        70, 0.125))
    # The one-row sequences split too: decode partitions, their merge, prefill partitions, theirs.
    assert "; pa::reduce_kernel<64>; " in pa.last_launch() and "prefill_reduce_kernel" in pa.last_launch()
    for b, n in enumerate(lens):
        if n:
            want = oracle.prefill(q[None, cu[b]:cu[b + 1]], inp["k"], inp["v"], inp["bt"][b:b + 1], inp["ctx"][b:b + 1],
                                  0.125, "bf16")[0]
            close(got[cu[b]:cu[b + 1]], want)


def test_prefill_split_workspace_checks(pa, dev):
    """A missing or short workspace is refused before any launch; without a
    split the size is 0 and none is needed."""
    L = pa.lib()
    inp = prefill_case(1, 70, 2, 1, 64, 16, [2048], seed=1, kv="f16", qt="f16")
    q, k, v, bt, c = dev_args(inp, dev)
    out = torch.full(q.shape, 7.0, device=dev)
    V = [pa.view(t) for t in (out, q, k, v, bt, c)]
    need = L.paged_attention_prefill_workspace_size(C.byref(V[1]), C.byref(V[2]), C.byref(V[4]), 0)
    assert need > 0 and need % 16 == 0
    for ws, n in ((None, 0), (torch.empty(need, dtype=torch.uint8, device=dev), need - 1)):
        rc = L.paged_attention_prefill_split(*[C.byref(x) for x in V], None, 0, 0.125, 1.0, 1.0, 0,
                                             ws.data_ptr() if ws is not None else None, n, None)
        assert rc == 3, rc
    torch.cuda.synchronize()
    assert bool((out == 7.0).all())
    short = prefill_case(1, 70, 2, 1, 64, 16, [100], seed=1, kv="f16", qt="f16")
    v3 = [pa.view(t) for t in dev_args(short, dev)]
    assert L.paged_attention_prefill_workspace_size(C.byref(v3[0]), C.byref(v3[1]), C.byref(v3[3]), 0) == 0


def test_varlen_split_overlapping_ranges(pa, dev):
    """Ranges that overlap (each in itself well formed) number more blocks than
    the workspace and the grid are sized for: what does not fit is not served,
    and nothing beyond the workspace is written.  Sequences 0 and 2 are the same
    rows, keys and values, so the rows that are served have one result."""
    L, H, D, S, n = pa.lib(), 12, 64, 512, 2048
    inp = oracle.paged_inputs(1, 1, H, D, 16, [n], seed=12, kv_dtype="f16")
    q = np.random.default_rng(12).standard_normal((S, H, D), dtype=np.float32)
    dq = to_dev(q, "f32", dev)
    t = [torch.full((S, H, D), 7.0, device=dev), dq, to_dev(inp["k"], "f16", dev), to_dev(inp["v"], "f16", dev),
         torch.from_numpy(np.repeat(inp["bt"], 3, 0)).to(dev), torch.full((3,), n, dtype=torch.int32, device=dev),
         torch.tensor([0, S, 0, S], dtype=torch.int32, device=dev)]
    V = [pa.view(x) for x in t]
    need = L.paged_attention_prefill_workspace_size(C.byref(V[1]), C.byref(V[2]), C.byref(V[4]), S)
    assert need > 0
    guard = 1 << 20
    ws = torch.full((need + 2 * guard,), 0xA5, dtype=torch.uint8, device=dev)
    print("overlapping ranges", flush=True)
    pa.check(L.paged_attention_prefill_split(*[C.byref(x) for x in V], S, 0.125, 1.0, 1.0, 0, ws.data_ptr() + guard,
                                             need, torch.cuda.current_stream().cuda_stream))
    assert "prefill_reduce_kernel" in pa.last_launch(), pa.last_launch()
    assert bool((ws[:guard] == 0xA5).all()) and bool((ws[guard + need:] == 0xA5).all())
    got = to_host(t[0])
    # 132 units of 64 rows and a head: blocks 7 .. 3 of both sequences, block 2 of one.
    want = oracle.prefill(q[None], inp["k"], inp["v"], inp["bt"], inp["ctx"], 0.125, "f16")[0]
    close(got[128:], want[128:])
    assert np.all(got[:128] == 7.0)


@pytest.mark.parametrize("npf,mb,split", [(6, 64, False), (6, 128, True), (2, 64, True)])
def test_varlen_split_rule(pa, dev, npf, mb, split):
    """A variable-length batch whose partitions outnumber the CUs splits only from
    longer contexts on; every sequence against the oracle."""
    HKV, G, D, S = 2, 4, 128, 128
    lens = [1] * 4 + [S] * npf
    ctx = [33, 7, 64, 1] + [mb * 16 - 5 * i for i in range(npf)]
    inp = oracle.paged_inputs(len(lens), 1, HKV, D, 16, ctx, seed=9, kv_dtype="f16")
    q = oracle.quantize(np.random.default_rng(9).standard_normal((sum(lens), G * HKV, D), dtype=np.float32), "f16")
    cu = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    print("varlen split rule", npf, mb, flush=True)
    got = to_host(pa.paged_attention_prefill_varlen(
        to_dev(q, "f16", dev), to_dev(inp["k"], "f16", dev), to_dev(inp["v"], "f16", dev),
        torch.from_numpy(inp["bt"]).to(dev), torch.from_numpy(inp["ctx"]).to(dev), torch.from_numpy(cu).to(dev), S, 0.1))
    assert ("prefill_reduce_kernel" in pa.last_launch()) == split, pa.last_launch()
    for b in range(len(lens)):
        close(got[cu[b]:cu[b + 1]], oracle.prefill(q[None, cu[b]:cu[b + 1]], inp["k"], inp["v"], inp["bt"][b:b + 1],
                                                   inp["ctx"][b:b + 1], 0.1, "f16")[0])


@pytest.mark.parametrize("lens,cut", [([70], False), ([70, 69], False), ([70, 1], True), ([70, 1, 0], True)])
def test_varlen_decode_rows_possible(pa, dev, lens, cut):
    """The decode rows' split is planned only where the batch's row count leaves a
    sequence with one row; every sequence against the oracle."""
    HKV, G, D = 2, 2, 64
    ctx = [3000 - 7 * i if n else 5 for i, n in enumerate(lens)]
    inp = oracle.paged_inputs(len(lens), 1, HKV, D, 16, ctx, seed=4, kv_dtype="f16")
    q = oracle.quantize(np.random.default_rng(4).standard_normal((sum(lens), G * HKV, D), dtype=np.float32), "f16")
    cu = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    print("decode rows possible", lens, flush=True)
    got = to_host(pa.paged_attention_prefill_varlen(
        to_dev(q, "f16", dev), to_dev(inp["k"], "f16", dev), to_dev(inp["v"], "f16", dev),
        torch.from_numpy(inp["bt"]).to(dev), torch.from_numpy(inp["ctx"]).to(dev), torch.from_numpy(cu).to(dev), 70, 0.1))
    assert ("pa::reduce_kernel" in pa.last_launch()) == cut, pa.last_launch()
    for b, n in enumerate(lens):
        if n:
            close(got[cu[b]:cu[b + 1]], oracle.prefill(q[None, cu[b]:cu[b + 1]], inp["k"], inp["v"], inp["bt"][b:b + 1],
                                                       inp["ctx"][b:b + 1], 0.1, "f16")[0])
