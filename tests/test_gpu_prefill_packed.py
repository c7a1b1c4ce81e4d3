"""The prefill kernels pack a GQA group's heads into the rows of a block (row R
is head R % G of chunk row R / G): odd groups whose rows cross the 32-, 64-,
128- and 256-row block edges, against the CPU oracle, in the 4-wave kernel's
two modes, the 8-wave kernel, a variable-length batch and the fp32-precision
kernel."""
import numpy as np
import pytest
import torch

import oracle
from _helpers import close, to_dev, to_host
from test_gpu_prefill import dev_args, prefill_case, want_of

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("G", [3, 7, 16])
@pytest.mark.parametrize("entry", ["paged_attention_prefill_wmma", "paged_attention_prefill"])
def test_packed_rows(pa, dev, G, entry):
    cus = torch.cuda.get_device_properties(dev).multi_processor_count
    wide = -(-cus // (2 * G))  # KV heads of a grid of at least two blocks per CU
    for HKV, B, S, ctx in ((2, 2, 65, [65, 150]), (1, 3, 1, [1, 40, 0]), (1, 2, 43, [64, 20]), (wide, 2, 130, [130, 131])):
        print("packed", G, entry, HKV, B, S, flush=True)
        inp = prefill_case(B, S, HKV * G, HKV, 32, 16, ctx, seed=G + S, kv="bf16", qt="bf16")
        close(to_host(getattr(pa, entry)(*dev_args(inp, dev), 0.2)), want_of(inp, 0.2))


@pytest.mark.parametrize("kv", ["f16", "bf16"])
def test_packed_rows_8_wave(pa, dev, kv):
    cus = torch.cuda.get_device_properties(dev).multi_processor_count
    G, HKV, S = 7, 3, 300
    B = -(-cus // (G * HKV))
    print("packed 8-wave", kv, B, flush=True)
    inp = prefill_case(B, S, HKV * G, HKV, 32, 16, [S + 3 * (i % 5) for i in range(B)], seed=3, kv=kv, qt=kv)
    got = to_host(pa.paged_attention_prefill_wmma(*dev_args(inp, dev), 0.2))
    assert pa.last_launch().startswith("pa::prefill_pp_kernel<"), pa.last_launch()
    close(got, want_of(inp, 0.2))


def test_packed_rows_varlen(pa, dev):
    """Row counts around the block edges of a group of 5, a bound on the row
    count beyond the batch's rows."""
    G, HKV, D = 5, 2, 64
    lens, ctx = [13, 1, 0, 26, 51, 64], [13, 30, 9, 90, 60, 64]
    inp = oracle.paged_inputs(len(lens), 1, HKV, D, 16, ctx, seed=8, kv_dtype="f16")
    q = np.random.default_rng(8).standard_normal((sum(lens), G * HKV, D), dtype=np.float32)
    cu = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    print("packed varlen", flush=True)
    got = to_host(pa.paged_attention_prefill_varlen(
        to_dev(q, "f32", dev), to_dev(inp["k"], "f16", dev), to_dev(inp["v"], "f16", dev),
        torch.from_numpy(inp["bt"]).to(dev), torch.from_numpy(inp["ctx"]).to(dev), torch.from_numpy(cu).to(dev),
        1 << 20, 0.125))
    for b, n in enumerate(lens):
        if n:
            want = oracle.prefill(q[None, cu[b]:cu[b + 1]], inp["k"], inp["v"], inp["bt"][b:b + 1], inp["ctx"][b:b + 1],
                                  0.125, "f16")[0]
            close(got[cu[b]:cu[b + 1]], want)


@pytest.mark.parametrize("HKV", [3, 8])
@pytest.mark.parametrize("rows,ctx", [(65, 70), (16, 1500)])
def test_packed_heads_turn(pa, dev, HKV, rows, ctx):
    """The order of a sequence's packed heads moves on with the sequence: every
    sequence and head is served once, in a uniform and a variable-length batch
    that wrap around the heads, also where contexts are split (16 rows)."""
    G, D, B = 4, 32, 11
    inp = prefill_case(B, rows, HKV * G, HKV, D, 16, [ctx + 3 * b for b in range(B)], seed=HKV + rows, kv="f16", qt="f16")
    want = want_of(inp, 0.2)
    args = dev_args(inp, dev)
    print("heads turn", HKV, rows, ctx, flush=True)
    close(to_host(pa.paged_attention_prefill_wmma(*args, 0.2)), want)
    close(to_host(pa.paged_attention_prefill(*args, 0.2)), want)
    cu = torch.arange(B + 1, dtype=torch.int32, device=dev) * rows
    q, *rest = args
    got = pa.paged_attention_prefill_varlen(q.reshape(B * rows, HKV * G, D), *rest, cu, rows, 0.2)
    close(to_host(got).reshape(want.shape), want)


@pytest.mark.parametrize("B,rows", [(1, 700), (3, 260), (66, 40), (130, 17)])
def test_packed_varlen_many_blocks(pa, dev, B, rows):
    """A variable-length batch of many packed blocks (up to 175 to a sequence) over
    one to three chunks of 64 sequences, empty and one-row ones between: every
    row once, as the prefill of its sequence alone."""
    HKV, G, D = 1, 16, 32
    lens = [[rows, rows - 1 - i % 7, 0, 1, 5][0 if i in (0, B - 1) else i % 5] for i in range(B)]
    ctx = [n + 3 * (i % 9) for i, n in enumerate(lens)]
    inp = oracle.paged_inputs(B, 1, HKV, D, 16, ctx, seed=B, kv_dtype="f16")
    q = oracle.quantize(np.random.default_rng(B).standard_normal((sum(lens), G * HKV, D), dtype=np.float32), "f16")
    cu = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    print("packed varlen blocks", B, rows, flush=True)
    got = to_host(pa.paged_attention_prefill_varlen(
        to_dev(q, "f16", dev), to_dev(inp["k"], "f16", dev), to_dev(inp["v"], "f16", dev),
        torch.from_numpy(inp["bt"]).to(dev), torch.from_numpy(inp["ctx"]).to(dev), torch.from_numpy(cu).to(dev),
        rows, 0.2))
    for b, n in enumerate(lens):
        if n:
            want = oracle.prefill(q[None, cu[b]:cu[b + 1]], inp["k"], inp["v"], inp["bt"][b:b + 1], inp["ctx"][b:b + 1],
                                  0.2, "f16")[0]
            close(got[cu[b]:cu[b + 1]], want)
