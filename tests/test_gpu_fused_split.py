"""GPU parity of explicit splits into short partitions over grids that fill the
GPU, one query head per KV head: such a paged_attention_v3 call runs as ONE
kernel launch, over whole contexts (the library's own plan; the merge rule makes
any partitions one softmax, kernels/paged_attn_v3.cu:128-166), and leaves the
workspace alone.  The caller's own partitions of the same inputs run through
pa_v3_partition + pa_v3_reduce (kernels/paged_attn_v3.cu:33-123) beside it.

Checked against the oracle: the output (the parity tolerance), equal scores
(K = 0), a bad block id poisoning only its row, a scaled FP8 cache, the
workspace left untouched, and the two-launch path on the same inputs.
"""
import ctypes as C

import numpy as np
import pytest
import torch

import oracle
from _helpers import ATOL32, RTOL32, close, decode_case, dev_inputs, to_host

pytestmark = pytest.mark.gpu


def two_launch(pa, out, q, k, v, bt, ctx, scale, S, ws):
    V = pa.view
    st = torch.cuda.current_stream().cuda_stream
    pa.check(pa.lib().pa_v3_partition(C.byref(V(out)), C.byref(V(q)), C.byref(V(k)), C.byref(V(v)),
                                      C.byref(V(bt)), C.byref(V(ctx)), scale, S, ws.data_ptr(), ws.numel(), st))
    pa.check(pa.lib().pa_v3_reduce(C.byref(V(out)), C.byref(V(q)), C.byref(V(k)), C.byref(V(bt)),
                                   C.byref(V(ctx)), S, ws.data_ptr(), ws.numel(), st))


def grid_rows(dev, H, lo=1):
    cus = torch.cuda.get_device_properties(dev).multi_processor_count
    return -(-cus * lo // H)


CASES = [  # kv, D, BS, MB, S
    ("f16", 64, 16, 64, 64),    # 16-token partitions, one page each
    ("f16", 64, 16, 64, 40),    # 26-token partitions
    ("bf16", 128, 16, 32, 24),  # 22-token partitions
    ("f32", 64, 8, 64, 48),     # 11-token partitions
    ("f16", 256, 32, 16, 64),   # 8-token partitions, a quarter of a page
    ("f16", 32, 16, 32, 64),    # two heads packed per work-group (64-byte rows)
    ("bf16", 64, 1, 64, 64),    # one token per page and per partition
    ("f16", 64, 5, 50, 33),     # page size not a multiple of the token slots
]


@pytest.mark.parametrize("kv,D,BS,MB,S", CASES)
def test_fused_split_matches_oracle(pa, dev, kv, D, BS, MB, S):
    """Ragged contexts (empty, one token, the whole table, beyond the table,
    random) in one launch, against the oracle and the caller's partitions
    in two launches on the same inputs."""
    H = 8
    kvb = {"f16": 2, "bf16": 2, "f32": 4}[kv]
    lo = 2 if D * kvb < 128 else 1
    B = grid_rows(dev, H, lo)
    maxctx = MB * BS
    rng = np.random.default_rng(D * 131 + S)
    ctx = rng.integers(1, maxctx + 1, size=B).astype(np.int32)
    ctx[:4] = [0, 1, maxctx, maxctx - 1]
    inp = decode_case(B, H, H, D, BS, ctx.tolist(), seed=70 + S, kv=kv, q=kv, mb=MB)
    q, k, v, bt, _ = dev_inputs(inp, dev)
    ctx_run = inp["ctx"].copy()
    ctx_run[4] = maxctx + 1  # beyond the table: NaN row
    cd = torch.from_numpy(ctx_run).to(dev)
    got = to_host(pa.paged_attention_v3(q, k, v, bt, cd, 0.125, S))
    launched = pa.last_launch()
    assert "reduce_kernel" not in launched and launched.count("decode_kernel") == 1, launched
    assert np.all(got[0] == 0.0)
    assert np.all(np.isnan(got[4]))
    want = oracle.decode(inp["q_f32"], inp["k"], inp["v"], inp["bt"], ctx_run, 0.125, kv)
    tol = dict(atol=ATOL32, rtol=RTOL32) if kv == "f32" else {}
    live = np.ones(B, bool)
    live[[0, 4]] = False
    close(got[live], want[live], **tol)
    # The two-launch split over the same partitions.
    ws = torch.zeros(pa.workspace_size(q, k, bt, S), dtype=torch.uint8, device=dev)
    out2 = torch.empty((B, H, D), dtype=torch.float32, device=dev)
    two_launch(pa, out2, q, k, v, bt, cd, 0.125, S, ws)
    torch.cuda.synchronize()
    close(got[live], to_host(out2)[live], **tol)


@pytest.mark.parametrize("S", [16, 33, 64])
def test_fused_split_equal_scores(pa, dev, S):
    """With K = 0 every score is 0, every partition's maximum the same: the
    output is the plain mean of V over each row's context, uncut and over the
    caller's partitions (empty ones included: ctx 1, 2, 7 leave most of the
    16-64 empty).  The one launch leaves the workspace (filled with 0xFF) alone."""
    H, D, BS, MB = 8, 64, 16, 64
    B = grid_rows(dev, H)
    maxctx = MB * BS
    rng = np.random.default_rng(S)
    ctx = rng.integers(1, maxctx + 1, size=B).astype(np.int32)
    ctx[:5] = [1, 2, 7, S + 1, maxctx]
    inp = decode_case(B, H, H, D, BS, ctx.tolist(), seed=5, kv="f32", q="f32", mb=MB)
    q, _, v, bt, cd = dev_inputs(inp, dev)
    k = torch.zeros_like(v)
    need = pa.workspace_size(q, k, bt, S)
    ws = torch.full((need,), 0xFF, dtype=torch.uint8, device=dev)
    got = to_host(pa.paged_attention_v3(q, k, v, bt, cd, 1.0, S, workspace=ws))
    assert "reduce_kernel" not in pa.last_launch(), pa.last_launch()
    assert bool((ws == 0xFF).all())
    want = oracle.decode(inp["q_f32"], np.zeros_like(inp["k"]), inp["v"], inp["bt"], inp["ctx"], 1.0, "f32")
    close(got, want, atol=ATOL32, rtol=RTOL32)
    out2 = torch.empty((B, H, D), dtype=torch.float32, device=dev)
    two_launch(pa, out2, q, k, v, bt, cd, 1.0, S, ws)
    close(to_host(out2), want, atol=ATOL32, rtol=RTOL32)


def test_fused_split_bad_block_id(pa, dev):
    """A block id outside the pool in one sequence's table: that row is NaN
    (every head) and every other row matches the oracle, uncut and over the
    caller's partitions."""
    H, D, BS, MB, S = 8, 64, 16, 64, 64
    B = grid_rows(dev, H)
    maxctx = MB * BS
    inp = decode_case(B, H, H, D, BS, [maxctx] * B, seed=9, kv="f16", q="f16", mb=MB)
    q, k, v, _, cd = dev_inputs(inp, dev)
    bt_h = inp["bt"].copy()
    nb = inp["k"].shape[0]
    bt_h[3, 10] = nb + 5  # page 10 = tokens 160..175: partition 10 of 16-token partitions
    bt = torch.from_numpy(bt_h).to(dev)
    got = to_host(pa.paged_attention_v3(q, k, v, bt, cd, 0.125, S))
    assert "reduce_kernel" not in pa.last_launch(), pa.last_launch()
    assert np.all(np.isnan(got[3]))
    keep = np.arange(B) != 3
    want = oracle.decode(inp["q_f32"][keep], inp["k"], inp["v"], inp["bt"][keep], inp["ctx"][keep], 0.125, "f16")
    close(got[keep], want)
    ws = torch.zeros(pa.workspace_size(q, k, bt, S), dtype=torch.uint8, device=dev)
    out2 = torch.empty((B, H, D), dtype=torch.float32, device=dev)
    two_launch(pa, out2, q, k, v, bt, cd, 0.125, S, ws)
    got = to_host(out2)
    assert np.all(np.isnan(got[3]))
    close(got[keep], want)


@pytest.mark.parametrize("D", [64, 128])
def test_fused_split_fp8_scaled(pa, dev, D):
    """An FP8 E4M3 cache with per-tensor scales (k_scale folded into the
    softmax scale, v_scale applied to the merged output) in one launch, against
    the oracle on the dequantised cache, against a split that runs as two
    launches, and (k_scale joined to the scale by the caller) against the
    caller's 64 partitions."""
    from test_gpu_decode import fp8_case, fp8_dev
    H, BS, MB = 8, 16, 32
    lo = 2 if D < 128 else 1
    B = grid_rows(dev, H, lo)
    maxctx = MB * BS
    rng = np.random.default_rng(D)
    ctx = rng.integers(1, maxctx + 1, size=B).astype(np.int32)
    ctx[:3] = [1, maxctx, 2]
    inp, k8, v8, kf, vf = fp8_case(B, H, H, D, BS, ctx.tolist(), seed=D + 3, k_scale=0.05, v_scale=0.02)
    bt = torch.from_numpy(inp["bt"]).to(dev)
    cd = torch.from_numpy(inp["ctx"]).to(dev)
    q = torch.from_numpy(inp["q_f32"]).to(dev).half()
    k, v = fp8_dev(k8, dev), fp8_dev(v8, dev)
    S = 64
    got = to_host(pa.paged_attention_v3(q, k, v, bt, cd, 0.1, S, k_scale=0.05, v_scale=0.02))
    assert "reduce_kernel" not in pa.last_launch(), pa.last_launch()
    q32 = oracle.to_float(oracle.quantize(inp["q_f32"], "f16"), "f16")
    close(got, oracle.decode(q32, kf, vf, inp["bt"], inp["ctx"], 0.1, "f32"))
    # Beside it, a split of five partitions (the caller's: two launches).
    got5 = to_host(pa.paged_attention_v3(q, k, v, bt, cd, 0.1, 5, k_scale=0.05, v_scale=0.02))
    assert "reduce_kernel" in pa.last_launch(), pa.last_launch()
    close(got, got5)
    ws = torch.zeros(pa.workspace_size(q, k, bt, S), dtype=torch.uint8, device=dev)
    out2 = torch.empty((B, H, D), dtype=torch.float32, device=dev)
    two_launch(pa, out2, q, k, v, bt, cd, 0.1 * 0.05, S, ws)
    close(got, 0.02 * to_host(out2))


def test_small_grid_keeps_two_launches(pa, dev):
    """A grid of one work-group per (row, head) that would not fill the GPU
    keeps the partition kernel and the reduce (both launched by one call)."""
    H, D, BS, MB, S = 8, 64, 16, 64, 64
    B = 2
    inp = decode_case(B, H, H, D, BS, [MB * BS, 300], seed=11, kv="f16", q="f16", mb=MB)
    q, k, v, bt, cd = dev_inputs(inp, dev)
    got = to_host(pa.paged_attention_v3(q, k, v, bt, cd, 0.125, S))
    assert "reduce_kernel" in pa.last_launch(), pa.last_launch()
    close(got, oracle.decode(inp["q_f32"], inp["k"], inp["v"], inp["bt"], inp["ctx"], 0.125, "f16"))
