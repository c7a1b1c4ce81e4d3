"""The library's own decode plan where it replaces or refines a call's split,
against the CPU oracle: explicit counts it may replace (fewer planned, as many,
and more than asked for) where it is the faster, packed splits, and batches of nearly equal
contexts on the matrix-core kernel, which are not cut."""
import ctypes as C

import numpy as np
import pytest
import torch

from _helpers import close, decode_case, dev_inputs, oracle_decode_rows, to_host
from test_gpu_prefill32 import attention64, case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,H,HKV,D,ctx,S", [
    (1, 8, 1, 64, [8192], 16),             # the plan wants more partitions: held to 16
    (3, 8, 8, 128, [3000, 1, 0], 64),      # fewer than asked
    (2, 12, 4, 32, [700, 5000], 17),       # odd group, ragged
    (16, 16, 16, 128, [4096] * 16, 64),    # packed heads
    (16, 16, 16, 64, [4096] * 16, 64),
    (40, 8, 8, 32, [600] * 40, 8),         # uncut
])
@pytest.mark.parametrize("kv", ["f16", "bf16"])
def test_explicit_count_on_own_plan(pa, dev, B, H, HKV, D, ctx, S, kv):
    inp = decode_case(B, H, HKV, D, 16, ctx, seed=B + S, kv=kv, q=kv)
    q, k, v, bt, c = dev_inputs(inp, dev)
    print("own plan", B, H, HKV, D, S, kv, flush=True)
    got = to_host(pa.paged_attention_v3(q, k, v, bt, c, 0.1, S))
    close(got, oracle_decode_rows(inp["q_f32"], inp["k"], inp["v"], inp["bt"], inp["ctx"], 0.1, kv))
    # The explicit split's workspace is still asked for.
    need, V = pa.workspace_size(q, k, bt, S), pa.view
    out = torch.empty((B, H, D), device=dev)
    views = [V(t) for t in (out, q, k, v, bt, c)]
    rc = pa.lib().paged_attention_v3(*[C.byref(x) for x in views], 0.1, S, None, 0, None)
    assert need > 0 and rc == 3


@pytest.mark.parametrize("kv", ["f16", "bf16"])
@pytest.mark.parametrize("lens", ["equal", "nearly", "ragged", "empty and beyond", "one more"])
def test_equal_contexts_uncut(pa, dev, kv, lens):
    """A work-group per (sequence, KV head) or more fills the GPU, groups of
    eight: equal contexts run whole, others in partitions, by the same call; so
    do equal ones whose units leave a round of the GPU mostly empty.  Partitions
    write the workspace, whole contexts do not."""
    cus = torch.cuda.get_device_properties(dev).multi_processor_count
    HKV, G, D, B = 8, 8, 64, -(-cus // 8) + (lens == "one more")
    assert B <= 64
    n = np.full(B, 3008)
    if lens == "nearly":
        n -= np.arange(B) % 300
    elif lens == "ragged":
        n = np.random.default_rng(1).integers(1, 3009, B)
        n[3] = 3008
    elif lens == "empty and beyond":
        n[5], n[7] = 0, 17
    inp = decode_case(B, HKV * G, HKV, D, 16, n.tolist(), seed=3, kv=kv, q=kv, mb=188)
    q, k, v, bt, c = dev_inputs(inp, dev)
    ctx = inp["ctx"].copy()
    if lens == "empty and beyond":
        ctx[7] = 188 * 16 + 1
        c = torch.from_numpy(ctx).to(dev)
    print("uncut", lens, kv, flush=True)
    ws = torch.full((pa.workspace_size(q, k, bt, 0),), 0xA5, dtype=torch.uint8, device=dev)
    got = to_host(pa.paged_attention_v3(q, k, v, bt, c, 0.125, 0, workspace=ws))
    assert bool((ws == 0xA5).all()) == (lens in ("equal", "nearly", "empty and beyond"))
    assert "decode_mfma_kernel" in pa.last_launch() and "reduce_kernel" in pa.last_launch(), pa.last_launch()
    if lens == "empty and beyond":
        assert np.all(got[5] == 0.0) and np.isnan(got[7]).all()
        got[7] = 0.0
        ctx[7] = 0
    close(got, oracle_decode_rows(inp["q_f32"], inp["k"], inp["v"], inp["bt"], ctx, 0.125, kv))


@pytest.mark.parametrize("D", [32, 64, 128, 256])
@pytest.mark.parametrize("S", [0, 16])
def test_matrix_decode_q_range(pa, dev, D, S):
    """fp32 q beyond fp16's range, large and small elements mixed in a row,
    tiny and zero rows, over an fp16 cache with groups of eight.  Tolerance: q
    and the weights carry 22 bits each, and a score of up to 30 log2 units moves
    its weight by 30 * 2^-22 of itself: 1e-5."""
    ctx = [700, 1, 2049]
    q, k, v, bt, c, k32, v32 = case(3, 1, 16, 2, D, 16, ctx, "f16", "f32", D + S)
    q[0, 0, :8] *= 3e5
    q[0, 0, 8:, ::2] *= 1e6
    q[1, 0] *= 1e-30
    q[2, 0, 3] = 0.0
    q[2, 0, 4:9] *= 1e30
    print("q range", D, S, flush=True)
    for b, scale in ((0, 2e-7), (1, 0.1), (2, 2e-31)):
        one = slice(b, b + 1)
        got = to_host(pa.paged_attention_v3(q[one, 0].to(dev), k.to(dev), v.to(dev), torch.from_numpy(bt[one]).to(dev),
                                            torch.from_numpy(c[one]).to(dev), scale, S))
        assert "decode_mfma_kernel" in pa.last_launch(), pa.last_launch()
        want = attention64(q[one], k32, v32, bt[one], c[one], scale)[:, 0]
        err = float((torch.from_numpy(got).double() - want).norm() / want.norm())
        assert err < 1e-5, (b, err)


@pytest.mark.parametrize("kv", ["f16", "bf16"])
@pytest.mark.parametrize("S", [0, 1, 16])
def test_matrix_decode_non_finite_scores(pa, dev, kv, S):
    """A NaN or +Inf score makes its row NaN, as on the vector kernel, and so do
    scores that are all -Inf; -Inf among others is a weight of 0."""
    q, k, v, bt, c, k32, v32 = case(4, 1, 16, 2, 64, 16, [40, 40, 1, 700], kv, kv, 5)
    q[:, :, :, 2] = q[:, :, :, 2].abs() + 1  # (the sign of the scores below)
    for b, key, head, val in ((0, 7, 0, "nan"), (1, 30, 1, "inf"), (2, 0, 0, "-inf"), (3, 300, 1, "-inf")):
        page = int(bt[b, key // 16])
        k[page, key % 16, head, 2] = float(val)
        k32[page, key % 16, head, 2] = float(val)
    print("non-finite scores", kv, S, flush=True)
    got = to_host(pa.paged_attention_v3(q[:, 0].to(dev), k.to(dev), v.to(dev), torch.from_numpy(bt).to(dev),
                                        torch.from_numpy(c).to(dev), 0.125, S))
    assert "decode_mfma" in pa.last_launch(), pa.last_launch()
    want = attention64(q, k32, v32, bt, c, 0.125)[:, 0].float().numpy()
    assert np.isnan(want[0, :8]).all() and np.isnan(want[2, :8]).all() and np.isfinite(want[3]).all()
    close(got, want)
    assert np.array_equal(np.isnan(got), np.isnan(want))


@pytest.mark.parametrize("kv,qt", [("bf16", "f32"), ("bf16", "f16"), ("bf16", "bf16"), ("f16", "f32"), ("f16", "f16")])
@pytest.mark.parametrize("D", [32, 64, 128, 256])
def test_explicit_count_precision(pa, dev, kv, qt, D):
    """Explicit counts over groups of eight: fp32 weights (bf16 caches: three
    bf16 pieces; fp16: 22 bits).  Tolerance: N(0, 1) scores of up to 8 carry a
    rounding of 8 * 2^-24 (fp16 pieces 2^-22) and sums a few 2^-24: 1e-6."""
    ctx = [700, 1, 2049, 64]
    q, k, v, bt, c, k32, v32 = case(4, 1, 16, 2, D, 16, ctx, kv, qt, D)
    print("explicit precision", kv, qt, D, flush=True)
    got = to_host(pa.paged_attention_v3(q[:, 0].to(dev), k.to(dev), v.to(dev), torch.from_numpy(bt).to(dev),
                                        torch.from_numpy(c).to(dev), D ** -0.5, 64))
    assert ("decode_mfma32_kernel" if kv == "bf16" else "decode_mfma_kernel") in pa.last_launch(), pa.last_launch()
    want = attention64(q, k32, v32, bt, c, D ** -0.5)[:, 0]
    err = float((torch.from_numpy(got).double() - want).norm() / want.norm())
    print(f"error {err:.2e}", flush=True)
    assert err < 1e-6, err


@pytest.mark.parametrize("qt", ["f32", "bf16"])
def test_explicit_count_infinities(pa, dev, qt):
    """Inf in K and V over a bf16 cache reaches the outputs as a chain of fp32
    products carries it."""
    q, k, v, bt, c, k32, v32 = case(2, 1, 16, 2, 64, 16, [500, 40], "bf16", qt, 3)
    for x, x32, b, key, head, dim, val in ((v, v32, 0, 123, 0, 5, float("inf")), (v, v32, 0, 200, 1, 7, float("-inf")),
                                           (v, v32, 1, 3, 1, 9, float("inf")), (k, k32, 1, 11, 0, 2, float("inf"))):
        page = int(bt[b, key // 16])
        x[page, key % 16, head, dim] = val
        x32[page, key % 16, head, dim] = val
    print("infinities", qt, flush=True)
    got = to_host(pa.paged_attention_v3(q[:, 0].to(dev), k.to(dev), v.to(dev), torch.from_numpy(bt).to(dev),
                                        torch.from_numpy(c).to(dev), 0.125, 64))
    want = attention64(q, k32, v32, bt, c, 0.125)[:, 0].float().numpy()
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isinf(got), np.isinf(want))
    assert np.array_equal(got[np.isinf(got)], want[np.isinf(want)])
    fine = np.isfinite(want)
    close(got[fine], want[fine])


@pytest.mark.parametrize("B,H,HKV,D,ctx,packed", [
    (32, 16, 16, 128, 4096, 4), (16, 16, 16, 128, 8192, 8),   # four work-groups of two heads per CU
    (16, 16, 16, 128, 2048, 0), (32, 12, 12, 64, 8192, 0), (32, 32, 8, 128, 4096, 0), (24, 16, 16, 128, 8192, 0)])
def test_packed_split_rule(pa, dev, B, H, HKV, D, ctx, packed):
    """Which splits take the partitions of packed heads (a share of 256 CUs each,
    evenly); the others are pa_plan_partitions'.  Sizes only: nothing is launched."""
    cus = torch.cuda.get_device_properties(dev).multi_processor_count
    if cus != 256:
        pytest.skip("sizes chosen for 256 CUs")
    ptr, MB = torch.empty(64, device=dev).data_ptr(), ctx // 16
    T = type(pa.view(torch.empty(1)))
    q = T.make(ptr, 1, (B, H, D), (H * D, D, 1))
    k = T.make(ptr, 1, (B * MB, 16, HKV, D), (16 * HKV * D, HKV * D, D, 1))
    bt = T.make(ptr, 4, (B, MB), (MB, 1))
    size = pa.lib().paged_attention_v3_workspace_size(C.byref(q), C.byref(k), C.byref(bt), 0)
    tok, n = C.c_int64(), C.c_int64()
    pa.check(pa.lib().pa_plan_partitions(B, H, HKV, D, ctx, cus, C.byref(tok), C.byref(n)))
    parts = packed or n.value
    rows = B * H * parts
    up = lambda x: (x + 255) // 256 * 256
    assert size == up(rows * D * 4) + 2 * up(rows * 4), (size / (B * H * (D + 2) * 4), parts)


@pytest.mark.parametrize("kv,B,H,HKV,D,ctx,S,own", [
    ("f16", 1, 12, 12, 64, 2048, 64, True),     # a few units
    ("f16", 16, 12, 12, 64, 2048, 64, False),   # nearly a full GPU
    ("f16", 64, 12, 12, 64, 512, 16, False),    # (16 partitions: half of a work-group's slots)
    ("f16", 64, 12, 12, 64, 512, 64, True),     # rounds of slots, uncut
    ("f16", 64, 12, 12, 64, 4096, 64, False),   # more pages than a work-group stages
    ("f16", 4, 16, 16, 128, 512, 32, False),    # uncut, but a few units
    ("f16", 32, 32, 8, 128, 1024, 32, True),    # groups of four that fill the GPU
    ("f16", 32, 32, 8, 128, 2048, 16, False),   # chunks of 128 tokens
    ("fp8", 8, 64, 8, 128, 1024, 32, False),    # groups of eight on the vector kernel
    ("bf16", 8, 64, 8, 128, 1024, 32, True)])   # and on the matrix cores
def test_explicit_count_route(pa, dev, kv, B, H, HKV, D, ctx, S, own):
    """Which explicit counts run the library's plan: the caller's own partitions
    write their partial sums to the end of the workspace.  Both are the attention
    of the same rows."""
    if torch.cuda.get_device_properties(dev).multi_processor_count != 256:
        pytest.skip("sizes chosen for 256 CUs")
    MB = ctx // 16
    g = torch.Generator(device=dev).manual_seed(1)
    dt = {"f16": torch.float16, "bf16": torch.bfloat16, "fp8": torch.float8_e4m3fn}[kv]
    q = torch.randn((B, H, D), device=dev, generator=g).half() if kv != "bf16" else torch.randn(
        (B, H, D), device=dev, generator=g).bfloat16()
    k, v = (torch.randn((B * MB, 16, HKV, D), device=dev, generator=g).half().to(dt) for _ in range(2))
    bt = torch.randperm(B * MB, device=dev, generator=g).int().view(B, MB)
    c = torch.full((B,), ctx, dtype=torch.int32, device=dev)
    need = pa.workspace_size(q, k, bt, S)
    ws = torch.full((need,), 0xA5, dtype=torch.uint8, device=dev)
    rows = B * H * S
    last = (rows * D * 4 + 255) // 256 * 256 + (rows * 4 + 255) // 256 * 256 + rows * 4 - 4
    print("route", kv, B, H, HKV, D, ctx, S, flush=True)
    got = pa.paged_attention_v3(q, k, v, bt, c, 0.1, S, workspace=ws)
    assert bool((ws[last:last + 4] == 0xA5).all()) == own, pa.last_launch()
    want = torch.empty_like(got)
    V = [pa.view(t) for t in (want, q, k, v, bt, c)]
    st = torch.cuda.current_stream().cuda_stream
    pa.check(pa.lib().pa_v3_partition(*[C.byref(x) for x in V], 0.1, S, ws.data_ptr(), need, st))
    pa.check(pa.lib().pa_v3_reduce(*[C.byref(V[i]) for i in (0, 1, 2, 4, 5)], S, ws.data_ptr(), need, st))
    close(to_host(got), to_host(want))
