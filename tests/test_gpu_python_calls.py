"""The Python functions' native calls: results and output types as the
torch operators', what they convert and refuse, and eager execution inside a
torch.compile'd function."""
import pytest
import torch

from _helpers import decode_case, dev_inputs
from test_gpu_prefill import dev_args, prefill_case

pytestmark = pytest.mark.gpu


def test_python_calls_equal_operators(pa, dev):
    ops = pa.torch_ops()
    q, k, v, bt, c = dev_inputs(decode_case(3, 8, 2, 64, 16, [2000, 1, 700], seed=2, kv="bf16", q="bf16"), dev)
    print("python calls", flush=True)
    want = ops.paged_attention_v3(q, k, v, bt, c, 0.1, 0)
    for wide in (bt.long(), bt):
        assert torch.equal(pa.paged_attention_v3(q, k, v, wide, c.long(), 0.1, 0), want)
    out = torch.empty_like(q)
    ws = torch.empty(pa.workspace_size(q, k, bt, 0), dtype=torch.uint8, device=dev)
    assert pa.paged_attention_v3(q, k, v, bt, c, 0.1, 0, out=out, workspace=ws) is out
    assert torch.equal(out, want.bfloat16())
    assert torch.equal(pa.paged_attention_v3(q, k, v, bt, c, 0.1, 0, workspace=ws[:256]), want)  # too small: its own
    strided = torch.empty((3, 64, 8), dtype=q.dtype, device=dev).transpose(1, 2).copy_(q)
    assert torch.equal(pa.paged_attention_v3(strided, k, v, bt, c, 0.1, 0), want)
    for f, g in ((pa.paged_attention, ops.paged_attention), (pa.paged_attention_v2, ops.paged_attention_v2)):
        assert torch.equal(f(q, k, v, bt, c, 0.1, out_dtype=torch.float16), g(q, k, v, bt, c, 0.1).half())
    a = dev_args(prefill_case(2, 70, 4, 2, 64, 16, [70, 1100], seed=1, kv="f16", qt="f16"), dev)
    assert torch.equal(pa.paged_attention_prefill_wmma(*a, 0.2), ops.paged_attention_prefill_wmma(*a, 0.2))
    assert torch.equal(pa.paged_attention_prefill(*a, 0.2), ops.paged_attention_prefill(*a, 0.2))


def test_python_calls_refuse(pa, dev):
    q, k, v, bt, c = dev_inputs(decode_case(2, 4, 2, 64, 16, [20, 30], seed=2, kv="f16", q="f16"), dev)
    print("refusals", flush=True)
    with pytest.raises(RuntimeError, match="q must be on CUDA"):
        pa.paged_attention(q.cpu(), k, v, bt, c, 0.1)
    with pytest.raises(RuntimeError, match="kv cache must be on CUDA"):
        pa.paged_attention_v3(q, k.cpu(), v, bt, c, 0.1, 0)
    with pytest.raises(RuntimeError, match=r"q must be \[B, H, D\]"):
        pa.paged_attention_v2(q[0], k, v, bt, c, 0.1)
    with pytest.raises(RuntimeError, match="n_head must be divisible by n_kv_head"):
        pa.paged_attention_v3(q[:, :3].contiguous(), k, v, bt, c, 0.1, 0)
    with pytest.raises(RuntimeError, match="out must have the shape of q"):
        pa.paged_attention(q, k, v, bt, c, 0.1, out=torch.empty((2, 4, 32), device=dev))
    with pytest.raises(RuntimeError, match="max_q_len must be non-negative"):
        pa.paged_attention_prefill_varlen(q, k, v, bt, c, torch.tensor([0, 1, 2], device=dev), -1, 0.1)


def test_python_calls_inside_compile(pa, dev):
    """The call ends the compiled graph and runs eagerly; q that requires grad is accepted."""
    q, k, v, bt, c = dev_inputs(decode_case(2, 4, 2, 64, 16, [20, 30], seed=2, kv="f16", q="f16"), dev)
    print("compile", flush=True)

    def layer(x):
        return pa.paged_attention_v3(x * 2, k, v, bt, c, 0.1, 0) + 1

    want = layer(q)
    assert torch.equal(torch.compile(layer, backend="eager")(q), want)
    assert torch.equal(layer(q.clone().requires_grad_()).detach(), want)


def test_python_calls_without_operator_library(pa, dev, monkeypatch, tmp_path):
    """With libpagedattn.so alone the functions give the same results."""
    import sys
    ops = sys.modules[pa.paged_attention.__module__]
    q, k, v, bt, c = dev_inputs(decode_case(3, 8, 2, 64, 16, [2000, 1, 700], seed=2, kv="bf16", q="bf16"), dev)
    a = dev_args(prefill_case(2, 70, 4, 2, 64, 16, [70, 1100], seed=1, kv="f16", qt="f16"), dev)
    cu = torch.tensor([0, 70, 140], device=dev)
    k8 = torch.randn((5, 16, 2, 64), device=dev).to(torch.float8_e4m3fn)
    key = torch.randn((7, 2, 64), device=dev)

    def calls():
        kc, vc = torch.zeros_like(k8), torch.zeros_like(k8)
        pa.write_kv(kc, vc, key, key.flip(0), torch.arange(7, device=dev) * 3, 0.5, 0.25)
        return [pa.paged_attention(q, k, v, bt, c, 0.1), pa.paged_attention_v2(q, k, v, bt, c, 0.1),
                pa.paged_attention_v3(q, k, v, bt.long(), c.long(), 0.1, 0, out_dtype=torch.bfloat16),
                pa.paged_attention_v3(q, k, v, bt, c, 0.1, 5, k_scale=0.5, v_scale=2.0),
                pa.paged_attention_prefill_wmma(*a, 0.2), pa.paged_attention_prefill(*a, 0.2),
                pa.paged_attention_prefill_varlen(a[0].reshape(140, 4, 64), *a[1:], cu, 70, 0.2),
                kc.view(torch.uint8), vc.view(torch.uint8)]

    print("without the operator library", flush=True)
    want = calls()
    monkeypatch.setattr(ops, "_ops", None)
    monkeypatch.setattr(ops, "_torch_path", lambda: tmp_path / "none.so")
    assert ops._native() is ops._CAbi
    for x, y in zip(calls(), want):
        assert x.dtype == y.dtype and torch.equal(x, y)
    with pytest.raises(RuntimeError, match=r"q must be \[B, H, D\]"):
        pa.paged_attention_v2(q[0], k, v, bt, c, 0.1)
