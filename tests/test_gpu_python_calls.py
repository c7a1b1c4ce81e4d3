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
