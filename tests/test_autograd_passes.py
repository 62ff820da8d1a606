"""How often the attention ops run in a derivative: on the GPU a node that gets no cotangent launches nothing. The CPU
cases take the GPU's rule over the dense path; the GPU cases run under the rule itself, on the Python nodes (a mode counts
their ops) and on the native ones (a profiler counts their ranges)."""

import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode

from ebr_amd.fused_attn import fused_attention, ops


class _Count(TorchDispatchMode):
    def __init__(self):
        super().__init__()
        self.calls = []

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        if func.namespace == "ebr_fused":
            self.calls.append(func.__name__.split(".")[0])
        return func(*args, **(kwargs or {}))


@pytest.fixture
def gpu_rule(monkeypatch):
    monkeypatch.setattr(ops, "_skips_unused", lambda q: True)


def _inputs(n=7, device="cpu"):
    g = torch.Generator().manual_seed(3)
    ts = [torch.randn((2, 2, 9, 16), generator=g, dtype=torch.float64).to(device) for _ in range(n)]
    return [t.requires_grad_(True) for t in ts[:4]], ts[4:]


@pytest.mark.parametrize("device", ["cpu", pytest.param("cuda", marks=pytest.mark.gpu)])
def test_second_derivative_runs_each_op_once(request, device):
    if device == "cpu":
        request.getfixturevalue("gpu_rule")
    (q, k, v, do), cot = _inputs(device=device)
    with _Count() as seen:
        o = fused_attention(q, k, v)
        first = torch.autograd.grad(o, (q, k, v), do, create_graph=True)
        torch.autograd.grad(first, (q, k, v, do), cot)
    assert seen.calls == ["attn_fwd", "attn_bwd", "attn_bwd_bwd"]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_native_second_derivative_runs_each_op_once(dtype):
    g = torch.Generator().manual_seed(3)
    q, k, v, do, *cot = (torch.randn((2, 2, 9, 16), generator=g).to("cuda", dtype).requires_grad_(i < 4)
                         for i in range(7))
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU]) as prof:
        o = fused_attention(q, k, v)
        first = torch.autograd.grad(o, (q, k, v), do, create_graph=True)
        torch.autograd.grad(first, (q, k, v, do), cot)
    assert "CppNode" in o.grad_fn.name()
    counts = {e.key: e.count for e in prof.key_averages() if e.key.startswith("ebr_fused::")}
    assert counts == {"ebr_fused::attn_fwd": 1, "ebr_fused::attn_bwd": 1, "ebr_fused::attn_bwd_bwd": 1}


def test_second_derivative_with_a_use_of_the_output_runs_the_backward_again(gpu_rule):
    (q, k, v, do), cot = _inputs()
    with _Count() as seen:
        o = fused_attention(q, k, v)
        first = torch.autograd.grad(o, (q, k, v), do, create_graph=True)
        got = torch.autograd.grad([*first, o], (q, k, v), [*cot, do.detach()])
    assert seen.calls == ["attn_fwd", "attn_bwd", "attn_bwd_bwd", "attn_bwd"]

    def plain(q, k, v):
        return torch.softmax(q @ k.transpose(-1, -2) * 0.25, dim=-1) @ v

    o = plain(q, k, v)
    first = torch.autograd.grad(o, (q, k, v), do, create_graph=True)
    want = torch.autograd.grad([*first, o], (q, k, v), [*cot, do.detach()])
    for a, b in zip(got, want):
        torch.testing.assert_close(a, b, rtol=1e-10, atol=1e-10)


@pytest.mark.parametrize("used", [0, 1, 2])
def test_one_cotangent_alone(gpu_rule, used):
    """A cotangent for one of dq, dk, dv alone still reaches every input."""
    (q, k, v, do), cot = _inputs()
    o = fused_attention(q, k, v)
    first = torch.autograd.grad(o, (q, k, v), do, create_graph=True)
    got = torch.autograd.grad(first[used], (q, k, do), cot[used], allow_unused=True)
    o = torch.softmax(q @ k.transpose(-1, -2) * 0.25, dim=-1) @ v
    first = torch.autograd.grad(o, (q, k, v), do, create_graph=True)
    want = torch.autograd.grad(first[used], (q, k, do), cot[used], allow_unused=True)
    for a, b in zip(got, want):
        torch.testing.assert_close(a, torch.zeros_like(a) if b is None else b, rtol=1e-10, atol=1e-10)
