"""The native host path (``ebr_amd._host``): it gives the Python nodes' bits for every derivative, and leaves to them
every call that a mode, a transform, a hook or an argument check has to see."""

import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode
from torch.utils._python_dispatch import TorchDispatchMode

from ebr_amd import _host, block, descent, linear
from ebr_amd.fused_attn import fused_attention
from ebr_amd.fused_attn.rope_split import rope_split
from ebr_amd.layers import RotaryTable2D

gpu = pytest.mark.gpu
BF16, F16, F32 = torch.bfloat16, torch.float16, torch.float32


def _randn(shape, dtype, seed, device="cuda"):
    g = torch.Generator().manual_seed(seed)
    return torch.randn(shape, generator=g).to(device=device, dtype=dtype)


def _second_order(fn, xs, cots, seed=50):
    """Outputs, gradients and the gradients' derivatives of ``fn`` for every input."""
    xs = [x.detach().requires_grad_(True) for x in xs]
    ys = fn(*xs)
    ys = ys if isinstance(ys, tuple) else (ys,)
    cots = [c.detach().requires_grad_(True) for c in cots]
    first = torch.autograd.grad(ys, xs, cots, create_graph=True)
    wrt = [*xs, *cots]
    second = torch.autograd.grad(first, wrt, [_randn(t.shape, t.dtype, seed + i) for i, t in enumerate(first)],
                                 allow_unused=True)
    return [*ys, *first, *second]


def _same(got, want):
    assert len(got) == len(want)
    for a, b in zip(got, want):
        assert (a is None) == (b is None)
        if a is not None:
            assert a.dtype == b.dtype and a.shape == b.shape and a.stride() == b.stride()
            assert torch.equal(a, b)


def _attn_inputs(dtype, shape, views, seed=0):
    B, H, L, D = shape
    if views == "qkv":
        qkv = _randn((B, L, 3 * H * D), dtype, seed)
        return [t.view(B, L, H, D).transpose(1, 2) for t in qkv.split(H * D, dim=-1)]
    if views == "misaligned":  # rows that start 2 or 4 bytes past a 16-byte boundary: copied before the launch
        return [_randn((B, H, L, D + 1), dtype, seed + i)[..., 1:] for i in range(3)]
    return [_randn(shape, dtype, seed + i) for i in range(3)]


CASES = [
    ("attn", BF16, (2, 3, 17, 64), None), ("attn", F16, (1, 2, 130, 32), "qkv"), ("attn", F32, (2, 2, 33, 20), None),
    ("attn", F32, (1, 2, 140, 64), "misaligned"), ("attn", BF16, (1, 2, 100, 128), "qkv"),
    ("attn", BF16, (1, 1, 9, 200), None), ("rope", BF16, None, None), ("rope", F32, None, "scaled"),
    ("norm", BF16, None, None), ("norm", torch.float64, None, None), ("swiglu", F16, None, "view"),
    ("linear", BF16, None, None), ("linear", F32, None, "view"),
]


def _run(kind, dtype, shape, extra):
    if kind == "attn":
        cot = _randn(shape, dtype, 9)
        return _second_order(lambda q, k, v: fused_attention(q, k, v, 0.2), _attn_inputs(dtype, shape, extra), [cot])
    if kind == "rope":
        rope = RotaryTable2D(16, 3, 5).cuda()
        qs = torch.tensor([0.5, 2.0], device="cuda") if extra else None
        return _second_order(lambda x: rope_split(x, *rope(), 2, qs), [_randn((4, 15, 96), dtype, 1)],
                             [_randn((4, 2, 15, 16), dtype, 2 + i) for i in range(3)])
    if kind == "norm":
        return _second_order(lambda x: block.rms_norm(x, 1e-5), [_randn((3, 7, 24), dtype, 1)],
                             [_randn((3, 7, 24), dtype, 2)])
    if kind == "swiglu":
        x = _randn((5, 2, 48), dtype, 1)
        x = x.transpose(0, 1) if extra == "view" else x
        return _second_order(block.swiglu, [x], [_randn((*x.shape[:-1], 24), dtype, 2)])
    x = _randn((2, 1024, 32), dtype, 1)  # two split-K partials of 1,024 rows
    x = x[:, ::2] if extra == "view" else x
    return _second_order(linear.linear, [x, _randn((48, 32), dtype, 3)], [_randn((*x.shape[:-1], 48), dtype, 2)])


@gpu
@pytest.mark.parametrize("kind,dtype,shape,extra", CASES)
def test_same_bits_as_the_python_nodes(monkeypatch, kind, dtype, shape, extra):
    assert _host.module() is not None
    got = _run(kind, dtype, shape, extra)
    monkeypatch.setattr(_host, "module", lambda: None)
    _same(got, _run(kind, dtype, shape, extra))


@gpu
@pytest.mark.parametrize("dtype", [BF16, F16, F32, torch.float64])
@pytest.mark.parametrize("shape", [(3, 512), (7, 27), (5, 1032), (2, 2, 4104), (9, 8)])
@pytest.mark.parametrize("kind", ["norm", "add_norm", "swiglu"])
def test_sums_inside_the_kernels_round_as_their_own(monkeypatch, kind, shape, dtype):
    """The residual sum and the second derivative's gradient sums, folded into the norm's and SwiGLU's kernels, against
    kernels of their own; row widths of every variant (vectors in registers, streamed, odd)."""
    shape = (*shape[:-1], 2 * shape[-1]) if kind == "swiglu" else shape
    x, r = (_randn(shape, dtype, i) for i in range(2))
    out = (*shape[:-1], shape[-1] // 2) if kind == "swiglu" else shape

    def go():
        # squared, so that the second derivative reaches the forward's node both ways
        if kind == "norm":
            return _second_order(lambda a: block.rms_norm(a, 1e-5).square(), [x], [_randn(out, dtype, 3)])
        if kind == "add_norm":
            return _second_order(lambda a, b: block.add_rms_norm(a, b, 1e-5).square(), [x, r], [_randn(out, dtype, 3)])
        return _second_order(lambda a: block.swiglu(a).square(), [x], [_randn(out, dtype, 3)])

    got = go()
    monkeypatch.setattr(_host, "module", lambda: None)
    _same(got, go())


@gpu
@pytest.mark.parametrize("dtype", [BF16, F16])
@pytest.mark.parametrize("rows,N,K", [(2048, 48, 32), (4096, 7, 9), (8192, 40, 24), (16384, 33, 65), (16384, 256, 6144)])
def test_split_weight_gradients(dtype, rows, N, K):
    """2, 4, 8 and 16 partial products (8 where the output is large), whole vectors and odd sizes."""
    x, dy = _randn((rows, K), dtype, 1), _randn((rows, N), dtype, 2)
    w = _randn((N, K), dtype, 3).requires_grad_(True)
    (got,) = torch.autograd.grad(linear.linear(x, w), w, dy)
    want = dy.double().t() @ x.double()
    # fp32 sums of exact products, rounded once: half an ulp of the dtype, plus the sums' own error
    eps = torch.finfo(dtype).eps
    assert ((got.double() - want).abs() <= 0.51 * eps * want.abs() + 1e-5 * rows**0.5).all()
    assert torch.equal(got, linear.weight_grad(dy, x))  # the partials' sum and its rounding as ops of their own


@gpu
@pytest.mark.parametrize("dtype", [BF16, F32])
@pytest.mark.parametrize("per_row,masked", [(True, True), (False, False), (True, False)])
def test_descent_same_bits_as_the_python_nodes(monkeypatch, dtype, per_row, masked):
    B, L, C = 3, 10, 64

    def go():
        z, n, g = (_randn((B, L, C), dtype, i).requires_grad_(i != 1) for i in range(3))
        sig = torch.tensor([0.1, 0.2, 0.3], device="cuda").to(dtype).view(B, 1, 1) if per_row else 0.25
        act = torch.tensor([True, False, True], device="cuda").view(B, 1, 1) if masked else None
        vs = [descent.noisy_point(z, n, sig), descent.noisy_point_replayed(z, n), descent.normalize(z)]
        outs = [descent.step_and_project(v, g, sig, z, act) for v in vs]
        return [*vs, *outs, *torch.autograd.grad(outs, (z, g), [_randn((B, L, C), dtype, 7 + i) for i in range(3)])]

    got = go()
    monkeypatch.setattr(_host, "module", lambda: None)
    _same(got, go())


@gpu
def test_a_single_used_gradient_and_unused_outputs(monkeypatch):
    """Zero rows for the cotangents nobody gives, in attention and in the rotary split."""
    rope = RotaryTable2D(16, 3, 5).cuda()

    def go():
        x = _randn((2, 15, 96), BF16, 1).requires_grad_(True)
        q, k, v = rope_split(x, *rope(), 2)
        o = fused_attention(q, k, v)
        (dq,) = torch.autograd.grad(o, q, _randn(o.shape, BF16, 2), create_graph=True)
        return [*torch.autograd.grad(dq, x, _randn(dq.shape, BF16, 3), retain_graph=True),
                *torch.autograd.grad(k, x, _randn(k.shape, BF16, 4))]

    got = go()
    monkeypatch.setattr(_host, "module", lambda: None)
    _same(got, go())


@gpu
def test_plain_calls_take_it():
    q = _randn((1, 2, 16, 16), BF16, 0).requires_grad_(True)
    assert "CppNode" in block.add_rms_norm(q, q, 1e-5).grad_fn.name()
    x = _randn((1, 4, 24), BF16, 0).requires_grad_(True)
    rope = RotaryTable2D(4, 2, 2).cuda()
    for y in (fused_attention(q, q, q), block.rms_norm(q, 1e-5), block.swiglu(q), linear.linear(q, q[0, 0]),
              descent.normalize(q[0]), descent.step_and_project(q[0], q[0], 0.1, q[0], None),
              rope_split(x, *rope(), 2)[0]):
        assert "CppNode" in y.grad_fn.name()


@gpu
@pytest.mark.parametrize("path,kind", [("native", "norm"), ("native", "add_norm"), ("native", "swiglu"),
                                       ("python", "norm"), ("python", "swiglu")])
def test_a_second_derivative_alone_leaves_the_forward_node_usable(monkeypatch, kind, path):
    if path == "python":
        monkeypatch.setattr(_host, "module", lambda: None)
    x0, r = _randn((3, 5, 24), F32, 1), _randn((3, 5, 24), F32, 2)
    fn = {"norm": lambda x: block.rms_norm(x, 1e-5), "swiglu": block.swiglu,
          "add_norm": lambda x: block.add_rms_norm(x, r, 1e-5)}[kind]

    def graph():
        x = x0.clone().requires_grad_(True)
        z = x * 1
        y = fn(z)
        dy = _randn(y.shape, F32, 3)
        (g,) = torch.autograd.grad(y, z, dy, create_graph=True)
        return z, y, dy, g

    def first(y, z, dy, **kw):
        return torch.autograd.grad(y, z, dy, **kw)[0]

    z, y, dy, g = graph()
    h = first(g, z, x0)
    assert torch.equal(first(y, z, dy, create_graph=True), g)  # still there, once more and recorded
    again = first(y, z, dy, create_graph=True)
    assert torch.equal(first(again, z, x0), h)
    assert torch.equal(first(y, z, dy), g)  # and this pass uses it up
    with pytest.raises(RuntimeError, match="second time"):
        first(y, z, dy)
    z, y, dy, g = graph()
    assert torch.equal(first(y, z, dy), g)  # used up by the first derivative: the recorded gradient has its own
    assert torch.equal(first(g, z, x0), h)
    with pytest.raises(RuntimeError, match="second time"):
        first(y, z, dy)
    del z, y, dy, g, h, again
    before = torch.cuda.memory_allocated()
    z, y, dy, g = graph()
    first(g, z, x0)
    assert torch.cuda.memory_allocated() > before
    del z, y, dy, g  # what was set aside goes with the graph
    assert torch.cuda.memory_allocated() == before
    if kind != "add_norm":  # the sum is no tensor of the caller's
        z, y, dy, g = graph()
        first(g, z, x0)
        with torch.no_grad():
            z.add_(1)
        with pytest.raises(RuntimeError, match="inplace"):
            first(y, z, dy)


@gpu
def test_no_derivative_past_the_second():
    x = _randn((4, 16), F32, 0).requires_grad_(True)
    (g,) = torch.autograd.grad(block.rms_norm(x, 1e-5).square().sum(), x, create_graph=True)
    (h,) = torch.autograd.grad(g.square().sum(), x, create_graph=True)
    with pytest.raises(RuntimeError):
        h.sum().backward()
    q, k, v = (_randn((1, 1, 8, 16), F32, i).requires_grad_(True) for i in range(3))
    (g,) = torch.autograd.grad(fused_attention(q, k, v).square().sum(), q, create_graph=True)
    (h,) = torch.autograd.grad(g.square().sum(), q, create_graph=True)
    with pytest.raises(RuntimeError):
        torch.autograd.grad(h.sum(), q)


class _Seen(TorchDispatchMode):
    def __init__(self):
        super().__init__()
        self.ops = []

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        self.ops.append(str(func))
        return func(*args, **(kwargs or {}))


@gpu
def test_modes_transforms_and_hooks_see_the_ops():
    q, k, v = (_randn((1, 2, 9, 16), F32, i).requires_grad_(True) for i in range(3))
    with _Seen() as seen:
        want = fused_attention(q, k, v)
    assert "ebr_fused.attn_fwd.default" in seen.ops
    packed = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: packed.append(t.shape) or t, lambda t: t):
        o = fused_attention(q, k, v)
    assert len(packed) == 5 and torch.equal(o, want)
    g = torch.func.grad(lambda x: fused_attention(x, k.detach(), v.detach()).sum())(q.detach())
    assert torch.equal(g, torch.autograd.grad(want.sum(), q)[0])
    out = torch.compile(lambda x: fused_attention(x, k, v) * 2, backend="aot_eager", fullgraph=True)(q)
    assert torch.equal(out, want * 2)
    with pytest.raises((RuntimeError, NotImplementedError)):
        torch.func.jvp(lambda x: fused_attention(x, k.detach(), v.detach()), (q.detach(),), (q.detach(),))


def _rope_attn_case(dtype, device="cuda"):
    """rope_attention of 2 heads of 32 on a 3 x 4 grid: (fn, inputs)."""
    from ebr_amd.fused_attn.rope_split import rope_attention

    cos, sin = (t.to(dtype) if dtype == torch.float64 else t for t in RotaryTable2D(32, 3, 4).to(device)())
    xs = [_randn((2, 12, 192), dtype, 1, device), torch.tensor([0.7, 1.3], device=device)]
    fn = rope_attention if device == "cuda" else _parts
    return (lambda x, t: fn(x, cos, sin, 2, t)), xs


def _grads_case(kind):
    q = [_randn((2, 2, 9, 16), F32, i) for i in range(3)]
    x = _randn((2, 12, 24), F32, 4)
    if kind == "attn":
        return fused_attention, q
    if kind == "rope":
        cos, sin = RotaryTable2D(4, 3, 4).cuda()()
        return (lambda y: rope_split(y, cos, sin, 2)), [x]
    if kind == "rope_attn":
        return _rope_attn_case(F32)
    if kind == "norm":
        return (lambda y: block.rms_norm(y, 1e-5)), [x]
    if kind == "add_norm":
        return (lambda y, r: block.add_rms_norm(y, r, 1e-5)), [x, _randn(x.shape, F32, 5)]
    if kind == "swiglu":
        return block.swiglu, [x]
    if kind == "linear":
        return linear.linear, [x, _randn((5, 24), F32, 6)]
    if kind == "noisy":
        return (lambda z: descent.noisy_point(z, x, 0.3)), [x]
    act = torch.tensor([True, False], device="cuda").view(2, 1, 1)
    return (lambda v, g, z: descent.step_and_project(v, g, 0.1, z, act)), [_randn(x.shape, F32, i) for i in range(3)]


KINDS = ["attn", "rope", "rope_attn", "norm", "add_norm", "swiglu", "linear", "noisy", "step"]


def _nearly(a, b):
    torch.testing.assert_close(a, b, rtol=2e-6, atol=2e-6 * b.abs().max().item())  # fp32 sums in another order


@gpu
@pytest.mark.parametrize("kind", KINDS)
def test_batched_gradients(kind):
    """A plain forward, then backwards under vmap: first derivatives, and the derivatives of recorded ones."""
    fn, xs = _grads_case(kind)
    xs = [x.detach().requires_grad_(True) for x in xs]
    ys = fn(*xs)
    ys = ys if isinstance(ys, tuple) else (ys,)
    assert "CppNode" in ys[0].grad_fn.name()

    def both(outs, wrt, seed):
        cots = [_randn((3, *o.shape), o.dtype, seed + i) for i, o in enumerate(outs)]
        got = torch.autograd.grad(outs, wrt, cots, is_grads_batched=True, retain_graph=True)
        want = [torch.autograd.grad(outs, wrt, [c[i] for c in cots], retain_graph=True) for i in range(3)]
        for i, g in enumerate(got):
            _nearly(g, torch.stack([w[i] for w in want]))

    both(ys, xs, 20)
    if kind in ("noisy", "step"):  # first order only
        return
    cots = [_randn(y.shape, y.dtype, 30 + i).requires_grad_(True) for i, y in enumerate(ys)]
    if kind == "rope_attn":  # its node of dx alone, and the one that records dt too
        (dx,) = torch.autograd.grad(ys, xs[:1], cots, create_graph=True)
        both([dx], [*xs, *cots], 40)
        both([dx.square() + ys[0].repeat(1, 1, 3)], xs, 45)
    first = torch.autograd.grad(ys, xs, cots, create_graph=True)
    linear_in_x = kind in ("rope", "linear")  # no derivative of dx for x
    both(first, cots if linear_in_x else [*xs, *cots], 50)


@gpu
def test_vectorised_jacobian_and_hessian():
    q, k, v = (_randn((1, 1, 3, 16), F32, i) for i in range(3))
    for strategy in (torch.autograd.functional.jacobian, torch.autograd.functional.hessian):
        def fn(x):
            y = block.swiglu(block.rms_norm(fused_attention(x, k, v), 1e-5))
            return y if strategy is torch.autograd.functional.jacobian else y.square().sum()

        _nearly(strategy(fn, q, vectorize=True), strategy(fn, q))


@gpu
def test_a_mode_around_the_backward_alone_sees_the_ops():
    q, k, v = (_randn((1, 2, 9, 16), F32, i).requires_grad_(True) for i in range(3))
    x = _randn((4, 16), F32, 3).requires_grad_(True)
    o, n = fused_attention(q, k, v), block.swiglu(block.rms_norm(x, 1e-5))
    with _Seen() as seen:
        first = torch.autograd.grad([o, n], (q, k, v, x), [q.detach(), n.detach()], create_graph=True)
        torch.autograd.grad(first, (q, k, v, x), [t.detach() for t in first])
    for op in ("attn_bwd", "attn_bwd_bwd", "block_rmsnorm_bwd", "block_rmsnorm_bwd2", "block_swiglu_bwd",
               "block_swiglu_bwd2"):
        assert f"ebr_fused.{op}.default" in seen.ops
    packed = []
    o = fused_attention(q, k, v)
    with torch.autograd.graph.saved_tensors_hooks(lambda t: packed.append(t.shape) or t, lambda t: t):
        torch.autograd.grad(o, (q, k, v), q.detach(), create_graph=True)
    assert len(packed) == 7


def test_python_gradients_of_rope_attention():
    """The formulas behind the native rope-attention node, on the CPU in 64 bits, against autograd of the parts."""
    from ebr_amd.fused_attn import ops

    fn, (x, t) = _rope_attn_case(torch.float64, "cpu")
    cos, sin = (c.double() for c in RotaryTable2D(32, 3, 4)())
    x, t = x.requires_grad_(True), t.double().requires_grad_(True)
    dy = _randn((2, 12, 64), torch.float64, 3, "cpu").requires_grad_(True)
    c = _randn((2, 12, 192), torch.float64, 4, "cpu")
    want = torch.autograd.grad(fn(x, t), (x, t), dy, create_graph=True)
    second = torch.autograd.grad(want[0], (x, t, dy), c)
    q, k, v = rope_split(x, cos, sin, 2)
    q = q * t.view(1, 2, 1, 1)
    o, lse = torch.ops.ebr_fused.attn_fwd(q.detach(), k.detach(), v.detach(), 32**-0.5)
    saved = [u.detach().requires_grad_(True) for u in (q, k, v)]
    args = (t, *saved, dy, o, lse, cos, sin)
    got = _host.GRADS["rope_attention"](x.detach(), t, cos, sin, *saved, o, lse, 32**-0.5, True, dy, None, None, None)
    for a, b in zip(got, want):
        torch.testing.assert_close(a, b, rtol=1e-9, atol=1e-9)
    dq = ops._FusedAttnBwd.apply(*saved, o, lse, dy.reshape(2, 12, 2, 32).transpose(1, 2), 32**-0.5)[0]
    dt, hq, hk, hv, hdy = _host.GRADS["rope_attention_bwd"](*args, dq, 32**-0.5, True, c)
    dx, dt2 = _host.GRADS["rope_attention"](x.detach(), t, cos, sin, *saved, o, lse, 32**-0.5, True, None, hq, hk, hv)
    for a, b in zip((dx, dt + dt2, hdy), second):
        torch.testing.assert_close(a, b, rtol=1e-9, atol=1e-9)


@gpu
def test_refused_calls_stay_refused():
    q = _randn((1, 2, 9, 16), F32, 0)
    with pytest.raises(ValueError):
        fused_attention(q, q[:, :1], q)
    with pytest.raises(ValueError):
        fused_attention(q, q.half(), q)
    with pytest.raises(ValueError):
        fused_attention(*[_randn((1, 1, 4, 264), F32, 0)] * 3)
    with pytest.raises(ValueError):
        block.swiglu(_randn((3, 5), F32, 0))
    with pytest.raises(TypeError):
        descent.noisy_point(_randn((2, 3, 4), BF16, 0), _randn((2, 3, 4), BF16, 0), torch.ones((2, 1, 1)).cuda())
    with pytest.raises(ValueError):
        descent.step_and_project(*[_randn((2, 3, 4), F32, 0)] * 2, torch.ones((3, 1, 1)).cuda(),
                                 _randn((2, 3, 4), F32, 0), None)
    assert fused_attention(*[_randn((1, 2, 9, 20), BF16, 0)] * 3).shape == (1, 2, 9, 20)  # padded in Python
    assert fused_attention(*[_randn((0, 2, 9, 16), BF16, 0)] * 3).shape == (0, 2, 9, 16)


@gpu
def test_on_a_side_stream_and_from_threads():
    import threading

    q, k, v = (_randn((4, 2, 40, 64), BF16, i) for i in range(3))
    want = fused_attention(q, k, v)
    got = [None] * 4
    torch.cuda.synchronize()

    def work(i):
        s = torch.cuda.Stream()
        with torch.cuda.stream(s):
            x = q.clone().requires_grad_(True)
            o = fused_attention(x, k, v)
            (g,) = torch.autograd.grad(o, x, v)
        s.synchronize()
        got[i] = (o.detach(), g)

    ts = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    [t.start() for t in ts]
    [t.join() for t in ts]
    for o, g in got:
        assert torch.equal(o, want) and torch.equal(g, got[0][1])


def test_leaves_other_tensors_to_python():
    host = _host.module()
    if host is None:
        pytest.skip("the native host path is not built")
    x = torch.randn(2, 4, 8, 16)
    assert host.attention(x, x, x, None) is None and host.attention(1, None, "x", 0.5) is None
    assert host.rms_norm(x, 1e-5) is None and host.swiglu(x) is None and host.linear(x, x[0, 0]) is None
    assert host.noisy_point(x[0], x[0], 0.1, 1e-5) is None
    assert host.step_and_project(x[0], x[0], 0.1, x[0], None, 1e-5) is None
    assert host.rope_split(x[0], x[0, 0], x[0, 0], 2, None) is None
    with FakeTensorMode():
        f = torch.empty(2, 4, 8, 16, device="cuda")
        assert host.attention(f, f, f, None) is None and host.rms_norm(f, 1e-5) is None


def test_host_command_links_the_library_beside_it():
    from pathlib import Path

    from ebr_amd import build

    cmd = build.host_command(Path("x.so"))
    assert "-lebr_attn" in cmd and "-Wl,-rpath,$ORIGIN" in cmd and cmd[-1] == "x.so"


def _parts(qkv, cos, sin, heads, t):
    """rope_attention by its parts."""
    b, n, _ = qkv.shape
    q, k, v = rope_split(qkv, cos, sin, heads)
    y = fused_attention(q * t.to(q.dtype).view(1, heads, 1, 1), k, v)
    return y.transpose(1, 2).reshape(b, n, -1)


def _close(got, want, dtype, size):
    """Bits for what the parts round alike; the temperature's gradient to its sum's precision: the parts round every
    product and their sum to the dtype, an error of a few roundings of the products' 2-norm (``size``)."""
    for a, b in zip(got, want):
        assert (a is None) == (b is None)
        if a is None:
            continue
        if a.dim() == 1:
            scale = b.float().abs().max().clamp_min(size)
            assert ((a.float() - b.float()).abs().max() / scale).item() < {BF16: 3e-2, F16: 4e-3, F32: 1e-5}[dtype]
        else:
            assert torch.equal(a, b)


@gpu
@pytest.mark.parametrize("dtype", [BF16, F16, F32])
@pytest.mark.parametrize("B,grid,H,D", [(1, (3, 3), 1, 32), (3, (3, 5), 3, 64), (5, (7, 7), 4, 128), (2, (12, 12), 8, 32)])
def test_rope_attention_is_its_parts(dtype, B, grid, H, D):
    """Rows that fill no workgroup and rows that fill many; heads that no workgroup holds evenly."""
    from ebr_amd.fused_attn.rope_split import rope_attention

    N = grid[0] * grid[1]
    cos, sin = RotaryTable2D(D, *grid).cuda()()
    qkv, dy, c = _randn((B, N, 3 * H * D), dtype, 1), _randn((B, N, H * D), dtype, 2), _randn((B, N, 3 * H * D), dtype, 3)
    t0 = torch.linspace(0.7, 1.6, H, device="cuda")

    def go(fn):
        x, t, d = qkv.clone().requires_grad_(True), t0.clone().requires_grad_(True), dy.clone().requires_grad_(True)
        y = fn(x, cos, sin, H, t)
        assert y is not None
        (g,) = torch.autograd.grad(y, x, d, create_graph=True)
        second = torch.autograd.grad(g, (x, t, d), c, retain_graph=True)  # nothing uses y a second time
        both = torch.autograd.grad([g, y.float().square().to(dtype)], (x, t), [c, dy], retain_graph=True)
        gt = torch.autograd.grad(y, (x, t), dy, create_graph=True)  # every part recorded
        third = torch.autograd.grad(gt[0], (x, t), c)
        plain = torch.autograd.grad(fn(x, cos, sin, H, t.detach()), x, dy)  # an inference step
        return [y, g, *second, *both, *gt, *third, *plain]

    got, want = go(rope_attention), go(_parts)
    # a head's products dq * R q as independent values of the norms of g and qkv
    size = (want[1].float().norm() * qkv.float().norm() / (3 * H * (B * N * D) ** 0.5)).item()
    _close(got, want, dtype, size)
    assert torch.equal(go(rope_attention)[3], got[3])  # the same sums on every run


@gpu
@pytest.mark.parametrize("dtype,head_dim", [(BF16, 32), (F32, 16)])
def test_graded_blocks_test_rope_attention_first(dtype, head_dim):
    from ebr_amd import attention

    layer = attention.EnergyAttention(2 * head_dim, head_dim, 2, backend="fused", nograd_backend="fused").cuda()
    rope = RotaryTable2D(head_dim, 3, 3).cuda()()
    x = _randn((2, 9, 2 * head_dim), dtype, 1)
    layer(rope, x)
    assert not layer._node_verified
    with attention.second_order_window(True):
        layer(rope, x)
    assert layer._verified and layer._node_verified
    with _Seen():  # the parts run: nothing to test
        assert not attention.verify_rope_attention(device=x.device)


@gpu
def test_rope_attention_leaves_other_calls():
    from ebr_amd.fused_attn.rope_split import rope_attention

    t = torch.ones(2, device="cuda")
    for D in (16, 96, 20):  # no power of two of whole vectors
        cos, sin = RotaryTable2D(D, 2, 2).cuda()()
        assert rope_attention(_randn((1, 4, 6 * D), BF16, 0), cos, sin, 2, t) is None
    cos, sin = RotaryTable2D(32, 2, 2).cuda()()
    x = _randn((1, 4, 192), BF16, 0)
    assert rope_attention(x, cos, sin, 2, torch.ones(3, device="cuda")) is None
    assert rope_attention(x, cos, sin, 2, t.bfloat16()) is None and rope_attention(x, cos[1:], sin, 2, t) is None
    assert rope_attention(x.double(), cos, sin, 2, t) is None
    with _Seen() as seen:
        assert rope_attention(x, cos, sin, 2, t) is None
    assert not seen.ops
