"""Performance cases of the framework: the calls that a training or an inference program makes through the public entry
points, from one board to a full training batch.

A case is a dict of plain values. ``kind`` says which call it is:

- ``attn``     ``fused_attention`` on [B, H, L, D]. ``order`` 2 is a graded descent step (forward, gradient with
               ``create_graph``, and the derivative of that gradient); ``order`` 1 is an inference descent step (forward
               and gradient). ``views`` True passes q, k and v as the views of one [B, L, 3 H D] projection that the
               unfused rotary path passes; False passes the contiguous tensors of the fused rotary split.
- ``wrapper``  the pointwise work around one descent microstep, ``noisy_point`` and ``step_and_project``, with the
               gradients of both.
- ``block``    one ``EnergyReasoningBlock`` (projections, rotary split, attention, norms, SwiGLU) in a graded step: its
               output, its input gradient, and the derivatives of that gradient for the input and every weight.
- ``train``    ``train_step`` of the energy network: graded descent, cross entropy, backward.
- ``solve``    inference: descent microsteps without a graph, then the decoder's logits.
"""

import math

import torch
import torch.nn.functional as F

from ebr_amd import descent, energy
from ebr_amd.attention import prime_attention_self_test, second_order_window
from ebr_amd.fused_attn import fused_attention

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
SIZES = {"bf16": 2, "fp16": 2, "fp32": 4}
EPS = 1e-5
SIGMA = 0.05
ALPHA = 0.1
EXPANSION = 4.0
VOCAB = 11


def listed():
    return [
        # One 9 x 9 board in a graded step: nothing but launches and the host path.
        dict(name="attn_one_board", kind="attn", dtype="bf16", B=1, H=4, L=81, D=64, order=2, views=False),
        # 8 x 8 N-Queens in fp32: a debugging run's batch, and what the fp32 kernels see.
        dict(name="attn_nqueens_fp32", kind="attn", dtype="fp32", B=32, H=8, L=64, D=64, order=2, views=False),
        # Sudoku training: the attention of one graded step of the 768-board recipe.
        dict(name="attn_sudoku", kind="attn", dtype="bf16", B=768, H=8, L=81, D=64, order=2, views=False),
        # 10 x 10 multi-solution training: hidden 512 over 4 heads of 128.
        dict(name="attn_multi", kind="attn", dtype="bf16", B=768, H=4, L=100, D=128, order=2, views=False),
        # 30 x 30 Maze training: the longest sequences.
        dict(name="attn_maze", kind="attn", dtype="bf16", B=64, H=8, L=900, D=64, order=2, views=False),
        # Inference over 5120 latents of 10 x 10 boards: forward and gradient only.
        dict(name="attn_descent", kind="attn", dtype="bf16", B=5120, H=8, L=100, D=64, order=1, views=False),
        # fp16 with an odd length between the short and the long boards, read from projection views.
        dict(name="attn_fp16_views", kind="attn", dtype="fp16", B=16, H=8, L=333, D=64, order=2, views=True),
        # fp32 on a 20 x 20 board: exactness checks of a run on longer sequences.
        dict(name="attn_fp32_long", kind="attn", dtype="fp32", B=8, H=8, L=400, D=64, order=2, views=False),
        # The pointwise work around a training microstep, with some rows already finished.
        dict(name="wrapper_sudoku", kind="wrapper", dtype="bf16", B=384, L=81, C=512, masked=True),
        # One block of the training network in a graded step.
        dict(name="block_sudoku", kind="block", dtype="bf16", B=384, G=9, hidden=512, heads=8),
        # A whole (short) training step of the two-layer network.
        dict(name="train_sudoku", kind="train", dtype="bf16", B=384, G=9, hidden=512, heads=8, layers=2, steps=2),
        # Inference descent of the same network over 10 x 10 boards.
        dict(name="solve_boards", kind="solve", dtype="bf16", B=640, G=10, hidden=512, heads=8, layers=2, steps=2),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    kind = rng.choice(("short", "short", "short", "long", "long", "fp32", "fp32", "wrapper", "block", "train", "solve"))
    if kind in ("short", "long", "fp32"):
        H, D = rng.choice(((4, 64), (8, 64), (4, 128), (4, 32)))
        if kind == "fp32":
            dtype, L, most = "fp32", _log_int(rng, 9, 400), 20e9
        else:
            dtype = rng.choice(("bf16", "bf16", "bf16", "fp16"))
            L = rng.randint(9, 128) if kind == "short" else _log_int(rng, 129, 900)
            most = 600e9
        order = rng.choice((1, 2, 2))
        # the batch: from one board to the recipes' largest, bounded by the arithmetic of a pass
        per = (14 if order == 1 else 38) * L * L * D * H
        B = _log_int(rng, 1, max(1, min(1024 if order == 2 else 5120, int(most / per))))
        return dict(kind="attn", dtype=dtype, B=B, H=H, L=L, D=D, order=order, views=rng.random() < 0.3)
    if kind == "wrapper":
        L, C = rng.choice((rng.randint(16, 128), _log_int(rng, 129, 900))), rng.choice((256, 512))
        B = _log_int(rng, 1, max(1, min(768, int(16e6 / (L * C)))))
        return dict(kind="wrapper", dtype=rng.choice(("bf16", "bf16", "fp16", "fp32")), B=B, L=L, C=C,
                    masked=rng.random() < 0.5)
    hidden, heads = rng.choice(((256, 4), (512, 8), (512, 4)))
    G = rng.randint(4, 16)
    if kind == "block":
        return dict(kind="block", dtype="bf16", B=_log_int(rng, 1, max(1, int(30000 / (G * G)))), G=G, hidden=hidden,
                    heads=heads)
    if kind == "train":
        return dict(kind="train", dtype="bf16", B=_log_int(rng, 4, max(4, int(28000 / (G * G)))), G=G, hidden=hidden,
                    heads=heads, layers=rng.choice((1, 2)), steps=rng.choice((1, 2)))
    return dict(kind="solve", dtype="bf16", B=_log_int(rng, 1, max(1, int(60000 / (G * G)))), G=G, hidden=hidden,
                heads=heads, layers=2, steps=rng.choice((1, 2, 3)))


def _network(case):
    return energy.EnergyConfig(
        hidden_size=case["hidden"], num_heads=case["heads"], num_layers=case.get("layers", 1), expansion=EXPANSION,
        vocab_size=VOCAB, grid=(case["G"], case["G"]), rope_impl="fused", block_impl="fused", linear_impl="splitk",
    )


def _inputs(case, seed):
    """The tensors of a case, in a fixed order of draws, on the GPU."""
    dev = torch.device("cuda")
    g = torch.Generator(dev).manual_seed(seed)
    dt = DTYPES[case["dtype"]]

    def randn(*shape, dtype=dt):
        return torch.randn(shape, generator=g, device=dev, dtype=torch.float32).to(dtype)

    if case["kind"] == "attn":
        B, H, L, D = case["B"], case["H"], case["L"], case["D"]
        # q and k of unit variance: scores of unit variance at the scale D^-1/2, as normalised activations give
        if case["views"]:
            qkv = randn(B, L, 3 * H * D)
            q, k, v = (t.view(B, L, H, D).transpose(1, 2) for t in qkv.split(H * D, dim=-1))
        else:
            q, k, v = (randn(B, H, L, D) for _ in range(3))
        n = 1 if case["order"] == 1 else 4  # dO, and the cotangents of dQ, dK, dV
        return [q, k, v] + [randn(B, H, L, D) for _ in range(n)]
    if case["kind"] == "wrapper":
        B, L, C = case["B"], case["L"], case["C"]
        ts = {n: randn(B, L, C) for n in ("z", "noise", "g", "dv", "dout")}
        ts["sigma"] = (torch.rand((B, 1, 1), generator=g, device=dev) * SIGMA).to(dt)
        ts["alpha"] = (torch.rand((B, 1, 1), generator=g, device=dev) * ALPHA + 0.5 * ALPHA).to(dt)
        ts["active"] = torch.rand((B, 1, 1), generator=g, device=dev) < 0.8 if case["masked"] else None
        return ts
    B, L, C = case["B"], case["G"] ** 2, case["hidden"]
    ts = {"z": randn(B, L, C)}
    if case["kind"] == "block":
        ts["dy"], ts["c"] = randn(B, L, C), randn(B, L, C)
    else:
        ts["x"] = torch.randint(0, VOCAB, (B, L), generator=g, device=dev)
        ts["targets"] = torch.randint(0, VOCAB, (B, L), generator=g, device=dev)
        ts["noise"] = randn(B, L, C) * SIGMA
    return ts


def prepare(case, seed):
    ts = _inputs(case, seed)
    if case["kind"] == "attn":
        q, k, v = (t.detach().requires_grad_(True) for t in ts[:3])
        do = ts[3].requires_grad_(case["order"] == 2)
        return dict(case=case, q=q, k=k, v=v, do=do, cot=tuple(ts[4:]))
    if case["kind"] == "wrapper":
        for n in ("z", "g"):
            ts[n].requires_grad_(True)
        return dict(case=case, **ts)
    with torch.random.fork_rng(devices=["cuda"]):
        model, decoder = energy.build(_network(case), torch.device("cuda"), seed=seed)
    prime_attention_self_test(model)  # the attention's one-time self-test, as a program runs it at its start
    if case["kind"] == "solve":
        for p in model.parameters():
            p.requires_grad_(False)
    return dict(case=case, model=model, decoder=decoder, **ts)


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "attn":
        q, k, v, do = state["q"], state["k"], state["v"], state["do"]
        o = fused_attention(q, k, v)
        if case["order"] == 1:
            return [o.detach(), *torch.autograd.grad(o, (q, k, v), do)]
        first = torch.autograd.grad(o, (q, k, v), do, create_graph=True)
        second = torch.autograd.grad(first, (q, k, v, do), state["cot"])
        return [o.detach(), *(t.detach() for t in first), *second]
    if kind == "wrapper":
        z, g = state["z"], state["g"]
        v = descent.noisy_point(z, state["noise"], state["sigma"], EPS)
        (dz,) = torch.autograd.grad(v, z, state["dv"])
        w = v.detach().requires_grad_(True)
        out = descent.step_and_project(w, g, state["alpha"], z, state["active"], EPS)
        wrt = (w, g, z) if case["masked"] else (w, g)
        return [v.detach(), dz, out.detach(), *torch.autograd.grad(out, wrt, state["dout"])]
    model = state["model"]
    if kind == "block":
        layer = model.layers[0]
        x = state["z"].detach().requires_grad_(True)
        with second_order_window(True):
            y = layer(model.rope(), x)
        (dx,) = torch.autograd.grad(y, x, state["dy"], create_graph=True)
        second = torch.autograd.grad(dx, (x, *layer.parameters()), state["c"])
        return [y.detach(), dx.detach(), *second]
    if kind == "train":
        model.zero_grad(set_to_none=True)
        state["decoder"].zero_grad(set_to_none=True)
        loss = energy.train_step(model, state["decoder"], state["x"], state["z"], state["targets"],
                                 steps=case["steps"], alpha=ALPHA)
        grads = {n: p.grad for n, p in model.named_parameters()}
        grads["lm_head"] = state["decoder"].lm_head.weight.grad
        return {"loss": loss, "grads": grads}
    with torch.no_grad():
        x_emb = model.puzzle_embedding(state["x"], state["z"].dtype)
    noises = [state["noise"]] * case["steps"]
    v = energy.descend(model, state["z"], x_emb, case["steps"], ALPHA, create_graph=False, wrapper="fused",
                       noises=noises)
    with torch.no_grad():
        return {"logits": state["decoder"](v), "z": v.detach()}


# -- what a pass cannot do without -------------------------------------------------------------------------------------


def _attn_work(B, H, L, D, es, order):
    """The inputs and outputs of forward, gradient and its derivative, each once; the contractions of L x L x D."""
    tensors, stats = (4, 1) if order == 0 else (12, 2) if order == 1 else (24, 3)
    units = 2 if order == 0 else 7 if order == 1 else 19
    return (tensors * L * D * es + stats * 4 * L) * B * H, 2 * units * L * L * D * B * H


def _inter(hidden):
    return -(-round(EXPANSION * hidden * 2 / 3) // 256) * 256


def _block_work(case, order):
    """One block: its projections' products, its attention, and one read and one write of each tensor between them."""
    M, C, es = case["B"] * case["G"] ** 2, case["hidden"], SIZES[case["dtype"]]
    inter = _inter(C)
    weights = C * 3 * C + C * C + C * 2 * inter + inter * C
    H = case["heads"]
    ab, af = _attn_work(case["B"], H, case["G"] ** 2, C // H, es, order)
    # products with the weights: forward; its input gradient; and of both, the input and the weight gradients
    products = {0: 1, 1: 2, 2: 6}[order]
    # per token and order: qkv, attention's out, o_proj's out, norm, gate and up, the activation, down's out, norm
    widths = 3 * C + 2 * C + 2 * inter + inter + 3 * C
    passes = {0: 2, 1: 4, 2: 10}[order]
    return ab + passes * M * widths * es + products * weights * es, af + products * 2 * M * weights


def work(case):
    es = SIZES[case["dtype"]]
    if case["kind"] == "attn":
        b, f = _attn_work(case["B"], case["H"], case["L"], case["D"], es, case["order"])
        return {"bytes": float(b), "flops": float(f)}
    if case["kind"] == "wrapper":
        n = case["B"] * case["L"] * case["C"]
        # noisy point: z, noise -> v; its gradient: z, dv -> dz; step: v, g (z) -> out; its gradient: v, g, dout -> 2 (3)
        return {"bytes": float((3 + 3 + 3 + 5 + (2 if case["masked"] else 0)) * n * es), "flops": 30.0 * n}
    if case["kind"] == "block":
        b, f = _block_work(case, 2)
        return {"bytes": float(b), "flops": float(f)}
    per = _block_work(case, 2 if case["kind"] == "train" else 1)
    times = case["layers"] * case["steps"]
    latents = (6 if case["kind"] == "train" else 8) * case["B"] * case["G"] ** 2 * case["hidden"] * es * case["steps"]
    return {"bytes": float(times * per[0] + latents), "flops": float(times * per[1])}


def tolerance(case):
    # four times what the path shows against 64 bits over the listed cases and some forty drawn ones
    if case["kind"] == "attn":
        return {"bf16": {"rel": 1.2e-2, "max": 0.18}, "fp16": {"rel": 1.4e-3, "max": 0.02},
                "fp32": {"rel": 3e-6, "max": 5e-5}}[case["dtype"]]
    if case["kind"] == "wrapper":
        return {"bf16": {"rel": 1.2e-2, "max": 0.06}, "fp16": {"rel": 1.6e-3, "max": 8e-3},
                "fp32": {"rel": 1e-6, "max": 4e-6}}[case["dtype"]]
    return {"block": {"rel": 3e-2, "max": 0.17}, "train": {"rel": 3e-2, "max": 0.4},
            "solve": {"rel": 2.4e-2, "max": 0.11}}[case["kind"]]


# -- the same values in 64 bits, in plain torch ------------------------------------------------------------------------


def _exact_attention(q, k, v):
    s = torch.matmul(q, k.transpose(-1, -2)) * q.shape[-1] ** -0.5
    return torch.matmul(torch.softmax(s, dim=-1), v)


def _exact_attn(case, seed):
    ts = _inputs(case, seed)
    B, H, L = case["B"], case["H"], case["L"]
    step = max(1, int(2**25 / (H * L * L)))  # boards at a time: a few L x L matrices in 64 bits each
    parts = []
    for b in range(0, B, step):
        q, k, v, do, *cot = (t[b:b + step].double() for t in ts)
        leaves = [t.detach().contiguous().requires_grad_(True) for t in (q, k, v, do)]
        o = _exact_attention(*leaves[:3])
        if case["order"] == 1:
            out = [o, *torch.autograd.grad(o, leaves[:3], leaves[3])]
        else:
            first = torch.autograd.grad(o, leaves[:3], leaves[3], create_graph=True)
            out = [o, *first, *torch.autograd.grad(first, leaves, cot)]
        parts.append([t.detach() for t in out])
        del o, out, leaves
    return [torch.cat(p) for p in zip(*parts)]


def _exact_rms_norm(x, eps=EPS):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps)


def _exact_wrapper(case, seed):
    ts = _inputs(case, seed)
    d = {n: t.double() if t is not None and t.is_floating_point() else t for n, t in ts.items()}
    z, g = d["z"].requires_grad_(True), d["g"].requires_grad_(True)
    v = _exact_rms_norm(z) + d["noise"] * d["sigma"]
    (dz,) = torch.autograd.grad(v, z, d["dv"])
    w = v.detach().requires_grad_(True)
    u = w - d["alpha"] * g
    out = u / u.square().mean(dim=(1, 2), keepdim=True).sqrt().clamp_min(EPS)
    if case["masked"]:
        out = torch.where(d["active"], out, z)
    wrt = (w, g, z) if case["masked"] else (w, g)
    return [v.detach(), dz, out.detach(), *torch.autograd.grad(out, wrt, d["dout"])]


def _exact_rotation(case):
    """cos and sin of every cell and head column: rows turn the first half of the head, columns the second."""
    G, D = case["G"], case["hidden"] // case["heads"]
    half = D // 2
    inv = 1.0 / (10000.0 ** (torch.arange(0, half, 2, dtype=torch.float32) / half))
    ang = torch.arange(G, dtype=torch.float32)[:, None] * inv[None, :]
    cos, sin = ang.cos().double().repeat(1, 2), ang.sin().double().repeat(1, 2)
    rows, cols = torch.arange(G).repeat_interleave(G), torch.arange(G).repeat(G)
    return torch.cat((cos[rows], cos[cols]), -1).cuda(), torch.cat((sin[rows], sin[cols]), -1).cuda()


def _exact_rotate(x, cos, sin):
    a, b, c, d = x.chunk(4, dim=-1)
    return x * cos + torch.cat((-b, a, -d, c), dim=-1) * sin


def _exact_block(case, cast, h):
    """``cast``: the block's weights as they enter its products (rounded to the dtype, in 64 bits)."""
    B, L, C = h.shape
    H = case["heads"]
    cos, sin = _exact_rotation(case)
    q, k, v = (t.view(B, L, H, C // H).transpose(1, 2) for t in F.linear(h, cast["qkv_proj"]).split(C, dim=-1))
    q, k = _exact_rotate(q, cos, sin), _exact_rotate(k, cos, sin)
    q = q * cast["log_logit_scale"].exp().view(1, H, 1, 1)
    y = _exact_attention(q, k, v).transpose(1, 2).reshape(B, L, C)
    h = _exact_rms_norm(h + F.linear(y, cast["o_proj"]))
    gate, up = F.linear(h, cast["gate_up_proj"]).chunk(2, dim=-1)
    return _exact_rms_norm(h + F.linear(F.silu(gate) * up, cast["down_proj"]))


def _rounded(case, model):
    """Every weight rounded to the case's dtype and then in 64 bits, by its name in the model."""
    dt = DTYPES[case["dtype"]]
    return {n: p.detach().to(dt).double().requires_grad_(True) for n, p in model.named_parameters()}


def _layer(weights, i):
    # layers.<i>.<part>.<name>[.weight]
    return {n.split(".")[3]: w for n, w in weights.items() if n.startswith("layers.%d." % i)}


def exact(case, seed):
    if case["kind"] == "attn":
        return _exact_attn(case, seed)
    if case["kind"] == "wrapper":
        return _exact_wrapper(case, seed)
    state = prepare(case, seed)
    model, z = state["model"], state["z"].double()
    weights = _rounded(case, model)
    if case["kind"] == "block":
        own = _layer(weights, 0)
        x = z.requires_grad_(True)
        y = _exact_block(case, own, x)
        (dx,) = torch.autograd.grad(y, x, state["dy"].double(), create_graph=True)
        order = [n.split(".")[1] for n, _ in model.layers[0].named_parameters()]
        second = torch.autograd.grad(dx, (x, *(own[n] for n in order)), state["c"].double())
        return [y.detach(), dx.detach(), *second]
    lm = state["decoder"].lm_head.weight.detach().to(DTYPES[case["dtype"]]).double().requires_grad_(True)
    x_emb = F.embedding(state["x"], weights["embed"])

    def total(u):
        h = u + x_emb
        for i in range(case["layers"]):
            h = _exact_block(case, _layer(weights, i), h)
        return F.linear(h.mean(dim=1), weights["energy_head.weight"]).squeeze(-1)

    if case["kind"] == "train":
        v = z.requires_grad_(True)
        for _ in range(case["steps"]):
            (g,) = torch.autograd.grad(total(v).sum(), v, create_graph=True)
            v = v - ALPHA * g
        loss = F.cross_entropy(F.linear(v, lm).reshape(-1, VOCAB), state["targets"].reshape(-1))
        names = list(weights)
        grads = torch.autograd.grad(loss, [*weights.values(), lm], allow_unused=True)
        return {"loss": loss.detach(), "grads": dict(zip([*names, "lm_head"], grads))}
    v = z
    for _ in range(case["steps"]):
        u = (_exact_rms_norm(v) + state["noise"].double()).detach().requires_grad_(True)
        (g,) = torch.autograd.grad(total(u).sum(), u)
        u = u.detach() - ALPHA * g
        v = u / u.square().mean(dim=(1, 2), keepdim=True).sqrt().clamp_min(EPS)
    with torch.no_grad():
        return {"logits": F.linear(v, lm), "z": v}
