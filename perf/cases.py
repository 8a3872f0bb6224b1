"""Cases that time the framework's kernels through its public entry points, as a user's training or
inference program calls them.

Five kernel families, each over the range that the modules accept in use: the norms, the SwiGLU
activation, the rotary embedding, the cross-entropy loss and the optimizer update, plus the three
activation kernels of one decode step.  ``listed()`` holds one case per kind of use; ``draw(rng)``
gives another case of the same ranges.  A training case is forward and backward (through autograd),
an inference case the forward alone under ``no_grad``.

Bytes in ``work()`` count every call of the pass by itself: a forward reads its inputs and writes
its outputs, the backward reads the incoming gradient and what the forward saved, and writes the
gradients.
"""

from __future__ import annotations

import math

import torch
from torch import Tensor

from picotron_amd.nn import RMSNorm, RotaryEmbedding
from picotron_amd.nn.triton_kernels import (
    CrossEntropyWithFallback,
    triton_adamw_step,
    triton_apply_rotary_embedding_pair,
    triton_clip_grad_norm_and_step,
    triton_rms_norm,
    triton_swiglu,
)

DTYPES = {"fp32": torch.float32, "fp16": torch.float16, "bf16": torch.bfloat16}
SIZES = {"fp32": 4, "fp16": 2, "bf16": 2}
EPS = 1e-5
IGNORED = -100
LOSS_SCALE = 65536.0
THETA = 500_000.0
ADAMW = dict(lr=3e-4, betas=(0.9, 0.95), eps=1e-8, weight_decay=0.1)
MAX_NORM = 1.0


def listed() -> list[dict]:
    return [
        # one decode step of a bf16 decoder for 4 sequences: the residual add + norm, the rotation
        # of the new query and key at their position, and the gated activation (smallest calls)
        dict(name="decode_step", kind="decode", batch=4, hidden=4096, heads=32, kv_heads=8, head_dim=128,
             intermediate=14336, position=777, dtype="bf16"),
        # the block norm of a large decoder in bf16 training, 16k tokens
        dict(name="norm_bf16", kind="norm", rows=16384, cols=4096, dtype="bf16", weight="bf16", train=True),
        # the decoder block's residual add + norm as mixed-precision training runs it: an fp32
        # residual stream and an fp32 weight, micro-batch 8 x 2048 tokens
        dict(name="residual_norm_fp32", kind="residual_norm", rows=16384, cols=2048, dtype="fp32",
             weight="fp32", train=True),
        # a hidden size that is no multiple of 8 and an odd number of tokens (packed batches)
        dict(name="norm_ragged", kind="norm", rows=16383, cols=1370, dtype="bf16", weight="bf16", train=True),
        # the MLP activation of a large decoder in bf16 training, 16k tokens
        dict(name="swiglu_bf16", kind="swiglu", rows=16384, cols=14336, dtype="bf16", train=True),
        # the activation at a small decoder's width (2/3 of 4 x 1024) over an odd packed batch, fp16
        dict(name="swiglu_ragged", kind="swiglu", rows=16383, cols=2731, dtype="fp16", train=True),
        # grouped-query attention's rotation in training, on the (B, S, H, D) memory of projections
        dict(name="rope_bf16", kind="rope", batch=8, seq=2048, heads=32, kv_heads=8, head_dim=128,
             layout="rotate_half", dtype="bf16", train=True),
        # the notebook demo's rotation: interleaved pairs, 2 heads of 10 over 1 key head, fp16
        dict(name="rope_demo_fp16", kind="rope", batch=32, seq=256, heads=2, kv_heads=1, head_dim=10,
             layout="interleaved", dtype="fp16", train=True),
        # the train loop's loss call at a large vocabulary, bf16 logits
        dict(name="loss_bf16", kind="loss", batch=4, seq=2049, vocab=128256, dtype="bf16", ignored=0.0, train=True),
        # the notebook demo's loss call: GPT-2's vocabulary (rows start anywhere in a line), fp16
        # under a loss scale
        dict(name="loss_demo_fp16", kind="loss", batch=32, seq=256, vocab=50257, dtype="fp16", ignored=0.0, train=True),
        # the loss of a byte-level model (256 bytes and 4 special tokens), a third of the targets
        # masked as in instruction tuning
        dict(name="loss_bytes", kind="loss", batch=16, seq=1025, vocab=260, dtype="bf16", ignored=0.33, train=True),
        # the optimizer update of a 1.04e9-parameter decoder: clip the gradient norm, step
        dict(name="adamw_clip", kind="adamw", layers=16, hidden=2048, intermediate=8192, kv=512, vocab=32000,
             clip=True),
    ]


# ---------------------------------------------------------------------- drawn cases


def _log(rng, low: int, high: int) -> int:
    return max(low, min(high, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng) -> dict:
    kind = rng.choice(["decode", "norm", "norm", "residual_norm", "swiglu", "rope", "loss", "loss", "adamw"])
    dtype = rng.choice(["fp32", "fp16", "bf16", "bf16"])
    train = rng.random() < 0.8
    if kind == "decode":
        head_dim = rng.choice([16, 64, 80, 128])
        kv_heads = rng.choice([1, 2, 4, 8])
        heads = kv_heads * rng.choice([1, 2, 4, 8])
        return dict(kind=kind, batch=_log(rng, 1, 256), hidden=heads * head_dim, heads=heads, kv_heads=kv_heads,
                    head_dim=head_dim, intermediate=_log(rng, 64, 28672), position=_log(rng, 1, 8000), dtype=dtype)
    if kind in ("norm", "residual_norm"):
        cols = rng.choice([576, 768, 960, 1024, 2048, 4096, 5120, 8192, _log(rng, 20, 8192), _log(rng, 20, 8192)])
        rows = _log(rng, 1, max(2, min(65536, 16384 * 4096 // cols)))
        return dict(kind=kind, rows=rows, cols=cols, dtype=dtype, weight=rng.choice([dtype, "fp32"]), train=train)
    if kind == "swiglu":
        cols = rng.choice([1536, 2560, 5632, 8192, 14336, _log(rng, 64, 14336), _log(rng, 64, 14336)])
        return dict(kind=kind, rows=_log(rng, 1, 8192), cols=cols, dtype=dtype, train=train)
    if kind == "rope":
        kv_heads = rng.choice([1, 2, 4, 8])
        seq = _log(rng, 8, 4096)
        return dict(kind=kind, batch=_log(rng, 1, max(2, 8192 // seq)), seq=seq, heads=kv_heads * rng.choice([1, 2, 4]),
                    kv_heads=kv_heads, head_dim=rng.choice([8, 10, 16, 64, 64, 80, 96, 128, 128]),
                    layout=rng.choice(["interleaved", "rotate_half"]), dtype=dtype, train=train)
    if kind == "loss":
        vocab = rng.choice([32000, 32001, 50257, 50304, 65536, 128256, _log(rng, 64, 128256), _log(rng, 64, 128256)])
        most = 5 * 10**8 // (2 if dtype == "fp32" else 1) // vocab  # rows
        seq = _log(rng, 16, max(17, min(2049, most)))
        return dict(kind=kind, batch=_log(rng, 1, max(2, min(64, most // seq))), seq=seq, vocab=vocab, dtype=dtype,
                    ignored=rng.choice([0.0, 0.0, 0.33]), train=train)
    hidden = 64 * _log(rng, 1, 24)
    return dict(kind=kind, layers=_log(rng, 1, 16), hidden=hidden, intermediate=hidden * rng.choice([2, 3, 4]) + rng.choice([0, 0, 1]),
                kv=hidden // rng.choice([1, 2, 4]), vocab=_log(rng, 64, 50257), clip=rng.random() < 0.5)


# ---------------------------------------------------------------------- inputs


def _randn(shape, dtype: torch.dtype, gen: torch.Generator, scale: float = 1.0) -> Tensor:
    """Normal values made in slices, so that a large 16-bit tensor needs no fp32 copy of itself."""

    out = torch.empty(shape, dtype=dtype, device="cuda")
    flat = out.view(-1)
    for part in flat.split(1 << 28):
        part.copy_(torch.randn(part.numel(), generator=gen, device="cuda").mul_(scale))
    return out


def _tables(seq: int, head_dim: int) -> tuple[Tensor, Tensor]:
    inverse = 1.0 / (THETA ** (torch.arange(0, head_dim, 2, device="cuda", dtype=torch.float32) / head_dim))
    angles = torch.outer(torch.arange(seq, device="cuda", dtype=torch.float32), inverse)
    return angles.cos(), angles.sin()


def _adamw_shapes(case: dict) -> list[tuple[int, ...]]:
    """The parameters of a decoder with tied embeddings."""

    h, i, kv = case["hidden"], case["intermediate"], case["kv"]
    shapes: list[tuple[int, ...]] = [(case["vocab"], h)]
    for _ in range(case["layers"]):
        shapes += [(h,), (h, h), (kv, h), (kv, h), (h, h), (h,), (i, h), (i, h), (h, i)]
    return shapes + [(h,)]


def _adamw_inputs(case: dict, seed: int) -> tuple[dict[str, Tensor], list[tuple[int, tuple[int, ...]]]]:
    """Flat parameter, gradient and moment buffers (tensors padded to 64 elements) and each tensor's
    place in them, as a data-parallel trainer keeps them."""

    gen = torch.Generator(device="cuda").manual_seed(seed)
    places, total = [], 0
    for shape in _adamw_shapes(case):
        places.append((total, shape))
        total += (math.prod(shape) + 63) // 64 * 64
    flat = {"p": _randn((total,), torch.float32, gen, 0.02), "g": _randn((total,), torch.float32, gen, 1e-3),
            "m": _randn((total,), torch.float32, gen, 1e-4), "v": _randn((total,), torch.float32, gen, 1e-3).square_()}
    end = 0
    for offset, shape in [*places, (total, (0,))]:
        for t in flat.values():
            t[end:offset] = 0.0  # padding
        end = offset + math.prod(shape)
    return flat, places


def prepare(case: dict, seed: int) -> dict:
    kind = case["kind"]
    gen = torch.Generator(device="cuda").manual_seed(seed)
    s = dict(case)
    if kind == "adamw":
        flat, places = _adamw_inputs(case, seed)
        view = lambda t, o, shape: t[o:o + math.prod(shape)].view(shape)  # noqa: E731
        params = []
        for o, shape in places:
            p = torch.nn.Parameter(view(flat["p"], o, shape))
            p.grad = view(flat["g"], o, shape)
            params.append(p)
        optimizer = torch.optim.AdamW(params, **ADAMW)
        for p, (o, shape) in zip(params, places):  # a run under way: state from a checkpoint
            optimizer.state[p] = {"step": torch.tensor(100.0), "exp_avg": view(flat["m"], o, shape),
                                  "exp_avg_sq": view(flat["v"], o, shape)}
        s.update(flat=flat, optimizer=optimizer)
        return s
    dtype = DTYPES[case["dtype"]]
    if kind == "decode":
        b, h = case["batch"], case["hidden"]
        norm = RMSNorm(h, EPS, use_triton_rmsnorm=True).to("cuda", dtype)
        with torch.no_grad():
            norm.weight.copy_(1 + 0.1 * torch.randn(h, generator=gen, device="cuda"))
        cos, sin = _tables(case["position"] + 1, case["head_dim"])
        s.update(norm=norm, x=_randn((b, 1, h), dtype, gen), residual=_randn((b, 1, h), dtype, gen), cos=cos, sin=sin,
                 q=_randn((b, 1, case["heads"], case["head_dim"]), dtype, gen).transpose(1, 2),
                 k=_randn((b, 1, case["kv_heads"], case["head_dim"]), dtype, gen).transpose(1, 2),
                 gate=_randn((b, 1, case["intermediate"]), dtype, gen),
                 up=_randn((b, 1, case["intermediate"]), dtype, gen))
        return s
    train = case["train"]
    if kind in ("norm", "residual_norm"):
        rows, cols = case["rows"], case["cols"]
        norm = RMSNorm(cols, EPS, use_triton_rmsnorm=True).to("cuda", DTYPES[case["weight"]])
        with torch.no_grad():
            norm.weight.copy_(1 + 0.1 * torch.randn(cols, generator=gen, device="cuda"))
        s.update(norm=norm, x=_randn((rows, cols), dtype, gen).requires_grad_(train))
        if kind == "residual_norm":
            s.update(residual=_randn((rows, cols), dtype, gen).requires_grad_(train))
        if train:
            s.update(dy=_randn((rows, cols), dtype, gen, 0.1))
            if kind == "residual_norm":
                s.update(dh=_randn((rows, cols), dtype, gen, 0.1))
    elif kind == "swiglu":
        shape = (case["rows"], case["cols"])
        s.update(gate=_randn(shape, dtype, gen).requires_grad_(train), up=_randn(shape, dtype, gen).requires_grad_(train))
        if train:
            s.update(dy=_randn(shape, dtype, gen, 0.1))
    elif kind == "rope":
        b, n, d = case["batch"], case["seq"], case["head_dim"]
        rope = RotaryEmbedding(d, THETA, use_triton_rope=True, layout=case["layout"])
        make = lambda heads, scale: _randn((b, n, heads, d), dtype, gen, scale).transpose(1, 2)  # noqa: E731
        s.update(rope=rope, q=make(case["heads"], 1.0).requires_grad_(train), k=make(case["kv_heads"], 1.0).requires_grad_(train))
        with torch.no_grad():
            rope(s["q"][:1], s["k"][:1])  # the module's angle tables exist after a model's first step
        if train:
            s.update(dq=make(case["heads"], 0.1), dk=make(case["kv_heads"], 0.1))
    elif kind == "loss":
        b, n, v = case["batch"], case["seq"], case["vocab"]
        ids = torch.randint(0, v, (b, n), generator=gen, device="cuda")
        if case["ignored"]:
            ids = ids.masked_fill(torch.rand((b, n), generator=gen, device="cuda") < case["ignored"], IGNORED)
            ids[0, 1] = 0  # at least one target
        s.update(loss=CrossEntropyWithFallback(use_triton=True), ids=ids,
                 logits=_randn((b, n, v), dtype, gen, 2.0).requires_grad_(train))
    return s


# ---------------------------------------------------------------------- one pass


def run(s: dict):
    kind = s["kind"]
    if kind == "decode":
        with torch.no_grad():
            h, y = s["norm"].add_and_norm(s["x"], s["residual"])
            p = s["position"]
            q, k = triton_apply_rotary_embedding_pair(s["q"], s["k"], s["cos"][p:p + 1], s["sin"][p:p + 1], layout="rotate_half")
            return [h, y, q, k, triton_swiglu(s["gate"], s["up"])]
    if kind == "norm":
        norm = s["norm"]
        if not s["train"]:
            with torch.no_grad():
                return [norm(s["x"])]
        y = triton_rms_norm(s["x"], norm.weight, norm.eps)
        return [y.detach(), *torch.autograd.grad(y, [s["x"], norm.weight], s["dy"])]
    if kind == "residual_norm":
        norm = s["norm"]
        if not s["train"]:
            with torch.no_grad():
                return list(norm.add_and_norm(s["x"], s["residual"]))
        h, y = norm.add_and_norm(s["x"], s["residual"])
        dx, dw = torch.autograd.grad([h, y], [s["x"], norm.weight], [s["dh"], s["dy"]])
        return [h.detach(), y.detach(), dx, dw]
    if kind == "swiglu":
        if not s["train"]:
            with torch.no_grad():
                return [triton_swiglu(s["gate"], s["up"])]
        y = triton_swiglu(s["gate"], s["up"])
        return [y.detach(), *torch.autograd.grad(y, [s["gate"], s["up"]], s["dy"])]
    if kind == "rope":
        if not s["train"]:
            with torch.no_grad():
                return list(s["rope"](s["q"], s["k"]))
        q, k = s["rope"](s["q"], s["k"])
        return [q.detach(), k.detach(), *torch.autograd.grad([q, k], [s["q"], s["k"]], [s["dq"], s["dk"]])]
    if kind == "loss":
        logits, ids = s["logits"], s["ids"]
        if not s["train"]:
            with torch.no_grad():
                return [s["loss"](logits[:, :-1, :].transpose(1, 2), ids[:, 1:])]
        loss = s["loss"](logits[:, :-1, :].transpose(1, 2), ids[:, 1:])
        scaled = loss * LOSS_SCALE if s["dtype"] == "fp16" else loss
        return [loss.detach(), *torch.autograd.grad(scaled, [logits])]
    if s["clip"]:
        total = triton_clip_grad_norm_and_step(s["optimizer"], MAX_NORM)
        return [total, s["flat"]["g"], s["flat"]["p"], s["flat"]["m"], s["flat"]["v"]]
    triton_adamw_step(s["optimizer"])
    return [s["flat"]["p"], s["flat"]["m"], s["flat"]["v"]]


# ---------------------------------------------------------------------- what a pass needs


def work(case: dict) -> dict:
    kind = case["kind"]
    if kind == "adamw":
        n = sum(math.prod(shape) for shape in _adamw_shapes(case))
        # the norm reads the gradients; the step reads p, g, m, v and writes p, m, v (and the
        # clipped g)
        return {"bytes": 4 * n * (9 if case["clip"] else 7), "flops": 20 * n}
    e = SIZES[case["dtype"]]
    if kind == "decode":
        n = case["batch"] * (4 * case["hidden"] + 2 * (case["heads"] + case["kv_heads"]) * case["head_dim"] + 3 * case["intermediate"])
        return {"bytes": n * e + case["hidden"] * e + 4 * case["head_dim"], "flops": 8 * n}
    train = case["train"]
    if kind in ("norm", "residual_norm"):
        n, w = case["rows"] * case["cols"], case["cols"] * SIZES[case["weight"]]
        streams = (5 if train else 2) if kind == "norm" else (8 if train else 4)
        return {"bytes": streams * n * e + (3 if train else 1) * w + (2 if train else 1) * 4 * case["rows"],
                "flops": (14 if train else 5) * n}
    if kind == "swiglu":
        n = case["rows"] * case["cols"]
        return {"bytes": (8 if train else 3) * n * e, "flops": (16 if train else 6) * n}
    if kind == "rope":
        n = case["batch"] * case["seq"] * (case["heads"] + case["kv_heads"]) * case["head_dim"]
        return {"bytes": (4 if train else 2) * n * e + (2 if train else 1) * 4 * case["seq"] * case["head_dim"],
                "flops": (6 if train else 3) * n}
    b, n, v = case["batch"], case["seq"], case["vocab"]
    logits = b * (n - 1) * v
    if not train:
        return {"bytes": logits * e + 8 * b * n, "flops": 5 * logits}
    # the gradient covers all positions; fp16 reads the logits again in the backward, where the
    # loss scale arrives
    return {"bytes": (2 if case["dtype"] == "fp16" else 1) * logits * e + b * n * v * e + 16 * b * n, "flops": 8 * logits}


def tolerance(case: dict):
    kind = case["kind"]
    # about four times the error against 64 bits: one rounding to the storage type (bf16 1.7e-3,
    # fp16 2.1e-4 of the 2-norm; a norm of a rounded sum 2.5e-3) and the fp32 sums (2e-7).  The
    # loss gradient's norm is mostly the target elements' (bf16 4e-5 to 1.1e-3).
    if kind == "adamw":
        return {"rel": 4e-7}
    if kind == "loss":
        return {"rel": {"fp32": 2e-6, "fp16": 8e-4, "bf16": 4.5e-3}[case["dtype"]]}
    return {"rel": {"fp32": 2e-6, "fp16": 1e-3, "bf16": 8e-3}[case["dtype"]]}


# ---------------------------------------------------------------------- 64-bit results


def _rotate(x: Tensor, cos: Tensor, sin: Tensor, layout: str) -> Tensor:
    x, cos, sin = x.double(), cos.double(), sin.double()
    if layout == "interleaved":
        a, b = x[..., 0::2], x[..., 1::2]
        return torch.stack((a * cos - b * sin, a * sin + b * cos), -1).flatten(-2)
    a, b = x.chunk(2, -1)
    return torch.cat((a * cos - b * sin, a * sin + b * cos), -1)


def _norm64(h: Tensor, w: Tensor) -> tuple[Tensor, Tensor]:
    r = torch.rsqrt(h.square().mean(-1, keepdim=True) + EPS)
    return h * r * w, r


def exact(case: dict, seed: int):
    s, kind = prepare(case, seed), case["kind"]
    with torch.no_grad():
        if kind == "adamw":
            return _exact_adamw(case, s)
        if kind == "decode":
            h = s["x"].double() + s["residual"].double()
            y, _ = _norm64(h, s["norm"].weight.double())
            c, n = s["cos"][-1:], s["sin"][-1:]
            gate, up = s["gate"].double(), s["up"].double()
            return [h, y, _rotate(s["q"], c, n, "rotate_half"), _rotate(s["k"], c, n, "rotate_half"), gate * torch.sigmoid(gate) * up]
        if kind in ("norm", "residual_norm"):
            w, h = s["norm"].weight.double(), s["x"].double()
            if kind == "residual_norm":
                h = (h + s["residual"].double()).to(s["x"].dtype).double()  # stored in the storage type
            y, r = _norm64(h, w)
            out = [y] if kind == "norm" else [h, y]
            if case["train"]:
                g = s["dy"].double()
                dw = (g * h * r).sum(0)
                g = g * w
                dx = r * (g - h * r.square() * (g * h).mean(-1, keepdim=True))
                out += [dx if kind == "norm" else dx + s["dh"].double(), dw]
            return out
        if kind == "swiglu":
            gate, up = s["gate"].double(), s["up"].double()
            sig = torch.sigmoid(gate)
            if not case["train"]:
                return [gate * sig * up]
            d = s["dy"].double()
            return [gate * sig * up, d * up * sig * (1 + gate * (1 - sig)), d * gate * sig]
        if kind == "rope":
            cos, sin = _tables(case["seq"], case["head_dim"])
            out = [_rotate(s["q"], cos, sin, case["layout"]), _rotate(s["k"], cos, sin, case["layout"])]
            if case["train"]:
                out += [_rotate(s["dq"], cos, -sin, case["layout"]), _rotate(s["dk"], cos, -sin, case["layout"])]
            return out
        return _exact_loss(case, s)


def _exact_loss(case: dict, s: dict):
    logits, targets = s["logits"].detach(), s["ids"][:, 1:]
    kept = int((targets != IGNORED).sum())
    scale = LOSS_SCALE if case["dtype"] == "fp16" else 1.0
    grad = torch.zeros(logits.shape, dtype=torch.float64, device="cuda") if case["train"] else None
    total = torch.zeros((), dtype=torch.float64, device="cuda")
    step = max(1, (1 << 27) // case["vocab"])
    for b in range(case["batch"]):
        for t in range(0, case["seq"] - 1, step):
            tgt = targets[b, t:t + step]
            keep = (tgt != IGNORED)
            at = tgt.clamp_min(0)[:, None]
            logp = torch.log_softmax(logits[b, t:t + tgt.numel()].double(), -1)
            total -= (logp.gather(1, at)[:, 0] * keep).sum()
            if grad is not None:
                p = logp.exp_()
                p.scatter_add_(1, at, torch.full(at.shape, -1.0, dtype=torch.float64, device="cuda"))
                grad[b, t:t + tgt.numel()] = p * (keep[:, None] * (scale / kept))
    loss = total / kept
    return [loss] if grad is None else [loss, grad]


def _exact_adamw(case: dict, s: dict):
    flat = s["flat"]
    total = torch.zeros((), dtype=torch.float64, device="cuda")
    for part in flat["g"].split(1 << 28):
        total += part.double().square().sum()
    total = total.sqrt()
    coef = torch.clamp(MAX_NORM / (total + 1e-6), max=1.0) if case["clip"] else 1.0
    g, p, m, v = (flat[k].double() for k in "gpmv")
    g *= coef
    b1, b2 = ADAMW["betas"]
    m.lerp_(g, 1 - b1)
    v.mul_(b2).addcmul_(g, g, value=1 - b2)
    p.mul_(1 - ADAMW["lr"] * ADAMW["weight_decay"])
    p.addcdiv_(m, (v.sqrt() / math.sqrt(1 - b2**101)).add_(ADAMW["eps"]), value=-ADAMW["lr"] / (1 - b1**101))
    return [total, g, p, m, v] if case["clip"] else [p, m, v]
