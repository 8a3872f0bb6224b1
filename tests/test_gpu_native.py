"""The native launchers (csrc/native.cpp) against the general route of ops.py and adamw.py: the
same bits and the same refusals over the forms of a call, and what an autograd Function would have
seen where a call without a graph passes it by."""

from __future__ import annotations

import pytest
import torch
from torch.autograd import forward_ad

from gpu_util import randn
from picotron_amd import _lib, ops
from picotron_amd.nn import RMSNorm
from picotron_amd.nn.triton_kernels import (
    adamw,
    triton_adamw_step,
    triton_apply_rotary_embedding,
    triton_clip_grad_norm_and_step,
    triton_cross_entropy,
    triton_rms_norm,
    triton_swiglu,
)

pytestmark = pytest.mark.gpu

DTYPES = [torch.float32, torch.float16, torch.bfloat16]


def _same(a, b):
    if isinstance(a, (tuple, list)):
        assert isinstance(b, (tuple, list)) and len(a) == len(b)
        for x, y in zip(a, b):
            _same(x, y)
        return
    if a is None or b is None:
        assert a is b
        return
    assert a.shape == b.shape and a.stride() == b.stride() and a.dtype == b.dtype and a.device == b.device
    assert torch.equal(a, b)


def _both(monkeypatch, call, native=None, raises=None):
    """The result of a call as it is and through the general route (or the type of the exception
    `raises`, which both then have to raise).  `native`: whether the first one's launches all took
    (True) or all left (False) the native route; None where the form decides."""

    taken = []
    launch = ops._launch

    def recording(*args):
        out = launch(*args)
        taken.append(out is not None)
        return out

    def attempt():
        if raises is None:
            return call()
        with pytest.raises(raises) as caught:
            call()
        return caught.type

    with monkeypatch.context() as m:
        m.setattr(ops, "_launch", recording)
        out = attempt()
        m.setattr(ops, "_launch", lambda *args: None)
        ref = attempt()
    if native is not None:
        assert taken and all(t is native for t in taken), taken
    if raises is not None:
        assert out is ref
    else:
        _same(out, ref)
    return out


def _layouts(shape, dtype, gpu, seed):
    """(tensor, the launchers take it) in the layouts that reach the launchers, of one shape and
    dtype; then another dtype and an empty tensor."""

    t = randn(shape, dtype, gpu, seed)
    yield t, True
    yield randn((*shape[:-1], shape[-1] + 3), dtype, gpu, seed + 1)[..., :-3], False
    yield randn(tuple(reversed(shape)), dtype, gpu, seed + 2).permute(*range(len(shape) - 1, -1, -1)), False
    yield randn((1,) * len(shape), dtype, gpu, seed + 3).expand(shape), False
    yield randn((t.numel() + 1,), dtype, gpu, seed + 4)[1:].view(shape), True
    yield t.float() if dtype != torch.float32 else t.bfloat16(), False
    yield t[:0], False


@pytest.mark.parametrize("dtype", DTYPES)
def test_norm_and_swiglu_forms(gpu, monkeypatch, dtype):
    shape = (5, 3, 70)
    w = randn((70,), dtype, gpu, 1, 0.1, 1.0)
    base = randn(shape, dtype, gpu, 2)
    _, rstd = ops.rmsnorm_fwd(base, w, 1e-5)
    for t, plain in _layouts(shape, dtype, gpu, 10):
        # a norm takes rows of any of its types; two inputs of one call have to match
        _both(monkeypatch, lambda: ops.rmsnorm_fwd(t, w, 1e-5), native=plain or t.dtype != dtype)
        pair = dict(native=plain) if t.shape == base.shape and t.dtype == dtype else dict(raises=ValueError)
        _both(monkeypatch, lambda: ops.residual_rmsnorm_fwd(base, t, w, 1e-5), **pair)
        _both(monkeypatch, lambda: ops.swiglu_fwd(base, t), **pair)
        if t.numel():  # a gradient has its output's shape
            for need in ((True, True), (True, False), (False, True), (False, False)):
                _both(monkeypatch, lambda: ops.rmsnorm_bwd(t, base, w, rstd, *need), native=plain and any(need))
                _both(monkeypatch, lambda: ops.swiglu_bwd(t, base, base, *need), native=plain)
            _both(monkeypatch, lambda: ops.residual_rmsnorm_bwd(t, None, base, w, rstd), native=plain)
            _both(monkeypatch, lambda: ops.residual_rmsnorm_bwd(base, t, base, w, rstd, need_dw=False), native=plain)
    for bad in (w[:-1], w.view(1, 70), w.cpu(), w[::2]):
        _both(monkeypatch, lambda: ops.rmsnorm_fwd(base, bad, 1e-5), raises=ValueError)
    _both(monkeypatch, lambda: ops.rmsnorm_fwd(base, w.double(), 1e-5), raises=TypeError)
    _both(monkeypatch, lambda: ops.swiglu_fwd(base, base[:, :2]), raises=ValueError)
    _both(monkeypatch, lambda: ops.rmsnorm_fwd(base.cpu(), w.cpu(), 1e-5), raises=ValueError)
    _both(monkeypatch, lambda: ops.rmsnorm_bwd(base, base, w, rstd.view(-1)[1:]), raises=ValueError)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("layout", ["interleaved", "rotate_half"])
def test_rope_forms(gpu, monkeypatch, dtype, layout):
    cos, sin = randn((9, 8), torch.float32, gpu, 1), randn((9, 8), torch.float32, gpu, 2)
    q = randn((2, 7, 4, 16), dtype, gpu, 3).transpose(1, 2)
    keys = [randn((2, 7, 2, 16), dtype, gpu, 4).transpose(1, 2), randn((2, 2, 7, 16), dtype, gpu, 5),
            randn((2, 2, 7, 20), dtype, gpu, 6)[..., 2:18], randn((1, 1, 1, 16), dtype, gpu, 7).expand(2, 2, 7, 16),
            None]
    bad = [randn((2, 2, 16, 7), dtype, gpu, 8).transpose(2, 3), randn((2, 2, 7, 14), dtype, gpu, 9)]
    for inverse in (False, True):
        for k in keys:
            _both(monkeypatch, lambda: ops.rope(q, cos, sin, layout=layout, inverse=inverse, x1=k), native=True)
        for k in bad:
            _both(monkeypatch, lambda: ops.rope(q, cos, sin, layout=layout, inverse=inverse, x1=k), raises=ValueError)
    for c, s in ((cos.double(), sin.double()), (cos[:, :4], sin[:, :4]), (cos.t(), sin.t())):
        _both(monkeypatch, lambda: ops.rope(q, c, s, layout=layout), raises=ValueError)
    _both(monkeypatch, lambda: ops.rope(q, cos[:3], sin[:3], layout=layout), raises=_lib.HipKernelError)
    strided = randn((16, 9), torch.float32, gpu, 10)[:8].t()
    _both(monkeypatch, lambda: ops.rope(q, strided, sin, layout=layout), native=False)
    _both(monkeypatch, lambda: ops.rope(q, cos, sin, layout="other"), raises=ValueError)


@pytest.mark.parametrize("dtype", DTYPES)
def test_cross_entropy_forms(gpu, monkeypatch, dtype):
    b, s, v = 3, 6, 41
    logits = randn((b, s, v), dtype, gpu, 1, 2.0)
    ids = torch.randint(0, v, (b, s), device=gpu)
    ids[1, 2] = -100
    wide = randn((b, s + 2, v + 7), dtype, gpu, 2, 2.0)[:, 1:-1, 3:-4]
    fp16 = dtype == torch.float16

    def loss_of(x, t, shift, write, form):
        """(loss, gradient) of one call on a copy with x's layout, with the backward at 3."""

        x = torch.empty_strided(x.shape, x.stride(), dtype=x.dtype, device=gpu).copy_(x) if form != "expanded" else x
        grad = ops.ce_grad_buffer(x, 2 if shift else 1) if write and form == "out" else None
        if shift:
            loss, ws = ops.cross_entropy_shifted(x, t, write_grad=write, grad=None if fp16 else grad,
                                                 next_targets=shift == 2)
        else:
            loss, ws = ops.cross_entropy(x, t, write_grad=write, grad=None if fp16 else grad)
        if not write:
            return loss, None
        out = x if grad is None else grad
        kw = dict(workspace=ws, logits=x if fp16 and grad is not None else None)
        go = torch.full((), 3.0, device=gpu)
        if shift:
            ops.cross_entropy_shifted_scale_grad(out, t, go, next_targets=shift == 2, **kw)
        else:
            ops.cross_entropy_scale_grad(out, t, go, **kw)
        return loss, out.clone()

    calls = [(logits, ids, 1), (wide, ids, 1), (logits, ids[:, 1:], 2), (wide, ids[:, 1:], 2),
             (logits.transpose(0, 1).contiguous().transpose(0, 1), ids, 1),
             (logits.view(-1, v), ids.view(-1), 0), (logits.transpose(1, 2), ids, 0),
             (wide.transpose(1, 2), ids, 0), (logits[:, 0], ids[:, 0], 0)]
    bad = [(logits.view(-1, v), ids.view(-1)[:5], 0), (logits, ids[:, :3], 1), (logits, ids.int(), 1),
           (logits.transpose(0, 2).contiguous(), ids, 1)]
    for write, form in ((False, "in"), (True, "in"), (True, "out")):
        for x, t, shift in calls:
            _both(monkeypatch, lambda: loss_of(x, t, shift, write, form), native=True)
        for x, t, shift in bad:
            _both(monkeypatch, lambda: loss_of(x, t, shift, write, form), raises=ValueError)
    expanded = logits[:1].expand(b, s, v)
    _both(monkeypatch, lambda: loss_of(expanded, ids, 1, True, "expanded"), raises=ValueError)
    for x in (logits, wide, expanded):  # the gradient buffer itself: same strides and phase
        got = ops.ce_grad_buffer(x, 2)
        if x is expanded:
            assert got is None
        else:
            assert got.stride() == x.stride() and (got.data_ptr() - x.data_ptr()) % 128 == 0


def _optimizer(gpu, seed, groups=1):
    params = [torch.nn.Parameter(randn((n,), torch.float32, gpu, seed + n, 0.1)) for n in (1, 5, 1024, 4097, 30_000)]
    params.append(torch.nn.Parameter(randn((8,), torch.float32, gpu, seed)))  # never has a gradient
    split = [params] if groups == 1 else [params[:2], params[2:5], params[5:]]
    return params, torch.optim.AdamW([dict(params=p, lr=1e-3 * (i + 1)) for i, p in enumerate(split)], weight_decay=0.1)


@pytest.mark.parametrize("groups", [1, 3])
@pytest.mark.parametrize("clip", [None, 0.05])
def test_adamw_scan_takes_the_same_steps(gpu, monkeypatch, groups, clip):
    """Steps through the native scan and through the general plan: the same parameters, moments,
    step counts and norms; the scan is used from the second step on, and steps aside for a group
    whose counts differ."""

    runs = []
    for native in (True, False):
        params, opt = _optimizer(gpu, 3, groups)
        norms, used = [], []
        with monkeypatch.context() as m:
            if not native:
                m.setattr(adamw, "_scan", lambda optimizer: None)
            for step in range(4):
                for i, p in enumerate(params[:-1]):
                    p.grad = randn(p.shape, torch.float32, gpu, 100 * step + i)
                if step == 3:
                    opt.state[params[2]]["step"] += 5.0
                if native:
                    used.append(adamw._scan(opt) is not None)
                if clip is None:
                    triton_adamw_step(opt)
                else:
                    norms.append(triton_clip_grad_norm_and_step(opt, clip))
        if native:
            assert used == [False, True, True, False]
            steps = [opt.state[p]["step"] for p in params[:-1]]
            assert all(s.dtype == torch.float32 and not s.is_cuda for s in steps)
            assert [float(s) for s in steps] == [4.0, 4.0, 9.0, 4.0, 4.0]
        runs.append((params, [opt.state[p] for p in params[:-1]], norms))
    for a, b in zip(*(r[0] for r in runs)):
        assert torch.equal(a, b)
    for a, b in zip(*(r[1] for r in runs)):
        assert all(torch.equal(a[k], b[k]) for k in ("step", "exp_avg", "exp_avg_sq"))
    for a, b in zip(*(r[2] for r in runs)):
        assert torch.equal(a, b)


def test_adamw_scan_leaves_the_unusual_to_the_plan(gpu):
    def ready():
        params, opt = _optimizer(gpu, 9)
        for p in params[:-1]:
            p.grad = torch.ones_like(p)
        triton_adamw_step(opt)
        assert adamw._scan(opt) is not None
        return params, opt

    params, opt = ready()
    params[3].grad = torch.ones(2 * 4097, device=gpu)[::2]
    assert adamw._scan(opt) is None
    params, opt = ready()
    opt.state[params[2]]["exp_avg"] = torch.zeros(3, device=gpu)
    assert adamw._scan(opt) is None
    with pytest.raises(adamw.TritonAdamWUnavailable):
        triton_adamw_step(opt)
    for key, value in (("exp_avg_sq", torch.zeros(1024, device=gpu, dtype=torch.float64)),
                       ("step", torch.tensor(1.0, device=gpu)), ("step", 1.0)):
        params, opt = ready()
        opt.state[params[2]][key] = value
        assert adamw._scan(opt) is None
    params, opt = ready()
    opt.param_groups[0]["capturable"] = True
    assert adamw._scan(opt) is None
    params, opt = ready()
    version = opt.state[params[0]]["step"]._version
    triton_adamw_step(opt)
    assert opt.state[params[0]]["step"]._version > version


def test_calls_without_a_graph(gpu):
    """Without a gradient the entry points skip the autograd Function; forward-mode derivatives,
    functorch transforms and tracing still meet what they met before."""

    x, w = randn((6, 40), torch.float32, gpu, 1), randn((40,), torch.float32, gpu, 2, 0.1, 1.0)
    norm = RMSNorm(40, use_triton_rmsnorm=True).to(gpu)
    with torch.no_grad():
        norm.weight.copy_(w)
        y = norm(x)
    _same(y, norm(x).detach())
    assert not y.requires_grad and norm(x).requires_grad
    with torch.inference_mode():
        _same(norm(x).clone(), y)
    norm.weight.requires_grad_(False)
    with pytest.warns(RuntimeWarning, match="PyTorch fallback"):  # a Function has no jvp here
        with forward_ad.dual_level():
            tangent = forward_ad.unpack_dual(norm(forward_ad.make_dual(x, torch.ones_like(x)))).tangent
    ref = torch.func.jvp(norm._eager, (x,), (torch.ones_like(x),))[1]
    torch.testing.assert_close(tangent, ref, rtol=1e-5, atol=1e-6)
    batched = torch.func.vmap(norm)(x)  # refused by a Function without setup_context: the formula
    torch.testing.assert_close(batched, y, rtol=1e-5, atol=1e-6)
    with torch.no_grad():
        cos = randn((6, 20), torch.float32, gpu, 4)
        for got, ref in ((triton_rms_norm(x, w, 1e-5), ops.rmsnorm_fwd(x, w, 1e-5)[0]),
                         (triton_swiglu(x, x), ops.swiglu_fwd(x, x)),
                         (triton_apply_rotary_embedding(x.view(1, 1, 6, 40), cos, cos), ops.rope(x.view(1, 1, 6, 40), cos, cos)[0]),
                         (triton_cross_entropy(x, torch.arange(6, device=gpu)), ops.cross_entropy(x, torch.arange(6, device=gpu))[0])):
            _same(got, ref)


def test_a_refused_launch_raises(gpu):
    # 2^22 columns are more than a row of the kernels holds
    x = torch.zeros((1, 1 << 22), device=gpu)
    with pytest.raises(_lib.HipKernelError):
        ops.rmsnorm_fwd(x, torch.ones(1 << 22, device=gpu), 1e-5)


def test_without_the_extension(gpu, monkeypatch):
    """Every call has its ctypes route when the extension could not be loaded."""

    x, w = randn((6, 40), torch.float32, gpu, 1), randn((40,), torch.float32, gpu, 2, 0.1, 1.0)
    t = torch.arange(6, device=gpu)

    def results():
        logits = x.clone().requires_grad_(True)
        loss = triton_cross_entropy(logits, t, inplace=False)
        params, opt = _optimizer(gpu, 5)
        for p in params[:-1]:
            p.grad = torch.ones_like(p)
        triton_adamw_step(opt)
        return (*ops.rmsnorm_fwd(x, w, 1e-5), ops.swiglu_fwd(x, x), loss, torch.autograd.grad(loss, logits)[0],
                triton_clip_grad_norm_and_step(opt, 0.1), *params)

    with_it = results()
    monkeypatch.setattr(_lib, "native", None)
    monkeypatch.setattr(_lib, "_launchers", {})
    _same(results(), with_it)


def test_writes_leave_lazily_cloned_tensors_alone(gpu):
    """What a call writes gets a storage of its own first (parameters, gradients, moments, step
    counts, logits and gradient buffers written in place)."""

    logits, t = randn((6, 41), torch.float32, gpu, 1), torch.arange(6, device=gpu)
    kept = logits.clone()
    x = torch._lazy_clone(logits)
    _, ws = ops.cross_entropy(x, t, write_grad=True)
    assert torch.equal(logits, kept) and not torch.equal(x, kept)
    scaled = torch._lazy_clone(x)
    before = x.clone()
    ops.cross_entropy_scale_grad(scaled, t, torch.full((), 2.0, device=gpu), workspace=ws)
    assert torch.equal(x, before) and torch.equal(scaled, 2 * before)

    params, opt = _optimizer(gpu, 7)
    for p in params[:-1]:
        p.grad = torch.ones_like(p)
    triton_adamw_step(opt)
    shared = []
    for p in params[:-1]:
        state = opt.state[p]
        shared += [p.data, p.grad, *state.values()]
        p.data, p.grad = torch._lazy_clone(p.data), torch._lazy_clone(p.grad)
        opt.state[p] = {k: torch._lazy_clone(v) for k, v in state.items()}
    kept = [v.clone() for v in shared]
    assert adamw._scan(opt) is not None
    triton_clip_grad_norm_and_step(opt, 0.05)
    _same(shared, kept)
    assert float(opt.state[params[0]]["step"]) == 2.0 and not torch.equal(params[0], shared[0])


def test_adamw_scan_outlives_what_a_hash_drops(gpu, monkeypatch):
    """The scan's dict lookups hash parameters in Python, where other threads run too: step tensors,
    gradients and states that go away there stay valid until the scan is done with them."""

    params, opt = _optimizer(gpu, 11)
    for p in params[:-1]:
        p.grad = torch.ones_like(p)
    triton_adamw_step(opt)
    states = [opt.state[p] for p in params[:-1]]
    hashes = []

    def dropping(self):
        hashes.append(id(self))
        self.grad = None  # the parameter's own gradient, which the scan has just read
        if len(hashes) == 2:
            states[0].clear()  # and the step count of the parameter before
        return id(self)

    with monkeypatch.context() as m:
        m.setattr(torch.Tensor, "__hash__", dropping)
        found = _lib.extension().adamw_scan([params[:-1]], opt.state, 1024)
    assert len(hashes) == 5 and found is not None
    steps = found[3][0][4]
    assert [float(s) for s in steps] == [1.0] * 5
    assert found[3][0][1] == 5
