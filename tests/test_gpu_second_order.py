"""Second derivatives, forward-mode derivatives and batched gradients through the patched ops on the
GPU: the native kernels record nothing and read tensors by address, so these must come from
differentiable ops.  Against float64 autograd on the CPU; bars as for the first derivatives, 1e-5
(fp32) and 1e-2 (16 bits)."""
from __future__ import annotations

import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu


def _second(fn, leaves, dy, v):
    """Gradients of <first gradients, v> with respect to dy, the input and the weight."""
    grads = torch.autograd.grad(fn(*leaves), leaves, dy, create_graph=True)
    total = sum((a * b).sum() for a, b in zip(grads, v))
    return list(grads) + list(torch.autograd.grad(total, (dy, leaves[0], leaves[1])))


def _compare(fn, shapes, out_shape, dtype, scale):
    import amd_tuned_torch  # noqa: F401
    g = torch.Generator().manual_seed(5)
    base = [(torch.randn(s, generator=g) * c).to(dtype) for s, c in zip(shapes, scale)]
    dy = torch.randn(out_shape, generator=g).to(dtype)
    v = [torch.randn(s, generator=g).to(dtype) for s in shapes]
    results = []
    for dev, to in (("cuda", dtype), ("cpu", torch.float64)):
        leaves = [t.to(dev, to).requires_grad_() for t in base]
        results.append(_second(fn, leaves, dy.to(dev, to).requires_grad_(), [t.to(dev, to) for t in v]))
    bar = 1e-5 if dtype == torch.float32 else 1e-2
    for i, (got, ref) in enumerate(zip(*results)):
        err = (got.detach().double().cpu() - ref.detach()).abs().max().item() / ref.abs().max().item()
        assert err <= bar, f"output {i}: {err}"


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("shape", [(2, 64, 9, 13), (2, 64, 8, 16)])
def test_group_norm(shape, dtype):
    _compare(lambda x, w, b: F.group_norm(x, 32, w, b, 1e-5), (shape, shape[1:2], shape[1:2]), shape,
             dtype, (1.0, 1.0, 1.0))


@pytest.mark.parametrize("ci,co,size", [(24, 40, (11, 13)), (32, 128, (16, 16))])
def test_conv2d(ci, co, size):
    _compare(lambda x, w, b: F.conv2d(x, w, b, padding=1), ((2, ci) + size, (co, ci, 3, 3), (co,)),
             (2, co) + size, torch.float16, (1.0, (2 / (9 * ci)) ** 0.5, 1.0))


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("channel_last", [False, True])
def test_conv1d(channel_last, dtype):
    """F.conv1d in both layouts and causal_conv1d_fn with SiLU."""
    from amd_tuned_torch.causal_conv1d import causal_conv1d_fn

    def lay(x):
        return x.transpose(1, 2).contiguous().transpose(1, 2) if channel_last else x

    def causal(x, w, b):
        if x.is_cuda:
            return causal_conv1d_fn(lay(x), w.squeeze(1), b, activation="silu")
        return F.silu(F.conv1d(x, w, b, padding=3, groups=32)[..., :x.shape[2]])
    shapes = ((2, 32, 67), (32, 1, 4), (32,))
    _compare(lambda x, w, b: F.conv1d(lay(x), w, b, padding=3, groups=32), shapes, (2, 32, 70), dtype, (1.0, 0.5, 0.1))
    _compare(causal, shapes, (2, 32, 67), dtype, (1.0, 0.5, 0.1))


def _bar(got, ref, dtype):
    err = (got.detach().double().cpu() - ref.detach()).abs().max().item() / ref.abs().max().item()
    assert err <= (1e-5 if dtype == torch.float32 else 1e-2), err


def _forward_cases():
    import amd_tuned_torch as att
    return {
        "group_norm_odd": ((2, 64, 9, 13), (64,), lambda x, w: F.group_norm(x, 32, w, None, 1e-5)),
        "group_norm": ((2, 64, 8, 16), (64,), lambda x, w: F.group_norm(x, 32, w, None, 1e-5)),
        "group_norm_silu": ((2, 64, 9, 13), (64,), lambda x, w: att.group_norm_silu(x, 32, w, None, 1e-5)),
        "conv2d": ((2, 24, 11, 13), (40, 24, 3, 3), lambda x, w: F.conv2d(x, w, padding=1)),
        "conv1d": ((2, 32, 67), (32, 1, 4), lambda x, w: F.conv1d(x, w, padding=3, groups=32)),
    }


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("name", ["group_norm_odd", "group_norm", "group_norm_silu", "conv2d", "conv1d"])
def test_forward_mode(name, dtype):
    """The tangent of a dual input, in a level and through torch.func.jvp, after a plain call has
    chosen the shape's kernel."""
    import torch.autograd.forward_ad as fwad
    shape, wshape, fn = _forward_cases()[name]
    g = torch.Generator().manual_seed(6)
    x, t = (torch.randn(shape, generator=g).to(dtype) for _ in range(2))
    w = (torch.randn(wshape, generator=g) * 0.3).to(dtype)
    ref = torch.func.jvp(lambda v: fn(v, w.double()), (x.double(),), (t.double(),))
    x, t, w = x.cuda(), t.cuda(), w.cuda()
    fn(x, w)
    with fwad.dual_level():
        got = fwad.unpack_dual(fn(fwad.make_dual(x, t), w))
    assert got.tangent is not None
    for pair in (got, torch.func.jvp(lambda v: fn(v, w), (x,), (t,))):
        for a, r in zip(pair, ref):
            _bar(a, r, dtype)


@pytest.mark.parametrize("silu", [False, True])
def test_forward_mode_channels_last_group_norm(silu):
    """No tangent is dropped in silence: what the unpatched ops do, a value or an error."""
    import amd_tuned_torch as att
    import torch.autograd.forward_ad as fwad
    stock_gn = att._dispatch._STOCK_F["group_norm"]
    x, t = (torch.randn(2, 128, 8, 9, device="cuda").contiguous(memory_format=torch.channels_last) for _ in range(2))

    def run(fn):
        with fwad.dual_level():
            try:
                y = fwad.unpack_dual(fn(fwad.make_dual(x, t)))
            except RuntimeError as e:
                return str(e)
            assert y.tangent is not None
            return y.tangent
    if silu:
        fn, stock = lambda v: att.group_norm_silu(v, 32), lambda v: F.silu(stock_gn(v, 32))
    else:
        fn, stock = lambda v: F.group_norm(v, 32), lambda v: stock_gn(v, 32)
    fn(x)
    a, b = run(fn), run(stock)
    assert a == b if isinstance(b, str) else torch.equal(a, b)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("name", ["group_norm_odd", "group_norm", "conv2d"])
def test_dual_and_batched_gradients(name, dtype):
    """Forward over reverse (the incoming gradient is dual) and is_grads_batched=True: dx and dw are
    linear in dy, so the tangents and the batch's entries are gradients of their own."""
    import torch.autograd.forward_ad as fwad
    shape, wshape, fn = _forward_cases()[name]
    g = torch.Generator().manual_seed(7)
    x, w = torch.randn(shape, generator=g).to(dtype), (torch.randn(wshape, generator=g) * 0.3).to(dtype)
    refs = [x.double().requires_grad_(), w.double().requires_grad_()]
    y_ref = fn(*refs)
    dy, t = (torch.randn(y_ref.shape, generator=g).to(dtype) for _ in range(2))
    ref_dy, ref_t = (torch.autograd.grad(y_ref, refs, d.double(), retain_graph=True) for d in (dy, t))
    leaves = [x.cuda().requires_grad_(), w.cuda().requires_grad_()]
    y = fn(*leaves)
    dy, t = dy.cuda(), t.cuda()
    with fwad.dual_level():
        got = [fwad.unpack_dual(v) for v in torch.autograd.grad(y, leaves, fwad.make_dual(dy, t), retain_graph=True)]
    batch = torch.autograd.grad(y, leaves, torch.stack([dy, t]), is_grads_batched=True)
    for i in range(2):
        assert got[i].tangent is not None
        for a, r in ((got[i].primal, ref_dy[i]), (got[i].tangent, ref_t[i]), (batch[i][0], ref_dy[i]),
                     (batch[i][1], ref_t[i])):
            _bar(a, r, dtype)
