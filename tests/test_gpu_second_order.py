"""Second derivatives through the patched ops on the GPU: the native backward kernels record
nothing, so gradients taken with create_graph=True must come from differentiable ops.  Against
float64 autograd on the CPU; bars as for the first derivatives, 1e-5 (fp32) and 1e-2 (16 bits)."""
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
