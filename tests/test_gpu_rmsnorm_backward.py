"""The HIP RMSNorm backward against float64, at the edges of its row loop and row chunks."""

import pytest
import torch as t

from aiproj_amd.model import rmsnorm as rmsnorm_module
from aiproj_amd.model.rmsnorm import rmsnorm_forward

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,weight_dtype", [(t.bfloat16, t.bfloat16), (t.float16, t.float32), (t.float32, t.float32)])
@pytest.mark.parametrize("rows,d", [(1, 8), (3, 504), (5, 512), (4097, 520), (130, 2048), (9000, 1000), (7, 4096)])
def test_native_backward_against_float64(dtype, weight_dtype, rows, d):
    """Edges of the row loop (waves of 4 rows, 4096 waves) and of the 512-element chunks."""
    gen = t.Generator(device="cuda").manual_seed(rows + d)
    x, g = (t.randn(rows, d, generator=gen, device="cuda").to(dtype) for _ in range(2))
    w = (1 + 0.2 * t.randn(d, generator=gen, device="cuda")).to(weight_dtype)
    _, inv = rmsnorm_forward(x, w, 1e-5)
    dx, dw = rmsnorm_module._native_backward(x, w, inv, g)
    x64, w64, g64 = x.double(), w.double(), g.double()
    inv64 = 1 / t.sqrt(x64.square().mean(1, keepdim=True) + 1e-5)
    xhat, gw = x64 * inv64, g64 * w64
    want = inv64 * (gw - xhat * (gw * xhat).mean(1, keepdim=True)), (g64 * xhat).sum(0)
    # One rounding to the result's dtype (half an ulp) over float32 sums of up to 9000 terms.
    ulp = {t.bfloat16: 2.0 ** -8, t.float16: 2.0 ** -11, t.float32: 2e-6}
    for got, ref in zip((dx, dw), want):
        assert float((got.double() - ref).norm()) <= ulp[got.dtype] * float(ref.norm())


def test_native_backward_leaves_other_rows_to_pytorch():
    x = t.randn(6, 36, device="cuda")
    w = t.ones(36, device="cuda")
    assert rmsnorm_module._native_backward(x, w, t.ones(6, device="cuda"), x) is None       # not a multiple of 8
    x = t.randn(6, 65, device="cuda")[:, 1:]
    assert rmsnorm_module._native_backward(x, w.new_ones(64), t.ones(6, device="cuda"), x) is None   # unaligned rows


def test_batched_gradients_take_pytorch():
    """vmap over the backward (is_grads_batched) sees PyTorch operations, equal to one backward per gradient."""
    gen = t.Generator(device="cuda").manual_seed(3)
    x, w = t.randn(5, 64, generator=gen, device="cuda"), t.randn(64, generator=gen, device="cuda")
    grads = t.randn(3, 5, 64, generator=gen, device="cuda")
    x.requires_grad_(True)
    w.requires_grad_(True)
    out = rmsnorm_module.RMSNormFunction.apply(x, w, 1e-5)
    got = t.autograd.grad(out, (x, w), grads, retain_graph=True, is_grads_batched=True)
    for i in range(3):
        # float32 sums of 64 terms and fewer in two orders.
        for a, b in zip(got, t.autograd.grad(out, (x, w), grads[i], retain_graph=True)):
            assert float((a[i] - b).norm()) <= 1e-5 * float(b.norm())
