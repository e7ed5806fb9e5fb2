"""Head sizes 80, 96 and 112 on the eight-wave prompt-attention kernel, over its persistent
workgroups, item edges and scales, against the oracle."""

import math

import numpy as np
import pytest
import torch as t

import oracle
from aiproj_amd.kernals.flash_attention import flash_attention_forward

pytestmark = pytest.mark.gpu

# One rounding of the output and of the probabilities to the type, as for head size 64.
TOLERANCE = {t.float16: 2e-3, t.bfloat16: 1.6e-2}


@t.inference_mode()
@pytest.mark.parametrize("dtype", [t.float16, t.bfloat16])
@pytest.mark.parametrize("head_dim", [80, 96, 112])
@pytest.mark.parametrize("sign", [1, -1])
def test_wide_kernel_head_sizes(dtype, head_dim, sign):
    lengths = [1, 16, 31, 33, 63, 64, 65, 127, 129, 191, 257, 300] * 2
    gen = t.Generator(device="cuda").manual_seed(head_dim)
    q, k, v = (t.randn(sum(lengths), h, head_dim, device="cuda", generator=gen).to(dtype) for h in (8, 2, 2))
    cu = t.tensor([0] + list(np.cumsum(lengths)), dtype=t.int32, device="cuda")
    scale = sign / math.sqrt(head_dim)
    out, lse = flash_attention_forward(q, k, v, cu, max(lengths), scale)
    want, want_lse = oracle.causal_varlen_attention(*(x.double().cpu().numpy() for x in (q, k, v)), cu.cpu().numpy(),
                                                    max(lengths), scale)
    tol = TOLERANCE[dtype]
    t.testing.assert_close(out.double().cpu(), t.from_numpy(want), rtol=tol, atol=tol)
    t.testing.assert_close(lse.double().cpu(), t.from_numpy(want_lse), rtol=1e-3, atol=1e-3)


@t.inference_mode()
@pytest.mark.parametrize("dtype", [t.float16, t.bfloat16])
@pytest.mark.parametrize("head_dim,scale", [(d, s) for d in (64, 80, 96, 112, 128) for s in (-0.1, 0.0)]
                         + [(72, 0.1), (88, 0.1), (104, 0.1), (120, -0.1)])
def test_any_scale(dtype, head_dim, scale):
    """What the wide kernel leaves to the general one, on its rows of 64 and of 128 dims: scales that are
    not positive, and the other multiples of 8."""
    lengths = [1, 63, 65, 130]
    gen = t.Generator(device="cuda").manual_seed(head_dim)
    q, k, v = (t.randn(sum(lengths), h, head_dim, device="cuda", generator=gen).to(dtype) for h in (8, 2, 2))
    cu = t.tensor([0] + list(np.cumsum(lengths)), dtype=t.int32, device="cuda")
    out, lse = flash_attention_forward(q, k, v, cu, max(lengths), scale)
    want, want_lse = oracle.causal_varlen_attention(*(x.double().cpu().numpy() for x in (q, k, v)), cu.cpu().numpy(),
                                                    max(lengths), scale)
    tol = TOLERANCE[dtype]
    t.testing.assert_close(out.double().cpu(), t.from_numpy(want), rtol=tol, atol=tol)
    t.testing.assert_close(lse.double().cpu(), t.from_numpy(want_lse), rtol=1e-3, atol=1e-3)


@t.inference_mode()
@pytest.mark.parametrize("dtype,half_ulp", [(t.float16, 2.0 ** -11), (t.bfloat16, 2.0 ** -8)])
@pytest.mark.parametrize("head_dim", [80, 96, 112])
def test_largest_probability_is_exact(dtype, half_ulp, head_dim):
    """The last of 65 keys exceeds the others (all 0) by up to 2^8, in a block of its own, and
    alone has values: its probability is 1 in 16 bits, so the output has one rounding (and
    float32 error, below 4e-6) and no second one from the probability."""
    sequences, hq = 96, 4
    gen = t.Generator(device="cuda").manual_seed(head_dim)
    q, k, v = (t.zeros(65 * sequences, h, head_dim, device="cuda", dtype=dtype) for h in (hq, 1, 1))
    last = t.arange(64, 65 * sequences, 65, device="cuda")
    scores = 5.5 * t.rand(sequences, hq, 1, device="cuda", generator=gen)
    q[last] = (scores / math.sqrt(head_dim)).expand(-1, -1, head_dim).to(dtype)
    k[last] = 1
    v[last] = (1 + t.rand(sequences, 1, head_dim, device="cuda", generator=gen)).to(dtype)
    cu = t.arange(0, 65 * sequences + 1, 65, dtype=t.int32, device="cuda")
    out, _ = flash_attention_forward(q, k, v, cu, 65, 1 / math.sqrt(head_dim))
    e = t.exp(q[last].double().sum(-1, keepdim=True) / math.sqrt(head_dim))
    t.testing.assert_close(out[last].double(), v[last].double() * (e / (64 + e)), rtol=half_ulp + 4e-6, atol=0)


@t.inference_mode()
@pytest.mark.parametrize("dtype,head_dim", [(t.float16, 80), (t.bfloat16, 112)])
@pytest.mark.parametrize("count,longest", [(1, 32), (1, 33), (1, 64), (1, 65), (64, 64), (65, 64)])
def test_short_prompts_around_the_two_kernels(dtype, head_dim, count, longest):
    """Groups of four q heads: few prompts of 33 to 64 tokens run on the general kernel, up to a workgroup
    of 32 rows per CU (two KV heads, 64 prompts on 256 CUs); others on the wide one."""
    lengths = [longest] + [1 + (i * 7) % longest for i in range(1, count)]
    gen = t.Generator(device="cuda").manual_seed(head_dim)
    q, k, v = (t.randn(sum(lengths), h, head_dim, device="cuda", generator=gen).to(dtype) for h in (8, 2, 2))
    cu = t.tensor([0] + list(np.cumsum(lengths)), dtype=t.int32, device="cuda")
    scale = 1 / math.sqrt(head_dim)
    out, lse = flash_attention_forward(q, k, v, cu, longest, scale)
    want, want_lse = oracle.causal_varlen_attention(*(x.double().cpu().numpy() for x in (q, k, v)), cu.cpu().numpy(),
                                                    longest, scale)
    tol = TOLERANCE[dtype]
    t.testing.assert_close(out.double().cpu(), t.from_numpy(want), rtol=tol, atol=tol)
    t.testing.assert_close(lse.double().cpu(), t.from_numpy(want_lse), rtol=1e-3, atol=1e-3)


@t.inference_mode()
@pytest.mark.parametrize("head_dim", [80, 96, 112])
@pytest.mark.parametrize("size", [1e4, 1e12, 1e30])
def test_scores_of_any_size(head_dim, size):
    """One element of q that decides every score: finite, and the value of the key with the largest
    score, whose weight is 1 (the next one is more than e^100 below)."""
    gen = t.Generator(device="cuda").manual_seed(head_dim)
    n = 300
    q, k, v = (t.randn(n, h, head_dim, device="cuda", generator=gen).to(t.bfloat16) for h in (8, 2, 2))
    q[:, :, 3] = size
    k[:, :, 3] = (1 + t.randperm(n, device="cuda", generator=gen) % 64)[:, None] / 16
    cu = t.tensor([0, n], dtype=t.int32, device="cuda")
    out, lse = flash_attention_forward(q, k, v, cu, n, 1 / math.sqrt(head_dim))
    assert bool(t.isfinite(out).all()) and bool(t.isfinite(lse).all())
    for row in (0, 1, 63, 64, 150, 299):
        kk = k[:row + 1, 0, 3].float()
        best = kk == kk.max()
        if size == 1e4 and int(best.sum()) > 1:
            continue                                   # there the other dims decide between equal keys
        want = v[:row + 1, 0].double()[best]
        low, high = want.amin(0) - 0.02, want.amax(0) + 0.02
        for h in range(4):
            assert bool(((out[row, h] >= low) & (out[row, h] <= high)).all())
