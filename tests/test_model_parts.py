"""What the decoder model's shortcuts must see: replaced rotations, biases, other widths. On the
CPU, with the attention and the cache replaced by recorders."""

import types

import pytest
import torch as t

from aiproj_amd import _native
from aiproj_amd.model import transformer
from aiproj_amd.model.transformer import Attention, ModelConfig, RoPE, RowLinear, StepMeta, SwiGLU

CFG = ModelConfig(d_model=32, num_q_heads=4, num_kv_heads=2, head_dim=8, d_ff=16, max_seq_len=16)


class Cache:
    def append_kv(self, blocks, offsets, k, v):
        self.k, self.v = k, v


class Doubling(RoPE):
    """A rotation that is not the base one, in place as `apply_` is."""

    def apply_(self, x, positions, heads):
        x[:, :heads * self.head_dim] *= 2
        return x


class Only(t.nn.Module):
    def apply_(self, x, positions, heads):
        x[:, :heads * CFG.head_dim] *= 2
        return x


def replaced(kind):
    if kind == "subclass":
        return Doubling(CFG.head_dim, CFG.max_seq_len, 10000.0)
    if kind == "other module":
        return Only()
    rope = RoPE(CFG.head_dim, CFG.max_seq_len, 10000.0)
    rope.apply_ = types.MethodType(Doubling.apply_, rope)
    return rope


def attend(attn, mode, monkeypatch, h):
    """(q, k) that the attention sees."""
    seen, cache = {}, Cache()

    def prompt(q, k, v, *rest):
        seen["qk"] = q.clone(), k.clone()
        return q, None

    def step(q, k, v, *rest):
        seen["qk"] = q.clone(), k.clone()
        return q

    monkeypatch.setattr(transformer, "flash_attention_forward", prompt)
    monkeypatch.setattr(transformer, "append_decode_attention", step)
    ctx = types.SimpleNamespace(physical_blocks=None, block_offsets=None)
    attn(h, StepMeta(mode, t.arange(len(h)), ctx, t.tensor([0, len(h)]), len(h)), cache)
    return seen["qk"]


@t.no_grad()
@pytest.mark.parametrize("mode", ["prefill", "decode"])
@pytest.mark.parametrize("kind", ["subclass", "other module", "instance"])
def test_a_replaced_rotation_is_used(mode, kind, monkeypatch):
    attn = Attention(CFG)
    attn.rope = replaced(kind)
    # As if the projection's kernel took the rows: a replaced rotation must not get there.
    monkeypatch.setattr(transformer, "_takes_skinny", lambda x, w: x.shape[-1] == w.shape[1])
    monkeypatch.setattr(transformer, "_skinny", lambda entry, x, w, columns, *more: x @ w.T)
    h = t.randn(5, CFG.d_model)
    q, k = attend(attn, mode, monkeypatch, h)
    want = h @ attn.qkv_proj.weight.T
    t.testing.assert_close(q, 2 * want[:, :32].view(5, 4, 8))
    t.testing.assert_close(k, 2 * want[:, 32:48].view(5, 2, 8))


@t.no_grad()
@pytest.mark.parametrize("shape", [(5, 48), (5, 63), (5, 65), (5, 96), (1, 5, 64)])
def test_rows_of_another_width_do_not_reach_the_split(shape, monkeypatch):
    """A projection replaced by one of another width or rank: the kernel would read past its rows.
    It is not called; the views of the separate route judge the rows, as before."""
    def called():
        raise AssertionError("the kernel was called")

    monkeypatch.setattr(_native, "require_gpu", lambda *x, what: x[0].device)
    monkeypatch.setattr(_native, "lib", called)
    assert RoPE(8, 16, 10000.0).split(t.empty(shape), t.arange(5), 4, 2) is None


@t.no_grad()
@pytest.mark.parametrize("mode", ["prefill", "decode"])
def test_an_assigned_bias_is_added(mode, monkeypatch):
    """RowLinear is an nn.Linear: a bias that a program gives it counts, also where a decode step's
    projection would be done by the rotating or the gated kernel."""
    def kernel(*args):
        raise AssertionError("the kernel adds no bias")

    monkeypatch.setattr(transformer, "_takes_skinny", lambda x, w: True)
    monkeypatch.setattr(transformer, "_skinny", kernel)
    x = t.randn(5, CFG.d_model)
    layer = RowLinear(CFG.d_model, 24)
    layer.bias = t.nn.Parameter(t.randn(24))
    assert t.equal(layer(x), t.nn.functional.linear(x, layer.weight, layer.bias))

    attn = Attention(CFG)
    attn.rope = Doubling(CFG.head_dim, CFG.max_seq_len, 10000.0)
    for proj in (attn.qkv_proj, attn.o_proj):
        proj.bias = t.nn.Parameter(t.randn(proj.out_features))
    q, _ = attend(attn, mode, monkeypatch, x)
    t.testing.assert_close(q.flatten(1), 2 * (x @ attn.qkv_proj.weight.T + attn.qkv_proj.bias)[:, :32])

    ffn = SwiGLU(CFG)
    for proj in (ffn.gate_up, ffn.down):
        proj.bias = t.nn.Parameter(t.randn(proj.out_features))
    monkeypatch.setattr(transformer, "silu_mul", lambda gu, n: t.nn.functional.silu(gu[:, :n]) * gu[:, n:])
    gate, up = (x @ ffn.gate_up.weight.T + ffn.gate_up.bias).chunk(2, -1)
    t.testing.assert_close(ffn(x), (t.nn.functional.silu(gate) * up) @ ffn.down.weight.T + ffn.down.bias)
    attn.rope = RoPE(CFG.head_dim, CFG.max_seq_len, 10000.0)
    monkeypatch.setattr(RoPE, "split", lambda self, qkv, *rest: None)
    monkeypatch.setattr(RoPE, "apply_", Doubling.apply_)
    q, _ = attend(attn, mode, monkeypatch, x)
    t.testing.assert_close(q.flatten(1), 2 * (x @ attn.qkv_proj.weight.T + attn.qkv_proj.bias)[:, :32])


@t.no_grad()
def test_more_rows_than_the_kernel_takes_cost_no_checks(monkeypatch):
    """Above 64 rows a projection is torch's GEMM at once: the checks in front of the kernel would be host
    time of every layer."""
    def called(x, w):
        raise AssertionError("checked")

    monkeypatch.setattr(transformer, "_takes_skinny", called)
    monkeypatch.setattr(transformer, "silu_mul", lambda gu, n: gu[:, :n])
    monkeypatch.setattr(RoPE, "apply_", Doubling.apply_)
    h = t.randn(65, CFG.d_model)
    q, _ = attend(Attention(CFG), "decode", monkeypatch, h)
    assert q.shape == (65, CFG.num_q_heads, CFG.head_dim)
    assert SwiGLU(CFG)(h).shape == h.shape
