"""A decoder layer in one call (`cached_layer`) against its three operations called one by one:
the same outputs and cache bits, whatever the rows, the slots and the cache's type; and a layer
that it does not take still runs, by the operations that do."""

from __future__ import annotations

import pytest
import torch
from torch import nn

pytestmark = pytest.mark.gpu

DEV = "cuda"
D, HEADS = 256, 8


def _layers(**kw):
    torch.manual_seed(3)
    make = lambda: nn.TransformerEncoderLayer(  # noqa: E731
        D, HEADS, 1024, dropout=0.0, batch_first=True, norm_first=True,
        **{"activation": "gelu", **kw}).to(DEV).to(torch.bfloat16).eval()
    return make(), make()


def _inputs(n, slots, cache_dtype):
    g = torch.Generator(device=DEV).manual_seed(n)
    x = (torch.randn(n, D, generator=g, device=DEV) * 0.5).to(torch.bfloat16)
    k, v = (torch.randn(n + 3, HEADS, slots, D // HEADS, generator=g, device=DEV).to(cache_dtype)
            for _ in range(2))
    pos = torch.randint(-1, slots + 2, (n,), generator=g, device=DEV)
    rows = torch.randperm(n + 3, generator=g, device=DEV)[:n].contiguous()
    return x, k, v, pos, rows


@pytest.mark.parametrize("n,slots,cache_dtype", [(1, 50, torch.bfloat16), (2, 70, torch.float32),
                                                 (33, 50, torch.bfloat16), (0, 50, torch.bfloat16)])
@pytest.mark.parametrize("last", [False, True])
@torch.no_grad()
def test_cached_layer_is_its_operations(n, slots, cache_dtype, last):
    from cugo_amd import seq_decode as sd
    from cugo_amd.cugo_seq_attention50 import decode_attention_append

    layer, after = _layers()
    x, k, v, pos, rows = _inputs(n, slots, cache_dtype)
    norm = None if last else after.norm1
    h = sd.add_norm(x, None, layer.norm1)[1]
    sa = layer.self_attn
    qkv = [t.reshape(n, HEADS, D // HEADS).contiguous()
           for t in sd.linear(h, sa.in_proj_weight, sa.in_proj_bias).chunk(3, -1)]
    k2, v2 = k.clone(), v.clone()
    att = decode_attention_append(*qkv, k2, v2, pos, rows)
    want = sd.attention_tail(layer, att.reshape(n, D), x, norm)
    got = sd._layer(layer, h, x, HEADS, k, v, pos, rows, None, norm)
    for a, b in zip((got, k, v) if last else (*got, k, v), (want, k2, v2) if last else (*want, k2, v2)):
        assert torch.equal(torch.nan_to_num(a, nan=9.0), torch.nan_to_num(b, nan=9.0))


@torch.no_grad()
def test_other_layers_take_the_operations():
    """A ReLU layer and one without biases, each against the fused layer's own parts in float32."""
    from cugo_amd import seq_decode as sd

    for kw in ({"activation": "relu"}, {"bias": False}):
        layer, after = _layers(**kw)
        x, k, v, pos, rows = _inputs(9, 50, torch.bfloat16)
        pos = pos.clamp(0, 49)
        h = layer.norm1(x)
        sa = layer.self_attn
        out, ln = sd._layer(layer, h, x, HEADS, k, v, pos, rows, None, after.norm1)
        q = torch.nn.functional.linear(h, sa.in_proj_weight, sa.in_proj_bias).float().chunk(3, -1)[0]
        kk, vv = (t.index_select(0, rows).float() for t in (k, v))  # with the appended slots
        s = (q.view(9, HEADS, 1, -1) * kk).sum(-1) * (D // HEADS) ** -0.5
        s = s.masked_fill(torch.arange(50, device=DEV)[None, None] > pos[:, None, None], -1e30)
        a = (s.softmax(-1)[..., None] * vv).sum(2).reshape(9, D).to(torch.bfloat16)
        x1 = x + sa.out_proj(a)
        want = x1 + layer.linear2(layer.activation(layer.linear1(layer.norm2(x1))))
        assert float((out.float() - want.float()).norm() / want.float().norm()) < 1e-2
        assert torch.equal(ln, after.norm1(out)) or float(
            (ln.float() - after.norm1(out).float()).abs().max()) < 0.05
