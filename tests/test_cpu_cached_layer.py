"""CPU: what a decoder layer that no fused launch takes costs on the host."""

from __future__ import annotations

import pytest
import torch
from torch import nn

from cugo_amd import seq_decode as sd


@pytest.mark.parametrize("kw", [{"activation": "relu"}, {"dim_feedforward": 512}, {"bias": False}])
@pytest.mark.parametrize("last", [False, True])
@torch.no_grad()
def test_an_unfused_layer_is_examined_twice(monkeypatch, kw, last):
    """_layer asks whether the fused launches take the layer once for all of it and once for its
    feed-forward (whose input may fit where the whole does not), not again after the attention;
    and its result is the plain layer's on the same attention (here: the values)."""
    torch.manual_seed(0)
    layer = nn.TransformerEncoderLayer(
        256, 8, **{"dim_feedforward": 1024, "activation": "gelu", **kw}, dropout=0.0,
        batch_first=True, norm_first=True).double().eval()  # a type that no HIP launch takes
    norm = None if last else nn.LayerNorm(256).double()
    calls = []
    plain = sd._ffn_args
    monkeypatch.setattr(sd, "_ffn_args", lambda *a: calls.append(1) or plain(*a))
    monkeypatch.setattr(sd, "decode_attention_append", lambda q, k, v, *a, **kw: v)
    x = torch.randn(5, 256, dtype=torch.float64)
    h = layer.norm1(x)
    empty = torch.empty(0)
    out = sd._layer(layer, h, x, 8, empty, empty, empty, None, None, norm)
    assert len(calls) == 2
    sa = layer.self_attn
    v = torch.nn.functional.linear(h, sa.in_proj_weight, sa.in_proj_bias).chunk(3, -1)[2]
    x1 = x + sa.out_proj(v)
    want = x1 + layer.linear2(layer.activation(layer.linear1(layer.norm2(x1))))
    if last:
        torch.testing.assert_close(out, want)
    else:
        torch.testing.assert_close(out[0], want)
        torch.testing.assert_close(out[1], norm(want))
