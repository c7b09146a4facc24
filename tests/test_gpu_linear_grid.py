"""The linear layer's map from workgroups to tiles covers every tile once, whatever the number
of workgroups modulo the eight XCDs: an identity weight gives the input back."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [64, 320])  # one and three column tiles of 128
def test_linear_covers_every_tile(n):
    from cugo_amd import load_extension

    ext = load_extension()
    x = torch.randn(32 * 17, 64, device="cuda").to(torch.bfloat16)
    w = torch.eye(64, device="cuda").repeat(n // 64, 1).to(torch.bfloat16)
    wp = ext.mlp_pack_weight(w, n, 64)
    for blocks in range(1, 18):
        m = 32 * blocks - blocks % 3
        assert torch.equal(ext.linear(x[:m], wp, n, None), x[:m].repeat(1, n // 64)), m
