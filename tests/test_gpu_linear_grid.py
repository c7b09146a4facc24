"""The linear layers' map from workgroups to tiles covers every tile once, whatever the number
of workgroups modulo the eight XCDs, for every shape of tile: an identity weight gives the
input back, into outputs that hold NaN before each call."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda"
K = 64


@pytest.fixture(scope="module")
def ext():
    from cugo_amd import load_extension

    return load_extension()


def _nan(*shape):
    return torch.full(shape, float("nan"), dtype=torch.bfloat16, device=DEV)


@pytest.mark.parametrize("tile,rows", [(1, 32), (2, 64), (3, 64), (4, 128), (5, 64), (6, 128), (7, 32)])
@pytest.mark.parametrize("n", [64, 320])  # one and three column tiles of 128
@pytest.mark.parametrize("gelu", [False, True])
def test_linear_covers_every_tile(ext, tile, rows, n, gelu):
    g = torch.Generator(device=DEV).manual_seed(n + tile)
    w = torch.eye(K, device=DEV).repeat(n // K, 1).to(torch.bfloat16)
    wp = ext.mlp_pack_weight(w, n, K)
    for blocks in range(1, 18):
        m = rows * blocks - blocks % 3
        x = torch.randn(m, K, generator=g, device=DEV).to(torch.bfloat16)
        out = _nan(m, n)
        ext.linear(x, wp, n, None, gelu, tile=tile, out=out)
        want = torch.nn.functional.gelu(x) if gelu else x
        assert torch.equal(out, want.repeat(1, n // K)), m


@pytest.mark.parametrize("tile,rows", [(1, 32), (2, 32), (3, 16), (4, 64)])
def test_linear_add_layernorm_covers_every_tile(ext, tile, rows):
    n = 256
    g = torch.Generator(device=DEV).manual_seed(tile)
    wp = ext.mlp_pack_weight(torch.eye(K, device=DEV).repeat(n // K, 1).to(torch.bfloat16), n, K)
    one, zero = (torch.full((n,), v, dtype=torch.bfloat16, device=DEV) for v in (1.0, 0.0))
    for blocks in range(1, 18):
        m = rows * blocks - blocks % 3
        x = torch.randn(m, K, generator=g, device=DEV).to(torch.bfloat16)
        res = torch.randn(m, n, generator=g, device=DEV).to(torch.bfloat16)
        out, ln = _nan(m, n), _nan(m, n)
        ext.linear_add_layernorm(x, wp, None, res, one, zero, 1e-5, tile=tile, out=out, ln_out=ln)
        want = ext.add_layernorm(res, x.repeat(1, n // K), one, zero, 1e-5)
        assert torch.equal(out, want[0]) and torch.equal(ln, want[1]), m
