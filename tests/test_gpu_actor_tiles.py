"""The MLP actor's rows a tile, chosen by batch, change no row's result: a batch at each edge
of the choice (and one past it, and partial last tiles) gives the last rows of what a batch
of 128-row tiles gives, bit for bit, over the depths, widths and input types it takes.  (The last
ones, so that each batch has other rows: outputs may lie where an earlier batch's lay.)"""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda"
BIG = 16_384 + 130  # 128-row tiles, the last one partial


@pytest.fixture(scope="module")
def ext():
    from cugo_amd import load_extension

    return load_extension()


@pytest.mark.parametrize("blocks,features,actions,dtype,sizes", [
    (3, 720, 179, torch.float32, (1, 15, 16, 17, 300, 3072, 3073, 8192, 8193, 16384)),
    (3, 720, 179, torch.bfloat16, (1, 33, 3072, 3073, 8192, 8193, 16384)),
    (0, 8, 1, torch.float32, (5, 3100, 8200)),
    (4, 768, 255, torch.bfloat16, (5, 3100, 8200)),
    (1, 104, 30, torch.float32, (5, 3100, 8200)),
])
def test_actor_tiles_give_the_same_rows(ext, blocks, features, actions, dtype, sizes):
    from cugo_amd.rollout import ResidualMlpActor, mlp_forward, pack_actor

    torch.manual_seed(5)
    actor = ResidualMlpActor(blocks=blocks, features=features, actions=actions)
    with torch.no_grad():
        for p in actor.parameters():
            p.normal_(0.0, 0.05)
    packed = pack_actor(ext, actor.to(DEV).to(torch.bfloat16).eval())
    x = torch.rand((BIG, features), device=DEV).to(dtype)
    with torch.no_grad():
        want_l, want_v = mlp_forward(ext, packed, x)
        assert torch.isfinite(want_l.float()).all() and torch.isfinite(want_v).all()
        for n in sizes:
            part = x[BIG - n:].contiguous()
            copy = torch.full((n, features), float("nan"), dtype=torch.bfloat16, device=DEV)
            got_l, got_v = mlp_forward(ext, packed, part, copy)
            assert torch.equal(got_l, want_l[BIG - n:]), n
            assert torch.equal(got_v, want_v[BIG - n:]), n
            assert torch.equal(copy, part.to(torch.bfloat16)), n
