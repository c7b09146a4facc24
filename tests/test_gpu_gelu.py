"""The linear layer's GELU against torch's on every finite bf16 value."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda"


@pytest.fixture(scope="module")
def ext():
    from cugo_amd import load_extension

    return load_extension()


def test_gelu_of_every_bf16(ext):
    """Through an identity weight, every finite bf16 value (in order, so that whole
    wavefronts lie on either side of -4, and shuffled, so that most hold both): torch's
    F.gelu bit for bit up to the sign of zero."""
    bits = torch.arange(65536, dtype=torch.int32).to(torch.uint16).view(torch.int16)
    values = bits.view(torch.bfloat16)
    values = values[torch.isfinite(values.float())]
    g = torch.Generator().manual_seed(1)
    wp = ext.mlp_pack_weight(torch.eye(64, dtype=torch.bfloat16, device=DEV), 64, 64)
    for v in (values, values[torch.randperm(len(values), generator=g)]):
        x = v.view(-1, 64).to(DEV)
        plain = ext.linear(x, wp, 64, None)
        big = x.float().abs() >= 2.0 ** -126
        assert torch.equal(plain[big], x[big])
        assert torch.equal(ext.linear(x, wp, 64, None, gelu=True),
                           torch.nn.functional.gelu(plain))
