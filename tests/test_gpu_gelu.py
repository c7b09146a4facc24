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


def test_gelu_of_every_bf16_bias(ext):
    """The same through the bias of a zero input, so that infinities, NaN and the smallest
    values get there too: torch's bits, and NaN where it gives NaN."""
    bits = torch.arange(65536, dtype=torch.int32).to(torch.uint16).view(torch.int16)
    bias = bits.view(torch.bfloat16).to(DEV)
    wp = ext.mlp_pack_weight(torch.zeros((65536, 64), dtype=torch.bfloat16, device=DEV), 65536, 64)
    x = torch.zeros((3, 64), dtype=torch.bfloat16, device=DEV)
    plain = ext.linear(x, wp, 65536, bias)
    assert torch.equal(torch.isnan(plain), torch.isnan(bias).expand(3, -1))
    finite = torch.isfinite(plain)
    assert torch.equal(plain[finite], bias.expand(3, -1)[finite])
    got, want = ext.linear(x, wp, 65536, bias, gelu=True), torch.nn.functional.gelu(plain)
    assert torch.equal(torch.isnan(got), torch.isnan(want))
    number = ~torch.isnan(want)
    assert torch.equal(got.view(torch.int16)[number], want.view(torch.int16)[number])


def test_ffn_time_does_not_depend_on_its_inputs(ext):
    """Pre-activations of standard deviation 3, of which most wavefronts hold some below -4,
    cost a feed-forward launch about what those of 0.6 do (24.9 and 24.1 us measured at 12,288
    rows; a second evaluation for them made it 36): the fastest of interleaved launches."""
    g = torch.Generator(device=DEV).manual_seed(2)

    def rand(*shape, std=1.0):
        return (torch.randn(*shape, generator=g, device=DEV) * std).to(torch.bfloat16)

    n = 12288
    h, x, b1, b2 = rand(n, 256), rand(n, 256), rand(1024, std=0.0), rand(256)
    w2 = ext.mlp_pack_weight(rand(256, 1024, std=1 / 32), 256, 1024)
    times = {}
    w1 = {std: ext.mlp_pack_weight(rand(1024, 256, std=std / 16), 1024, 256) for std in (0.6, 3.0)}
    for _ in range(30):
        for std, w in w1.items():
            start, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            start.record()
            for _ in range(10):
                ext.ffn(h, x, w, b1, w2, b2)
            end.record()
            end.synchronize()
            times[std] = min(times.get(std, 1e9), start.elapsed_time(end))
    assert times[3.0] < 1.2 * times[0.6], times
