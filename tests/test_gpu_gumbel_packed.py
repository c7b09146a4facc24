"""The Gumbel-max draw over a row's legal actions alone against the draw over all of them."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda"


@pytest.fixture(scope="module")
def ext():
    from cugo_amd import load_extension

    return load_extension()


def _legal(n, a, counts, g):
    """counts[r % len(counts)] legal actions in row r (at most a)."""
    rank = torch.rand(n, a, generator=g, device=DEV).argsort(1).argsort(1)
    want = torch.tensor([counts[r % len(counts)] for r in range(n)], device=DEV)
    return rank < want[:, None]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n,a", [(4099, 179), (1, 179), (67, 192), (130, 16), (130, 15), (9, 1),
                                 (7681, 179), (8161, 192), (8192, 15), (32767, 179)])
def test_gumbel_packed_rows(ext, dtype, n, a):
    """Actions and log-probabilities of gumbel_sample_philox, which packs rows of few legal
    actions, against gumbel_sample on the same uniforms, which never does: the same bits, at
    0 to 33 legal actions a row (33 is past the packing), mixed within wavefronts and alike
    in them, with ties, infinities and the type's lowest value among the logits; the last four
    sizes are taken by the larger workgroups (a whole last one, one of a single row, odd rows)."""
    g = torch.Generator(device=DEV).manual_seed(n + a)
    epoch = torch.tensor([7], dtype=torch.int64, device=DEV)
    low = torch.finfo(dtype).min
    for counts in ([0], [1], [3, 16, 17, 31], [32], [5, 5, 5, 33], [0, 1, 2, 12]):
        legal = _legal(n, a, counts, g)
        for special in (None, 0.0, float("inf"), float("-inf"), low, -2e29):
            logits = (torch.randn(n, a, generator=g, device=DEV) * 3).to(dtype)
            if special is not None:
                hit = torch.rand(n, a, generator=g, device=DEV) < 0.5
                logits = torch.where(hit, torch.full_like(logits, special), logits)
            u = torch.empty((n, a), device=DEV)
            ext.gumbel_sample_philox(logits, legal, 99, epoch, 3, uniforms_out=u)
            want_a, want_lp = ext.gumbel_sample(logits, legal, u)
            got_a, got_lp = ext.gumbel_sample_philox(logits, legal, 99, epoch, 3)
            assert torch.equal(got_a, want_a), (counts, special)
            assert torch.equal(torch.nan_to_num(got_lp, nan=7.0),
                               torch.nan_to_num(want_lp, nan=7.0)), (counts, special)


def test_rows_past_the_packing_pay_for_one_way(ext):
    """Rows of 40 legal actions, which are not packed, take little longer than the draw on given
    uniforms over all actions (29.0 and 24.3 us measured at 65,536 rows; packing them first in
    vain made it 35.8): the fastest of interleaved launches."""
    n, a = 65536, 179
    g = torch.Generator(device=DEV).manual_seed(1)
    epoch = torch.tensor([7], dtype=torch.int64, device=DEV)
    legal = _legal(n, a, [40], g)
    logits = torch.randn(n, a, generator=g, device=DEV).to(torch.bfloat16)
    u = torch.rand(n, a, generator=g, device=DEV)
    calls = {"drawn": lambda: ext.gumbel_sample_philox(logits, legal, 99, epoch, 3),
             "given": lambda: ext.gumbel_sample(logits, legal, u)}
    times = {}
    for _ in range(30):
        for name, call in calls.items():
            start, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            start.record()
            for _ in range(10):
                call()
            end.record()
            end.synchronize()
            times[name] = min(times.get(name, 1e9), start.elapsed_time(end))
    assert times["drawn"] < 1.33 * times["given"], times
