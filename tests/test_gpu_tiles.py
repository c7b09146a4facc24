"""The engine kernels' games a tile, chosen by batch, change no row's result: every batch at
an edge of the choice (and one game past it, a partial last tile) gives the last rows of
what a batch of 64-game tiles gives, bit for bit.  (The last ones, so that each batch has other
games at its rows: outputs may lie where an earlier batch's lay.)"""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda"
BIG = 33_000  # past every smaller tile
BASE = 0x51CE5

EDGES = [1, 3, 257, 1024, 1025, 2049, 4096, 4097, 8193, 16384, 16385, 32768]


@pytest.fixture(scope="module")
def ext():
    from cugo_amd import load_extension

    return load_extension()


def _games(ext, n, base):
    """n games with fresh spares, dealt from seed base + i (+ BIG a generation)."""
    idx = torch.arange(n, dtype=torch.int64, device=DEV)
    gen = torch.zeros(n, dtype=torch.int32, device=DEV)
    s = {"states": ext.create(idx + base, idx & 1), "gen": gen,
         "sampler": ext.seed_samplers(n, base, gen),
         "spares": torch.empty((2 * n, 248), dtype=torch.uint8, device=DEV),
         "spare_gen": torch.zeros(2 * n, dtype=torch.int32, device=DEV)}
    ext.refill_spares(s["spares"], s["spare_gen"], gen, base, BIG)
    return s


def _play(ext, s, base, steps):
    out = ext.play_random(s["states"], s["sampler"], base, s["gen"], s["spares"], s["spare_gen"],
                          BIG, steps)
    return [*out, s["states"], s["sampler"], s["gen"]]


def _results(ext, n, first=0):
    """Every tiled operation on n games from the even `first` on, 37 random steps in (re-deals,
    stale spares and pending choices among them)."""
    base = BASE + first
    s = _games(ext, n, base)
    got = {"play": [t.clone() for t in _play(ext, s, base, 37)]}
    seen = ext.observe_sample(s["states"], s["sampler"])
    actions = seen[5]
    ids = torch.arange(n, dtype=torch.int64, device=DEV).flip(0).contiguous()
    got["observe"] = list(seen)
    indexed = [t.flip(0) for t in ext.observe_indexed(s["states"], ids)]
    assert all(torch.equal(a, b) for a, b in zip(indexed, seen[:5]))
    got["branch"] = ext.branch_indexed(s["states"], ids, actions.flip(0).contiguous())
    got["branch"] = [t.flip(0) for t in got["branch"]]
    both = ext.branch_observe_indexed(s["states"], ids, actions.flip(0).contiguous())
    got["branch_observe"] = [t.flip(0) for t in both]
    stepped = s["states"].clone()
    got["step"] = [*ext.step(stepped, actions), stepped]
    for bf16 in (False, True):
        t = {k: v.clone() for k, v in s.items()}
        features = torch.empty((n, 720), dtype=torch.bfloat16 if bf16 else torch.float32,
                               device=DEV)
        out = ext.step_observe_spares(t["states"], actions, base, t["gen"], t["sampler"],
                                      t["spares"], t["spare_gen"], features, BIG)
        got[f"step_observe{int(bf16)}"] = [*out, t["states"], t["gen"], t["sampler"]]
    out = ext.step_reset_spares(s["states"], actions, base, s["gen"], s["sampler"], s["spares"],
                                s["spare_gen"], BIG)
    got["step_reset"] = [*out, s["states"], s["gen"], s["sampler"]]
    idx = torch.arange(n, dtype=torch.int64, device=DEV)
    got["canonical"] = [ext.rollout_canonical(idx + base, idx & 1)]
    return got


@pytest.fixture(scope="module")
def big(ext):
    return _results(ext, BIG)


@pytest.mark.parametrize("n", EDGES)
def test_tile_choice_changes_no_row(ext, big, n):
    first = (BIG - n) & ~1
    got = _results(ext, n, first)
    for name, tensors in got.items():
        for k, t in enumerate(tensors):
            want = big[name][k][first:first + n]
            assert t.shape == want.shape and t.dtype == want.dtype
            assert torch.equal(t, want), (name, k, n)
