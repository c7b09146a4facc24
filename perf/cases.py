"""The work that users of this framework have it do, as cases that can be timed and compared.

Each kind of case is one use of the public entry points (`load_extension()`'s operations,
`cugo_amd.rollout`, `cugo_amd.seq_selfplay`, `cugo_amd.seq_decode`), over the sizes that
the self-play loops, the searches and the evaluations call it with:

  play       random-policy self-play, 32 decisions a call (`refill_spares`, `play_random`)
  env        one decision of a stepping loop (`observe_sample`, `step_reset_spares`)
  collect    the engine's part of one PPO collector step: the masked sample from the
             actor's logits and the step with the next observation
  branch     a search's expansion: children of some roots, with or without observations
  canonical  whole games played by the canonical rule (the rollouts of a search's leaves)
  actor      the MLP policy's forward pass
  decode     one KV append + attention of the sequence policy
  layer      one encoder layer of the sequence policy on one token a row
  seqstep    the policy's part of a sequence self-play step: the query tokens, the last
             step's events and the queries through all layers, and the readout's logits
"""

import math

import torch
import torch.nn.functional as F

SEED_BASE = 0x243F6A8885A308D3
FEATURES, ACTIONS, ROW_BYTES = 720, 179, 248
STEPS = 32          # decisions of one play call, and between two refills of the spares
HORIZON = 16        # rows of the collector's buffer that the passes go round in
D, HEADS, DH, HIDDEN = 256, 8, 32, 1024
DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}


def listed():
    return [
        # The headline workload: 65,536 resident games.
        {"name": "play_65536", "kind": "play", "batch": 65536},
        # A small resident batch: debugging runs, several players on one GPU, odd size.
        {"name": "play_3001", "kind": "play", "batch": 3001},
        # A stepping loop over few games (the latency of its two launches counts).
        {"name": "env_700", "kind": "env", "batch": 700},
        # The PPO collector's batch.
        {"name": "collect_32768", "kind": "collect", "batch": 32768},
        # A search over 4,096 roots x 256 children, observed for the next evaluation.
        {"name": "branch_1048576", "kind": "branch", "roots": 4096, "children": 1048576,
         "observe": True},
        # One shallow search: every child of a few dozen positions, states only.
        {"name": "branch_2500", "kind": "branch", "roots": 50, "children": 2500,
         "observe": False},
        # The canonical driver at the batch its bench times.
        {"name": "canonical_131072", "kind": "canonical", "games": 131072},
        # The MLP actor over the collector's batch, reading its bf16 buffer.
        {"name": "actor_32768", "kind": "actor", "rows": 32768, "dtype": "bf16"},
        # The same actor for a few hundred positions (an evaluation, a search's leaves),
        # on the float32 features that `observe` returns.
        {"name": "actor_300", "kind": "actor", "rows": 300, "dtype": "f32"},
        # Decode over 320-slot caches of ragged length, longest first as `cached_step` does.
        {"name": "decode_4096x320", "kind": "decode", "rows": 4096, "slots": 320,
         "fill": 0.53, "dtype": "bf16"},
        # One layer for a few hundred games.
        {"name": "layer_500", "kind": "layer", "rows": 500},
        # A sequence self-play step's network over a wave of 4,096 games (whole call).
        {"name": "seqstep_4096", "kind": "seqstep", "wave": 4096},
    ]


def _log_uniform(rng, low, high):
    return max(low, min(high, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng):
    kind = rng.choice(("play", "env", "collect", "branch", "canonical", "actor", "decode",
                       "layer", "seqstep"))
    if kind == "play":
        return {"kind": kind, "batch": _log_uniform(rng, 256, 65536)}
    if kind == "env":
        return {"kind": kind, "batch": _log_uniform(rng, 64, 65536)}
    if kind == "collect":
        return {"kind": kind, "batch": _log_uniform(rng, 256, 65536)}
    if kind == "branch":
        children = _log_uniform(rng, 500, 1048576)
        roots = max(1, children // rng.randint(4, 256))
        return {"kind": kind, "roots": min(roots, 8192), "children": children,
                "observe": rng.random() < 0.5}
    if kind == "canonical":
        return {"kind": kind, "games": _log_uniform(rng, 256, 262144)}
    if kind == "actor":
        return {"kind": kind, "rows": _log_uniform(rng, 1, 32768),
                "dtype": rng.choice(("bf16", "f32"))}
    if kind == "decode":
        return {"kind": kind, "rows": _log_uniform(rng, 16, 4096),
                "slots": rng.choice((50, 50, 131, 320)), "fill": round(rng.uniform(0.1, 0.95), 3),
                "dtype": rng.choice(("bf16", "bf16", "bf16", "f16", "f32"))}
    if kind == "layer":
        return {"kind": kind, "rows": _log_uniform(rng, 1, 16384)}
    return {"kind": kind, "wave": _log_uniform(rng, 32, 4096)}


# ------------------------------------------------------------------ game states ----

def _ext():
    from cugo_amd import load_extension

    return load_extension()


def _base(seed):
    return (SEED_BASE + seed * 0x9E3779B1) & (2**62 - 1)


def _resident(batch, seed):
    """Resident games part-way through (each row at its own stage), as any loop has them
    after its first few dozen decisions: states, samplers, generations and spares."""
    ext = _ext()
    base = _base(seed)
    idx = torch.arange(batch, dtype=torch.int64, device="cuda")
    s = {"ext": ext, "base": base, "states": ext.create(idx + base, idx & 1),
         "gen": torch.zeros(batch, dtype=torch.int32, device="cuda"),
         "spares": torch.empty((2 * batch, ROW_BYTES), dtype=torch.uint8, device="cuda"),
         "spare_gen": torch.zeros(2 * batch, dtype=torch.int32, device="cuda"), "t": 0}
    s["sampler"] = ext.seed_samplers(batch, base, s["gen"])
    for steps in (29, 20):
        ext.refill_spares(s["spares"], s["spare_gen"], s["gen"], base)
        ext.play_random(s["states"], s["sampler"], base, s["gen"], s["spares"], s["spare_gen"],
                        steps=steps)
    return s


def _roots(n, seed):
    """n positions 3 to 15 random decisions deep."""
    ext = _ext()
    base = _base(seed)
    idx = torch.arange(n, dtype=torch.int64, device="cuda")
    states = ext.create(idx + base, idx & 1)
    sampler = ext.seed_samplers(n, base, torch.zeros(n, dtype=torch.int32, device="cuda"))
    depth = 3 + (idx * 7 + seed) % 13
    for t in range(15):
        actions = ext.observe_sample(states, sampler)[5]
        ids = torch.nonzero(depth > t).squeeze(1)
        ext.step_indexed(states, ids, actions.index_select(0, ids))
    return ext, states


# -------------------------------------------------------------------- networks ----

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _randn(shape, std, g, dtype=torch.bfloat16):
    return (torch.randn(shape, generator=g, device="cuda") * std).to(dtype)


def _features(n, g):
    """Rows like `observe`'s: 0/1 features, one in six set, and two dozen scalars."""
    x = (torch.rand(n, FEATURES, generator=g, device="cuda") < 1 / 6).float()
    x[:, 453:479] = torch.rand(n, 26, generator=g, device="cuda")
    return x


def _actor_inputs(case, seed):
    from cugo_amd.rollout import ResidualMlpActor

    torch.manual_seed(seed)
    actor = ResidualMlpActor().to("cuda").to(torch.bfloat16).eval()
    return actor, _features(case["rows"], _gen(seed)).to(DTYPES[case["dtype"]])


def _policy(layers, seed):
    from cugo_amd.seq_selfplay import SeqPolicy

    torch.manual_seed(seed)
    return SeqPolicy(layers=layers).to("cuda").to(torch.bfloat16).eval()


def _cache(policy, rows, g):
    from cugo_amd.seq_selfplay import policy_cache

    cache = policy_cache(policy, rows, "cuda")
    for t in (cache.k, cache.v):  # layer by layer: the random numbers are float32
        for part in t:
            part.copy_(torch.randn(part.shape, generator=g, device="cuda") * 0.5)
    return cache


def _seq_inputs(case, seed):
    """A wave in the middle of its games: every game has its own number of events, one in
    five is over (its rows are skipped), one seat's row of each game takes the query."""
    w = case["wave"]
    g = _gen(seed)
    policy = _policy(4, seed)
    cache = _cache(policy, 2 * w, g)
    count = torch.randint(1, 40, (w,), generator=g, device="cuda")
    live = torch.rand(w, generator=g, device="cuda") < 0.8
    mover = torch.randint(0, 2, (w,), generator=g, device="cuda")
    gone = torch.full_like(count, -1)
    legal = torch.rand(w, ACTIONS, generator=g, device="cuda") < 0.06
    q_in = torch.zeros((w, 1024), dtype=torch.bfloat16, device="cuda")
    q_in[:, :FEATURES] = _features(w, g)
    q_in[:, FEATURES:FEATURES + ACTIONS] = legal
    pair = torch.zeros((3 * w, D), dtype=torch.bfloat16, device="cuda")
    pair[:2 * w] = _randn((2 * w, D), 0.5, g)
    return {"policy": policy, "cache": cache, "q_in": q_in, "pair": pair, "wave": w,
            "event_pos": torch.where(live, count, gone).repeat(2),
            "query_pos": torch.where(live, count + 1, gone),
            "query_rows": mover * w + torch.arange(w, device="cuda")}


def _decode_inputs(case, seed):
    g = _gen(seed)
    n, slots, dtype = case["rows"], case["slots"], DTYPES[case["dtype"]]
    q, kn, vn = (_randn((n, HEADS, DH), 0.5, g, dtype) for _ in range(3))
    keys, values = (_randn((n, HEADS, slots, DH), 0.5, g, dtype) for _ in range(2))
    # ragged: uniform up to twice the fill, cut at the last slot
    pos = (torch.rand(n, generator=g, device="cuda") * 2 * case["fill"] * slots).long()
    rows = torch.randperm(n, generator=g, device="cuda")
    return q, kn, vn, keys, values, pos.clamp_max(slots - 1), rows


def _layer_inputs(case, seed):
    n = case["rows"]
    g = _gen(seed)
    policy = _policy(1, seed)
    cache = _cache(policy, n, g)
    cache.length.copy_(torch.randint(1, 46, (n,), generator=g, device="cuda"))
    return policy, cache, _randn((n, D), 0.5, g)


# --------------------------------------------------------------------- prepare ----

def prepare(case, seed):
    kind = case["kind"]
    if kind in ("play", "env"):
        return {"kind": kind, **_resident(case["batch"], seed)}
    if kind == "collect":
        b = case["batch"]
        s = _resident(b, seed)
        s["features"] = torch.empty((HORIZON, b, FEATURES), dtype=torch.bfloat16, device="cuda")
        s["legal"] = torch.empty((HORIZON, b, ACTIONS), dtype=torch.bool, device="cuda")
        s["action"] = torch.empty((HORIZON, b), dtype=torch.int64, device="cuda")
        s["logp"], s["reward"] = (torch.empty((HORIZON, b), device="cuda") for _ in range(2))
        s["done"] = torch.empty((HORIZON, b), dtype=torch.bool, device="cuda")
        s["logits"] = _randn((b, ACTIONS), 1.0, _gen(seed))
        s["epoch"] = torch.ones(1, dtype=torch.int64, device="cuda")
        s["key"] = seed
        s["ext"].observe_bf16(s["states"], s["features"][0], legal=s["legal"][0])
        return {"kind": kind, **s}
    if kind == "branch":
        n = case["children"]
        ext, states = _roots(case["roots"], seed)
        ids = torch.arange(n, device="cuda") * case["roots"] // n
        legal = ext.observe(states)[1].index_select(0, ids)
        actions = ext.sample_uniform(legal, ext.seed_samplers(
            n, _base(seed), torch.zeros(n, dtype=torch.int32, device="cuda")))
        return {"kind": kind, "ext": ext, "states": states, "ids": ids, "actions": actions,
                "observe": case["observe"]}
    if kind == "canonical":
        i = torch.arange(case["games"], dtype=torch.int64, device="cuda")
        return {"kind": kind, "ext": _ext(), "seeds": i * -7046029254386353131 + _base(seed),
                "first": i & 1}
    if kind == "actor":
        from cugo_amd.rollout import pack_actor

        actor, x = _actor_inputs(case, seed)
        return {"kind": kind, "ext": _ext(), "x": x, "packed": pack_actor(_ext(), actor)}
    if kind == "decode":
        from cugo_amd.seq_decode import decode_order, order_pays

        q, kn, vn, keys, values, pos, rows = _decode_inputs(case, seed)
        # once a step, for the decodes of all its layers
        order = decode_order(pos, case["slots"]) if order_pays(len(pos), case["slots"]) else None
        return {"kind": kind, "args": (q, kn, vn, keys, values, pos, rows, None, order)}
    if kind == "layer":
        policy, cache, x = _layer_inputs(case, seed)
        policy.prepare()
        return {"kind": kind, "policy": policy, "cache": cache, "x": x}
    s = _seq_inputs(case, seed)
    s["policy"].prepare()
    s["pair_h"] = torch.zeros_like(s["pair"])
    # the waiting event rows' first norm, which the launch that made them has written
    n1 = s["policy"].encoder.layers[0].norm1
    with torch.no_grad():
        s["pair_h"][:2 * case["wave"]] = n1(s["pair"][:2 * case["wave"]])
    return {"kind": kind, **s}


# ------------------------------------------------------------------------- run ----

def _refill(s):
    if s["t"] % STEPS == 0:
        s["ext"].refill_spares(s["spares"], s["spare_gen"], s["gen"], s["base"])


@torch.no_grad()
def run(s):
    kind = s["kind"]
    if kind == "play":
        s["ext"].refill_spares(s["spares"], s["spare_gen"], s["gen"], s["base"])
        out = s["ext"].play_random(s["states"], s["sampler"], s["base"], s["gen"], s["spares"],
                                   s["spare_gen"], steps=STEPS)
        return [*out, s["states"], s["sampler"], s["gen"]]
    if kind == "env":
        _refill(s)
        s["t"] += 1
        seen = s["ext"].observe_sample(s["states"], s["sampler"])
        out = s["ext"].step_reset_spares(s["states"], seen[5], s["base"], s["gen"], s["sampler"],
                                         s["spares"], s["spare_gen"])
        return [*seen, *out, s["states"], s["sampler"], s["gen"]]
    if kind == "collect":
        _refill(s)
        t, s["t"] = s["t"], s["t"] + 1
        here, there = t % HORIZON, (t + 1) % HORIZON
        s["ext"].gumbel_sample_philox(s["logits"], s["legal"][here], s["key"], s["epoch"], t,
                                      actions=s["action"][here], logp=s["logp"][here])
        out = s["ext"].step_observe_spares(
            s["states"], s["action"][here], s["base"], s["gen"], s["sampler"], s["spares"],
            s["spare_gen"], s["features"][there], reward=s["reward"][here],
            done=s["done"][here], legal=s["legal"][there])
        return [*out, s["action"][here], s["logp"][here], s["states"], s["gen"]]
    if kind == "branch":
        call = s["ext"].branch_observe_indexed if s["observe"] else s["ext"].branch_indexed
        return list(call(s["states"], s["ids"], s["actions"]))
    if kind == "canonical":
        return s["ext"].rollout_canonical(s["seeds"], s["first"])
    if kind == "actor":
        from cugo_amd.rollout import mlp_forward

        return list(mlp_forward(s["ext"], s["packed"], s["x"]))
    if kind == "decode":
        from cugo_amd.cugo_seq_attention50 import decode_attention_append

        return [decode_attention_append(*s["args"]), s["args"][3], s["args"][4]]
    if kind == "layer":
        return [s["policy"].cached_step(s["cache"], s["x"]), s["cache"].k, s["cache"].v]
    from cugo_amd.seq_decode import cached_step_pair

    policy, w = s["policy"], s["wave"]
    policy.query_from_input(s["q_in"], out=s["pair"][2 * w:], norm_out=s["pair_h"][2 * w:])
    hidden, normed = cached_step_pair(policy, s["cache"], s["pair"], 2 * w, s["event_pos"],
                                      s["query_pos"], s["query_rows"], final_norm=policy.norm,
                                      h=s["pair_h"])
    return [policy.readout(hidden, normed), s["cache"].k, s["cache"].v]


# ------------------------------------------------------------------------ work ----

OBSERVED = 4 * FEATURES + ACTIONS + 4  # float32 features, mask, player, done, status
STEP_OUT = 9                           # reward, done, nagari, status, committed


def work(case):
    kind = case["kind"]
    if kind == "play":  # every step's observation, action and outcome; the rows once
        b = case["batch"]
        return {"bytes": b * (STEPS * (OBSERVED + 8 + STEP_OUT) + 2 * ROW_BYTES + 24), "flops": 0}
    if kind == "env":
        return {"bytes": case["batch"] * (2 * ROW_BYTES + OBSERVED + 16 + 8 + STEP_OUT),
                "flops": 0}
    if kind == "collect":
        step = 2 * ROW_BYTES + 8 + STEP_OUT + 2 * FEATURES + ACTIONS + 4
        return {"bytes": case["batch"] * (step + 3 * ACTIONS + 12), "flops": 0}
    if kind == "branch":
        child = 16 + ROW_BYTES + STEP_OUT + (OBSERVED if case["observe"] else 0)
        return {"bytes": case["children"] * child + case["roots"] * ROW_BYTES, "flops": 0}
    if kind == "canonical":
        return {"bytes": case["games"] * 56, "flops": 0}
    if kind == "actor":
        n, macs = case["rows"], FEATURES * 512 + 6 * 512 * 512 + 512 * (ACTIONS + 1)
        size = 2 if case["dtype"] == "bf16" else 4
        return {"bytes": 2 * macs + n * (FEATURES * size + 2 * ACTIONS + 4), "flops": 2 * n * macs}
    if kind == "decode":
        n, slots, fill = case["rows"], case["slots"], case["fill"]
        # the mean of a uniform length up to 2 fill, cut at 1, in slots
        mean = slots * (fill if fill <= 0.5 else 1 - 1 / (4 * fill))
        size = 4 if case["dtype"] == "f32" else 2
        return {"bytes": n * (2 * mean + 6) * D * size + 16 * n, "flops": 4 * n * mean * D}
    macs = D * 3 * D + D * D + 2 * D * HIDDEN  # one layer, one token
    if kind == "layer":
        n, mean = case["rows"], 23
        return {"bytes": 2 * macs + n * (2 * mean + 4) * 2 * D + 8 * n,
                "flops": n * (2 * macs + 4 * mean * D)}
    w, mean = case["wave"], 20
    query, head = (FEATURES + ACTIONS) * 512 + 512 * D, D * D + D * ACTIONS
    # 3 w tokens through three layers and the in-projection of the fourth, w through the
    # rest of it; one game in five is over, its cache rows are not read
    tokens = w * (3 * (3 * macs + D * 3 * D) + macs - D * 3 * D + query + head)
    cache = 0.8 * w * mean * 2 * 2 * D * (4 + 3 * 2)
    return {"bytes": 2 * (4 * macs + query + head) + cache
            + w * (2 * (FEATURES + ACTIONS) + 2 * 2 * 2 * D + 2 * ACTIONS),
            "flops": 2 * tokens + 4 * 0.8 * w * mean * D * (4 + 3 * 2)}


# ------------------------------------------------------------------- tolerance ----

def tolerance(case):
    kind = case["kind"]
    if kind in ("play", "env", "branch", "canonical"):
        return "exact"  # integers, masks, rows, and features that are exact by contract
    if kind == "collect":  # all of it but the log-probability, a float32 sum over 179
        return {"rel": 1e-6, "max": 1e-5}
    if kind == "actor":    # bf16 operands through eight layers, fp32 sums
        return {"rel": 1.5e-2, "max": 1.2e-1}
    if kind == "decode":   # one rounding of the result to the cache's type
        return {"bf16": {"rel": 6e-3, "max": 3e-2}, "f16": {"rel": 1e-3, "max": 5e-3},
                "f32": {"rel": 2e-6, "max": 2e-5}}[case["dtype"]]
    if kind == "layer":
        return {"rel": 8e-3, "max": 8e-2}
    return {"rel": 2e-2, "max": 2e-1}


# ----------------------------------------------------------------------- exact ----

def _exact_actor(case, seed):
    actor, x = _actor_inputs(case, seed)
    p = {k: v.detach().double() for k, v in actor.state_dict().items()}

    def lin(v, name):
        return F.linear(v, p[name + ".weight"], p[name + ".bias"])

    def norm(v, name):
        return F.layer_norm(v, (512,), p[name + ".weight"], p[name + ".bias"], 1e-5)

    h = lin(x.to(torch.bfloat16).double(), "inp")  # the path's operands are bf16
    for b in range(3):
        z = torch.relu(lin(norm(h, f"blocks.{b}.norm"), f"blocks.{b}.fc1"))
        h = h + lin(z, f"blocks.{b}.fc2")
    z = norm(h, "norm")
    return [lin(z, "logits"), lin(z, "value").squeeze(-1)]


def _exact_attend(q, keys, values, pos, rows, part=64):
    """q [n, heads, dh] over slots 0..pos of cache rows `rows`, in float64; NaN for a
    negative pos."""
    out = torch.empty(q.shape, dtype=torch.float64, device=q.device)
    slots = torch.arange(keys.shape[2], device=q.device)
    for i in range(0, len(q), part):
        at = slice(i, i + part)
        k, v = (t.index_select(0, rows[at]).double() for t in (keys, values))
        s = (k * q[at].double().unsqueeze(2)).sum(-1) * DH ** -0.5
        s = s.masked_fill(slots > pos[at, None, None], -math.inf)
        out[at] = (torch.softmax(s, -1).unsqueeze(-1) * v).sum(2)
    return out


def _exact_layer(layer, x, att_of):
    """One pre-norm encoder layer on x in float64; att_of(q, k, v) attends."""
    p = {k: v.detach().double() for k, v in layer.state_dict().items()}
    n = len(x)
    h = F.layer_norm(x, (D,), p["norm1.weight"], p["norm1.bias"], 1e-5)
    qkv = F.linear(h, p["self_attn.in_proj_weight"], p["self_attn.in_proj_bias"])
    q, k, v = (t.reshape(n, HEADS, DH) for t in qkv.chunk(3, -1))
    a = att_of(q, k, v).reshape(n, D)
    x = x + F.linear(a, p["self_attn.out_proj.weight"], p["self_attn.out_proj.bias"])
    h = F.layer_norm(x, (D,), p["norm2.weight"], p["norm2.bias"], 1e-5)
    u = F.gelu(F.linear(h, p["linear1.weight"], p["linear1.bias"]))
    return x + F.linear(u, p["linear2.weight"], p["linear2.bias"])


def _put(cache, rows, pos, new):
    """new [n, heads, dh] into slot pos[i] of cache row rows[i], where pos >= 0."""
    kept = torch.nonzero(pos >= 0).squeeze(1)
    cache[rows[kept], :, pos[kept]] = new[kept]


@torch.no_grad()
def exact(case, seed):
    kind = case["kind"]
    if kind == "actor":
        return _exact_actor(case, seed)
    if kind == "decode":
        q, kn, vn, keys, values, pos, rows = _decode_inputs(case, seed)
        keys, values = keys.double(), values.double()
        _put(keys, rows, pos, kn.double())
        _put(values, rows, pos, vn.double())
        return [_exact_attend(q, keys, values, pos, rows), keys, values]
    if kind == "layer":
        policy, cache, x = _layer_inputs(case, seed)
        keys, values, pos = cache.k.double(), cache.v.double(), cache.length
        rows = torch.arange(len(x), device="cuda")

        def attend(q, k, v):
            _put(keys[0], rows, pos, k)
            _put(values[0], rows, pos, v)
            return _exact_attend(q, keys[0], values[0], pos, rows)

        return [_exact_layer(policy.encoder.layers[0], x.double(), attend), keys, values]
    if kind != "seqstep":
        return None  # a rules engine: whole numbers, bytes, and features exact by contract
    s = _seq_inputs(case, seed)
    policy, w = s["policy"], s["wave"]
    p = {k: v.detach().double() for k, v in policy.state_dict().items()}
    x = s["pair"].double()
    width = FEATURES + ACTIONS
    u = F.gelu(F.linear(s["q_in"][:, :width].double(), p["query_in.0.weight"],
                        p["query_in.0.bias"]))
    x[2 * w:] = F.linear(u, p["query_in.2.weight"], p["query_in.2.bias"]) + p["token_type"][2]
    rows_e = torch.arange(2 * w, device="cuda")
    keys, values = s["cache"].k.double(), s["cache"].v.double()
    for i, layer in enumerate(policy.encoder.layers):
        def attend(q, k, v, i=i):
            for t, new in ((keys[i], k), (values[i], v)):
                _put(t, rows_e, s["event_pos"], new[:2 * w])
                _put(t, s["query_rows"], s["query_pos"], new[2 * w:])
            # a row's event lies below its query's slot, so one put serves both
            return torch.cat([_exact_attend(q[:2 * w], keys[i], values[i], s["event_pos"], rows_e),
                              _exact_attend(q[2 * w:], keys[i], values[i], s["query_pos"],
                                            s["query_rows"])])

        x = _exact_layer(layer, x, attend)
    z = F.layer_norm(x[2 * w:], (D,), p["norm.weight"], p["norm.bias"], 1e-5)
    u = F.gelu(F.linear(z, p["head.0.weight"], p["head.0.bias"]))
    return [F.linear(u, p["head.2.weight"], p["head.2.bias"]), keys, values]
