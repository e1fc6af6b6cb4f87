"""The work a user has this library do, as cases that can be timed and compared.

Seven kinds of call, each through the public entry points of burn_dragon_amd:

  decode    one greedy token for every sequence of a batch        BDH.forward_with_state, T = 1
  generate  a prompt and a few sampled tokens, one sequence       generation.prefill_state, sample_next_token
  prompt    a ragged prompt through a model on a carried state    BDH.forward_with_state, T > 1
  score     all tokens of a batch at once, no state               BDH.forward_fast
  step      one layer's recurrent state step                      recurrent.recurrent_attention, T = 1
  deferred  a run of state steps with logged updates, flushed     recurrent.state_step_deferred, StateLog.flush
  prefill   a long prompt of one layer in bf16                    recurrent.prefill_chunked, prefill_chunked_ex

Model sizes are those of the shipped configurations, of the test fixtures and of the benchmark; the number of
neurons per head is always multiplier * n_embd / n_head.  Weights are random (projections N(0, 0.02), embedding
N(0, 1)), so about half of a model's neurons fire; the single-layer kinds take activations relu(N(mu, 1)) of a stated
density.
"""
from __future__ import annotations

import math
from statistics import NormalDist

import torch

from burn_dragon_amd import BDH, BDHConfig, RotaryEmbedding, ffi
from burn_dragon_amd.generation import prefill_state, sample_next_token
from burn_dragon_amd.kernel.linear_attention import build_freqs
from burn_dragon_amd.recurrent import (StateLog, prefill_chunked, prefill_chunked_ex, recurrent_attention,
                                       state_step_deferred)

DEVICE = "cuda:0"
THETA = 65536.0


def _model(kind, name, layers, embd, heads, mult, vocab, rotary, **more):
    c = {"kind": kind, "layers": layers, "embd": embd, "heads": heads, "mult": mult, "vocab": vocab, "rotary": rotary}
    c.update(more)
    return {"name": name, **c} if name else c


def _layer(kind, name, batch, heads, latent, embd, **more):
    c = {"kind": kind, "batch": batch, "heads": heads, "latent": latent, "embd": embd}
    c.update(more)
    return {"name": name, **c} if name else c


def listed():
    return [
        # one user typing at the size of the shipped trained checkpoint: the smallest call, all latency
        _model("decode", "decode-checkpoint-b1", 4, 128, 4, 4, 69, "alibi", batch=1, state="f32"),
        # a batch server of the largest shipped configuration, its state kept in bf16
        _model("decode", "decode-large-bf16-b48", 8, 512, 8, 4, 256, "alibi", batch=48, state="bf16"),
        # one sequence through the many-neuron byte model (8192 per head): bound by weights and state rows
        _model("decode", "decode-8192-b1", 6, 256, 4, 128, 256, "rope", batch=1, state="f32"),
        # the largest model of the benchmark (16384 per head, 12 layers), a batch of conversations: 24 GiB of state
        _model("decode", "decode-16384-b8", 12, 512, 8, 256, 256, "rope", batch=8, state="f32"),
        # interactive generation with the default configuration: a 128-token prompt, 16 sampled tokens, the state (kept
        # lazily decayed meanwhile) brought up to date for the next turn
        _model("generate", "generate-default", 6, 256, 4, 4, 256, "alibi", prompt=128, tokens=16, state="f32", lazy=True),
        # ragged follow-up prompts of three conversations of the many-neuron byte model
        _model("prompt", "prompt-8192-b3-t500", 6, 256, 4, 128, 256, "rope", batch=3, time=500, state="f32", lazy=False),
        # scoring held-out text with the base configuration in the stateless form, ragged length
        _model("score", "score-base-b8-t511", 4, 256, 4, 4, 256, "alibi", batch=8, time=511, block=64),
        # the benchmark's headline: one layer, 32 sequences, 5 % of the neurons active
        _layer("step", "step-f32-b32", 32, 4, 8192, 256, rotary="rope", state="f32", density=0.05),
        # the sparsity sweep's middle: wide rows in bf16, denser activations
        _layer("step", "step-bf16-b8", 8, 8, 16384, 512, rotary="rope", state="bf16", density=0.10),
        # the same layer decoding 32 tokens with deferred state updates, flush included
        _layer("deferred", "deferred-f32-b32", 32, 4, 8192, 256, state="f32", density=0.05, steps=32),
        # the long prompt of eight fresh sequences
        _layer("prefill", "prefill-b8-t2048", 8, 4, 8192, 256, time=2048, rotary="rope", density=0.05, fresh=True),
        # ragged follow-up prompts on a carried, decaying state
        _layer("prefill", "prefill-alibi-b3-t777", 3, 4, 4096, 256, time=777, rotary="alibi", density=0.10, fresh=False),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


# layers, embd, heads, largest multiplier drawn for that width
_SIZES = [(4, 128, 4, 128), (4, 192, 4, 64), (4, 256, 4, 128), (6, 256, 4, 128), (8, 512, 8, 128), (12, 512, 8, 256)]


def _draw_model(rng, kind):
    layers, embd, heads, top = rng.choice(_SIZES)
    mult = 4 if rng.random() < 0.4 else _log_int(rng, 4, top)  # the shipped configurations all have 4
    rotary = rng.choice(["rope", "rope", "alibi", "alibi", "pope"])
    return _model(kind, None, layers, embd, heads, mult, rng.choice([69, 256]), rotary)


def draw(rng):
    kind = rng.choice(["decode", "decode", "decode", "generate", "prompt", "score", "step", "step", "deferred", "prefill"])
    if kind in ("decode", "generate", "prompt", "score"):
        c = _draw_model(rng, kind)
        latent = c["mult"] * c["embd"] // c["heads"]
        rows = c["layers"] * c["heads"] * latent * (2 if c["rotary"] == "pope" else 1)  # state rows of one sequence
        if kind == "score":
            c["block"] = rng.choice([64, 64, 128, 0])
        else:
            c["state"] = "bf16" if rng.random() < 0.25 else "f32"
        if kind in ("generate", "prompt"):  # calls after which a lazily decayed state is brought up to date
            c["lazy"] = c["rotary"] == "alibi" and rng.random() < 0.5
        if kind == "generate":
            c["prompt"], c["tokens"] = _log_int(rng, 16, 512), rng.randint(4, 24)
        elif kind == "decode":
            c["batch"] = _log_int(rng, 1, max(1, min(64, (1 << 31) // (rows * c["embd"]))))  # at most 8 GiB of state
        else:
            c["time"] = _log_int(rng, 24, 640)
            most = (3 << 33) // (c["layers"] * c["heads"] * latent * c["embd"])  # tokens: 0.15 TFLOP of projections
            c["time"] = max(16, min(c["time"], most))
            c["batch"] = _log_int(rng, 1, max(1, min(16, most // c["time"], (1 << 31) // (rows * c["embd"]))))
        return c
    heads, embd = rng.choice([(4, 256), (4, 256), (8, 512), (8, 512), (4, 128)])
    latent = _log_int(rng, 4, 256 if embd == 512 else 128) * (embd // heads)
    if kind == "step":
        rotary = rng.choice(["rope", "rope", "rope", "alibi", "pope"])
        rows = heads * latent * (2 if rotary == "pope" else 1)
        return _layer(kind, None, _log_int(rng, 1, max(1, min(64, (1 << 29) // (rows * embd)))), heads, latent, embd,
                      rotary=rotary, state=rng.choice(["f32", "f32", "bf16"]), density=rng.choice([0.01, 0.02, 0.05, 0.1, 0.2, 0.5]))
    if kind == "deferred":
        embd = max(embd, 256)
        return _layer(kind, None, _log_int(rng, 4, max(4, min(64, (1 << 28) // (heads * latent * embd)))), heads, latent, embd,
                      state=rng.choice(["f32", "f32", "bf16"]), density=rng.choice([0.02, 0.05, 0.1, 0.2]),
                      steps=rng.choice([8, 16, 32]))
    rotary = rng.choice(["rope", "rope", "rope", "alibi", "pope"])
    time = _log_int(rng, 64, 2048)
    wide = 2 if rotary == "pope" else 1
    batch = _log_int(rng, 1, max(1, min(16, (1 << 28) // (heads * latent * time * wide))))
    return _layer(kind, None, batch, heads, latent, embd, time=time, rotary=rotary,
                  density=rng.choice([0.05, 0.05, 0.1, 0.3]), fresh=rng.random() < 0.5)


# ---- inputs -----------------------------------------------------------------------------------------------------

def _sizes(case):
    """(latent neurons per head, state rows per head) of a case."""
    n = case["latent"] if "latent" in case else case["mult"] * case["embd"] // case["heads"]
    return n, (2 * n if case.get("rotary") == "pope" else n)


def _relu(g, shape, density, dtype=torch.float32):
    """relu(N(mu, 1)) with `density` of its values above zero, made a batch entry at a time."""
    mu = NormalDist().inv_cdf(density)
    x = torch.empty(shape, device=DEVICE, dtype=dtype)
    for b in range(shape[0]):
        x[b] = torch.relu(torch.randn(shape[1:], device=DEVICE, generator=g) + mu).to(dtype)
    return x


def _state(g, shape, dtype):
    """A state in use: N(0, 0.01)."""
    rho = torch.empty(shape, device=DEVICE, dtype=dtype)
    for part in rho:
        part.normal_(0.0, 0.01, generator=g)
    return rho


def _dtype(case):
    return torch.bfloat16 if case["state"] == "bf16" else torch.float32


def _prepare_model(case, g):
    h, d, V = case["heads"], case["embd"], case["vocab"]
    N, _ = _sizes(case)
    cfg = BDHConfig(n_layer=case["layers"], n_embd=d, n_head=h, mlp_internal_dim_multiplier=case["mult"], vocab_size=V)
    cfg.fused_kernels.set_rotary_embedding(RotaryEmbedding.parse(case["rotary"]))
    if case.get("block"):  # the fused branch with dense time blocks of that size
        cfg.fused_kernels.enabled = True
        cfg.fused_kernels.set_block_sizes(case["block"], case["block"])

    def normal(*shape, std=0.02):
        return std * torch.randn(shape, device=DEVICE, generator=g)

    weights = {"embed": normal(V, d, std=1.0), "encoder": normal(h, d, N), "encoder_v": normal(h, d, N),
               "decoder": normal(h * N, d), "lm_head": normal(d, V)}
    return BDH(cfg, DEVICE, weights=weights, rho_dtype=ffi.BF16 if case.get("state") == "bf16" else ffi.F32,
               alibi_lazy=case.get("lazy", False))


def _conversation(model, case, g, position):
    """A model state as a conversation of `position` tokens leaves it."""
    state = model.init_state()
    state.storage = _state(g, (case["layers"], case["batch"], case["heads"], _sizes(case)[1], case["embd"]), _dtype(case))
    for i, layer in enumerate(state.layers):
        layer.rho = state.storage[i]
    state.position = position
    return state


def prepare(case, seed):
    g = torch.Generator(device=DEVICE).manual_seed(int(seed))
    kind, d = case["kind"], case["embd"]
    s = {"kind": kind, "case": case}
    if kind in ("decode", "generate", "prompt", "score"):
        model = s["model"] = _prepare_model(case, g)
        if kind == "generate":
            s["prompt"] = torch.randint(0, case["vocab"], (case["prompt"],), device=DEVICE, generator=g).tolist()
            s["draws"] = g
            return s
        T = case.get("time", 1)
        s["tokens"] = torch.randint(0, case["vocab"], (case["batch"], T), device=DEVICE, generator=g)
        if kind != "score":
            s["state"] = _conversation(model, case, g, 64 + int(seed) % 1000)
        return s
    B, h, N, Nq = case["batch"], case["heads"], *_sizes(case)
    s["position"] = 64 + (int(seed) * 7919) % 4000
    s["rotary"] = RotaryEmbedding.parse(case.get("rotary", "rope"))
    s["freqs"] = build_freqs(N, THETA, s["rotary"], device=DEVICE).reshape(-1)
    if kind == "step":
        s["x"] = _relu(g, (B, h, 1, N), case["density"])
        s["v"] = torch.randn((B, 1, d), device=DEVICE, generator=g)
        s["rho"] = _state(g, (B, h, Nq, d), _dtype(case))
    elif kind == "deferred":
        s["x"] = [_relu(g, (B, h, N), case["density"]) for _ in range(case["steps"])]
        s["v"] = [torch.randn((B, d), device=DEVICE, generator=g) for _ in range(case["steps"])]
        s["rho"] = _state(g, (B, h, N, d), _dtype(case))
        s["log"] = StateLog(B, h, N, d, _dtype(case), case["steps"])
    else:
        T = case["time"]
        s["x"] = _relu(g, (B, h, T, N), case["density"], torch.bfloat16)
        s["v"] = torch.randn((B, T, d), device=DEVICE, generator=g).to(torch.bfloat16)
        s["rho"] = torch.zeros((B, h, Nq, d), device=DEVICE) if case["fresh"] else _state(g, (B, h, Nq, d), torch.float32)
    return s


# ---- one pass ---------------------------------------------------------------------------------------------------

def run(s):
    kind, case = s["kind"], s["case"]
    if kind == "decode":  # the token just chosen is the next call's input; it stays on the device
        logits, s["tokens"] = s["model"].forward_with_state(s["tokens"].reshape(-1, 1), s["state"], want_next=True)
        return logits, s["tokens"], s["state"].storage
    if kind == "generate":
        state, last = prefill_state(s["model"], s["prompt"])
        tokens = []
        for _ in range(case["tokens"]):
            token, last = sample_next_token(s["model"], state, last, 0.8, 40, s["draws"])
            tokens.append(token)
        s["model"].materialize_state(state)  # nothing to do unless lazily decayed
        return torch.cat(tokens), last, state.storage
    if kind == "prompt":
        logits = s["model"].forward_with_state(s["tokens"], s["state"])
        s["model"].materialize_state(s["state"])
        return logits, s["state"].storage
    if kind == "score":
        return s["model"].forward_fast(s["tokens"])
    if kind == "step":
        out = recurrent_attention(s["x"], s["v"], s["rho"], s["freqs"], s["position"], s["rotary"])
        s["position"] += 1
        return out, s["rho"]
    if kind == "deferred":
        outs = []
        for x, v in zip(s["x"], s["v"]):
            outs.append(state_step_deferred(s["log"], x, v, s["rho"], s["freqs"], s["position"]))
            s["position"] += 1
        s["log"].flush(s["rho"])
        return outs, s["rho"]
    fresh, position = case["fresh"], 0 if case["fresh"] else s["position"]
    if s["rotary"] == RotaryEmbedding.ROPE:
        out = prefill_chunked(s["x"], s["v"], s["rho"], s["freqs"], position, state_is_zero=fresh)
    else:
        out = prefill_chunked_ex(s["x"], s["v"], s["rho"], s["freqs"], position, rotary=s["rotary"], state_is_zero=fresh)
    if not fresh:
        s["position"] += case["time"]
    return out, s["rho"]


# ---- what a pass cannot do without ------------------------------------------------------------------------------

def _touched(case, density):
    """Share of the state rows that one token reads and writes: the pair-closed active rows under RoPE, the active
    rows of a lazily decayed state, every row where the whole state decays or carries a row for every neuron."""
    if case.get("rotary", "rope") == "rope":
        return 1.0 - (1.0 - density) ** 2
    return density if case.get("lazy") else 1.0


def work(case):
    h, d = case["heads"], case["embd"]
    N, Nq = _sizes(case)
    if case["kind"] in ("decode", "generate", "prompt", "score"):
        B = case.get("batch", 1)
        T = {"decode": 1, "generate": case.get("prompt", 0) + case.get("tokens", 0)}.get(case["kind"], case.get("time", 0))
        es = 2 if case.get("state") == "bf16" else 4
        M, L, V, rows = B * T, case["layers"], case["vocab"], case["layers"] * B * h * Nq
        weights = 4.0 * (3 * h * N * d + d * V)
        # D_x for every neuron, D_y for the half that fires, E for the quarter that passes both
        flops = 2.0 * M * (L * 1.75 * h * N * d + d * V)
        if case["kind"] == "score":  # causal scores and their product with the values
            return {"bytes": weights + 4.0 * M * (d + V), "flops": flops + L * B * h * float(T) * (T - 1) * (Nq + d)}
        if case["kind"] == "generate":  # the weights and the active state rows again for every token drawn
            share = _touched(case, 0.5)
            n = case["tokens"]
            return {"bytes": weights * (1 + n) + es * d * rows * (1 + 2.0 * n * share) + 4.0 * (n + 1) * (d + V),
                    "flops": flops + 4.0 * M * L * h * Nq * d * share}
        share = _touched(case, 0.5) if T == 1 else 1.0
        return {"bytes": weights + 2.0 * es * d * rows * share + 4.0 * M * (d + V),
                "flops": flops + 4.0 * M * L * h * Nq * d * _touched(case, 0.5)}
    B = case["batch"]
    slices = float(B * h)
    if case["kind"] == "step":
        share = _touched(case, case["density"])
        es = 2 if case["state"] == "bf16" else 4
        return {"bytes": slices * (2.0 * Nq * d * es * share + 4 * N + 4 * d) + 4.0 * (B * d + N), "flops": slices * 4.0 * Nq * d * share}
    if case["kind"] == "deferred":  # a step reads its rows; the rows any step touched are written once
        K, es = case["steps"], 2 if case["state"] == "bf16" else 4
        one = _touched(case, case["density"])
        union = 1.0 - (1.0 - one) ** K
        return {"bytes": slices * (Nq * d * es * (K * one + 2.0 * union) + K * (4 * N + 4 * d)) + 4.0 * K * B * d,
                "flops": slices * 4.0 * Nq * d * one * K}
    T = case["time"]
    return {"bytes": slices * (2.0 * T * N + 4.0 * T * d + (4.0 if case["fresh"] else 8.0) * Nq * d) + 2.0 * B * T * d,
            "flops": slices * (float(T) * (T - 1) * (Nq + d) + (2.0 if case["fresh"] else 4.0) * T * Nq * d)}


def tolerance(case):
    """About four times what the library's own forms of a call differ by (another order of the sums, another form of
    the same products), over these cases and two dozen drawn ones.  Seen: model steps in f32 5e-6 (largest element
    1e-4 of the root mean square), prompts 8e-7, single layers 1e-6; a bf16 state 1e-5 in one layer and 2e-4 through a
    model where each token is rounded alike, 8e-3 where a prompt is rounded once at its end instead of after every
    token; the bf16 prefill against f32 products 2e-3 (largest element 3e-2)."""
    kind, bf16 = case["kind"], case.get("state") == "bf16"
    if kind == "prefill":
        return {"rel": 8e-3, "max": 0.1}
    if bf16 and kind in ("step", "deferred"):
        return {"rel": 1e-4, "max": 3e-2}
    if bf16:
        return {"rel": 8e-4, "max": 6e-2, "differ": 0.01} if kind == "decode" else {"rel": 3e-2, "differ": 0.01}
    if kind in ("decode", "generate", "prompt"):
        return {"rel": 2e-5, "max": 4e-4, "differ": 0.01}
    return {"rel": 1e-5, "max": 1e-4}
