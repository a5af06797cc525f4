"""The calls whose speed this library is judged by: what a speech program
does with it through voxcpm_amd.ops, at VoxCPM2's shapes.

Every patch of speech takes one base-LM step, one DiT patch, one AudioVAE
chunk and one local-encoder call; a request takes an LM and an encoder
prefill before, and a program that does not stream decodes the whole
utterance at the end. The products and the attention are called on their own
too, over the rows that all of these give them.
"""
from __future__ import annotations

import dataclasses
import functools
import math

import torch

from voxcpm_amd import ops, synth

STACKS = {"base_lm": synth.VOXCPM2_BASE_LM, "residual_lm": synth.VOXCPM2_RESIDUAL_LM,
          "encoder": synth.VOXCPM2_ENCODER}
DITS = {"synthetic": synth.SYNTHETIC_DIT, "voxcpm2": synth.VOXCPM2_DIT}
VAE = synth.VOXCPM2_VAE
ROPE_POSITIONS = 4096


def listed() -> list[dict]:
    return [
        # The smallest call: one decode row through a 2048 x 2048 projection.
        dict(name="linear_row", kind="linear", weights="q8", m=1, k=2048, n=2048, out="f32"),
        # The DiT's 22 rows (two 11-row branches) through gate_up.
        dict(name="linear_dit", kind="linear", weights="q8", m=22, k=1024, n=8192, out="f32"),
        # A short prompt, rows and columns that fill no tile.
        dict(name="linear_ragged", kind="linear", weights="q8", m=77, k=6144, n=2055, out="f32"),
        # A long prompt through the LM's gate_up.
        dict(name="linear_prefill", kind="linear", weights="q8", m=777, k=2048, n=12288,
             out="f32"),
        # The checkpoint's own bf16 weights: the encoder's down projection.
        dict(name="linear_bf16", kind="linear", weights="bf16", m=333, k=4096, n=1024,
             out="f32"),
        # A second chunk of a long prompt: 300 rows behind 1500 cached keys.
        dict(name="attention_chunk", kind="attention", rows=300, sequences=1, past=1500,
             causal=True, heads=16, kv_heads=2, head_dim=128),
        # One whole decode step of the base LM, 1000 positions in.
        dict(name="lm_step", kind="stack", stack="base_lm", weights="q8", layers=28, rows=1,
             sequences=1, past=1000),
        # Two layers of the base LM over a prompt.
        dict(name="lm_prefill", kind="stack", stack="base_lm", weights="q8", layers=2, rows=617,
             sequences=1, past=0),
        # The local encoder over a 10 s voice prompt: 62 patches of 5 rows.
        dict(name="encoder_prompt", kind="stack", stack="encoder", weights="q8", layers=12,
             rows=310, sequences=62, past=0),
        # One whole patch of the sampler: ten steps of the released DiT.
        dict(name="dit_patch", kind="dit", dit="voxcpm2", weights="q8", call="patch"),
        # One patch's audio while streaming: 4 frames, the stream going on.
        dict(name="vae_patch", kind="vae", frames=4, reset=False),
        # A whole utterance decoded at once: 5 s of speech, a new stream.
        dict(name="vae_utterance", kind="vae", frames=125, reset=True),
    ]


def _log_int(rng, low: int, high: int) -> int:
    return min(high, int(math.exp(rng.uniform(math.log(low), math.log(high + 1)))))


def draw(rng) -> dict:
    kind = rng.choice(("linear", "linear", "attention", "stack", "stack", "dit", "vae"))
    if kind == "linear":
        weights = rng.choice(("q8", "q8", "bf16", "bf16_rows"))
        m = _log_int(rng, 1, 32 if weights == "bf16_rows" else 1024)
        k = 32 * _log_int(rng, 2, 192)
        return dict(kind=kind, weights=weights, m=m, k=k,
                    n=_log_int(rng, 64, min(16384, (1 << 25) // k)),
                    out=rng.choice(("f32", "f32", "bf16")) if weights == "q8" else "f32")
    if kind == "attention":
        heads, kv_heads, head_dim = rng.choice(((16, 2, 128), (16, 2, 128), (16, 16, 64),
                                                (8, 1, 128)))
        if rng.random() < 0.25:  # an encoder's patches
            sequences = _log_int(rng, 1, 120)
            return dict(kind=kind, rows=5 * sequences, sequences=sequences, past=0,
                        causal=False, heads=heads, kv_heads=kv_heads, head_dim=head_dim)
        return dict(kind=kind, rows=_log_int(rng, 1, 700), sequences=1,
                    past=rng.choice((0, _log_int(rng, 1, 1600))), causal=True, heads=heads,
                    kv_heads=kv_heads, head_dim=head_dim)
    if kind == "stack":
        stack = rng.choice(tuple(STACKS))
        weights = rng.choice(("q8", "q8", "bf16"))
        if stack == "encoder":
            sequences = _log_int(rng, 1, 120)
            return dict(kind=kind, stack=stack, weights=weights, layers=rng.randint(1, 4),
                        rows=5 * sequences, sequences=sequences, past=0)
        rows = _log_int(rng, 1, 800)
        return dict(kind=kind, stack=stack, weights=weights,
                    layers=rng.randint(1, 4 if rows < 200 else 1), rows=rows, sequences=1,
                    past=rng.choice((0, _log_int(rng, 1, 1600))))
    if kind == "dit":
        call = rng.choice(("velocity", "patch"))
        return dict(kind=kind, dit=rng.choice(tuple(DITS)), call=call,
                    weights="q8" if call == "patch" else rng.choice(("q8", "bf16")))
    return dict(kind=kind, frames=_log_int(rng, 1, 125), reset=rng.random() < 0.5)


# ---- inputs ----------------------------------------------------------------

class _Random:
    """Seeded device tensors with the laws of synth (see there)."""

    def __init__(self, seed: int):
        self.generator = torch.Generator(device="cuda")
        self.generator.manual_seed(seed)

    def normal(self, *shape, std: float = 1.0, mean: float = 0.0) -> torch.Tensor:
        return torch.randn(shape, device="cuda", generator=self.generator) * std + mean

    def blocks(self, n: int, k: int) -> torch.Tensor:
        """GGML Q8_0 blocks [n][k / 32][34]."""
        q = torch.randint(-127, 128, (n, k // 32, 32), dtype=torch.int8, device="cuda",
                          generator=self.generator)
        scale = (self.normal(n, k // 32).abs() * (0.02 / 127)).to(torch.float16)
        return torch.cat((scale.view(torch.uint8).view(n, k // 32, 2), q.view(torch.uint8)), 2)

    def bits(self, count: int, mean: float) -> torch.Tensor:
        """bf16 bits (int16) ~ N(mean, 0.02)."""
        return self.normal(count, std=0.02, mean=mean).to(torch.bfloat16).view(torch.int16)


def _layers(config, random: _Random) -> list[dict]:
    h = config.hidden
    return [{"input_norm": random.bits(h, 1.0), "qkv": random.blocks(config.qkv_width, h),
             "o": random.blocks(h, config.q_width), "post_norm": random.bits(h, 1.0),
             "gate_up": random.blocks(2 * config.ffn, h), "down": random.blocks(h, config.ffn)}
            for _ in range(config.layers)]


def _stack_config(case):
    return dataclasses.replace(STACKS[case["stack"]], layers=case["layers"])


def _stack_inputs(case, seed):
    """(config, weights, hidden, k cache, v cache, positions, cache rows)."""
    config, random = _stack_config(case), _Random(seed)
    weights = synth.StackWeightsHost(config, _layers(config, random),
                                     random.bits(config.hidden, 1.0))
    rows, past = case["rows"], case["past"]
    per_sequence = rows // case["sequences"]
    hidden = random.normal(rows, config.hidden)
    shape = (config.layers, config.kv_heads, past + rows, config.head_dim)
    caches = [random.normal(*shape, std=0.5) for _ in range(2)]
    cache_rows = torch.arange(past, past + rows, dtype=torch.int32, device="cuda")
    positions = past + (torch.arange(rows, dtype=torch.int32, device="cuda") % per_sequence)
    return config, weights, hidden, *caches, positions, cache_rows


def _dit_inputs(case, seed):
    """(config, device weights by name, mu, cond latent, noise)."""
    config, random = DITS[case["dit"]], _Random(seed)
    tensors = {"layers": _layers(config, random), "norm": random.bits(config.hidden, 1.0)}
    for name in synth.PROJECTIONS:
        if config.has_delta or not name.startswith("delta"):
            out, inner = synth.projection_shape(config, name)
            tensors[name] = (random.blocks(out, inner), random.bits(out, 0.0))
    mu = random.normal(2 * config.hidden).bfloat16().float()
    cond = random.normal(config.patch, config.feat).bfloat16().float()
    return config, tensors, mu, cond, random.normal(config.patch, config.feat)


def _vae_weights(random: _Random):
    def alpha(c):
        return random.normal(c, std=0.1, mean=1.0).abs() + 0.05

    t = {"in_depthwise": random.normal(VAE.latent, 7, std=7 ** -0.5),
         "in_depthwise_bias": random.normal(VAE.latent, std=0.02),
         "in_pointwise": random.normal(VAE.decoder_dim, VAE.latent, std=VAE.latent ** -0.5),
         "in_pointwise_bias": random.normal(VAE.decoder_dim, std=0.02), "blocks": []}
    for b, s in enumerate(VAE.rates):
        c_in, c = VAE.channels(b)
        units = [{"alpha_in": alpha(c), "depthwise": random.normal(c, 7, std=7 ** -0.5),
                  "depthwise_bias": random.normal(c, std=0.02), "alpha_out": alpha(c),
                  "pointwise": random.normal(c, c, std=0.5 * c ** -0.5),
                  "pointwise_bias": random.normal(c, std=0.02)} for _ in range(3)]
        t["blocks"].append({"stride": s, "scale": random.normal(c_in, std=0.05, mean=1.0),
                            "bias": random.normal(c_in, std=0.05), "alpha": alpha(c_in),
                            "up": random.normal(c_in, c, 2 * s, std=(2 * c_in) ** -0.5),
                            "up_bias": random.normal(c, std=0.02), "units": units})
    c = VAE.channels(len(VAE.rates) - 1)[1]
    t["out_alpha"] = alpha(c)
    t["out_conv"] = random.normal(c, 7, std=(7 * c) ** -0.5)
    t["out_bias"] = 0.01
    return synth.VaeWeightsHost(VAE, t)


def _vae_inputs(case, seed):
    random = _Random(seed)
    return _vae_weights(random), random.normal(case["frames"], VAE.latent)


def _linear_inputs(case, seed):
    """(x bf16, weights: Q8_0 blocks or bf16 rows)."""
    random = _Random(seed)
    x = random.normal(case["m"], case["k"]).bfloat16()
    if case["weights"] == "q8":
        return x, random.blocks(case["n"], case["k"])
    return x, random.normal(case["n"], case["k"], std=0.02).bfloat16()


def _attention_inputs(case, seed):
    """(q, k cache, v cache): scores spread by about two."""
    random = _Random(seed)
    heads, kv_heads, d = case["heads"], case["kv_heads"], case["head_dim"]
    keys = case["past"] + case["rows"]
    return (random.normal(case["rows"], heads, d, std=1.4),
            random.normal(kv_heads, keys, d, std=1.4), random.normal(kv_heads, keys, d))


def prepare(case, seed):
    # One stream for all work, set once, as a serving program has it (the
    # stacks, the DiT and the decoder replay their graphs on streams only).
    torch.cuda.set_stream(_stream())
    kind = case["kind"]
    if kind == "linear":
        x, w = _linear_inputs(case, seed)
        n, k = case["n"], case["k"]
        packed = ops.q8_pack(w, n, k) if case["weights"] == "q8" else \
            ops.bf16_pack(w) if case["weights"] == "bf16" else w
        return case, (x, packed, _scratch())
    if kind == "attention":
        return case, _attention_inputs(case, seed)
    if kind == "stack":
        config, weights, hidden, k, v, positions, cache_rows = _stack_inputs(case, seed)
        stack = ops.Stack(weights, _rope(config, torch.float32).cpu().numpy()
                          if config.rope else None, bf16_weights=case["weights"] == "bf16")
        return case, (stack, hidden, torch.empty_like(hidden), torch.empty_like(hidden),
                      positions, cache_rows, k, v)
    if kind == "dit":
        config, tensors, mu, cond, noise = _dit_inputs(case, seed)
        host = synth.DitWeightsHost(
            config, [{name: _host(t) for name, t in layer.items()}
                     for layer in tensors["layers"]], _host(tensors["norm"]),
            {name: (_host(tensors[name][0]), _host(tensors[name][1]))
             for name in synth.PROJECTIONS if name in tensors},
            _rope(config, torch.float32)[:3 + 2 * config.patch].cpu().numpy())
        dit = ops.Dit(host, bf16_weights=case["weights"] == "bf16")
        schedule = ops.euler_schedule(config.steps, config.sway, config.skip)
        return case, (dit, config, mu, cond, noise, torch.empty_like(noise), schedule)
    weights, latents = _vae_inputs(case, seed)
    vae = ops.Vae(weights)
    return case, (vae, latents, torch.empty(case["frames"] * VAE.hop, device="cuda"))


def run(state):
    case, held = state
    kind = case["kind"]
    if kind == "linear":
        x, w, scratch = held
        if case["weights"] == "bf16_rows":
            return ops.bf16_linear_rows(x, w)
        if case["weights"] == "bf16":
            return ops.bf16_linear(x, w, case["n"], scratch=scratch)
        if case["out"] == "bf16":
            return ops.q8_linear_bf16(x, w, case["n"], scratch=scratch)
        return ops.q8_linear(x, w, case["n"], scratch=scratch)
    if kind == "attention":
        q, k, v = held
        per_sequence = case["rows"] // case["sequences"]
        return ops.split_attention(q, k, v, per_sequence, per_sequence, case["past"],
                                   case["causal"], case["heads"], case["kv_heads"])
    if kind == "stack":
        stack, embedded, hidden, output, positions, cache_rows, k, v = held
        per_sequence = case["rows"] // case["sequences"]
        hidden.copy_(embedded)  # the step's embeddings
        stack.forward(hidden, output, positions, cache_rows, per_sequence, per_sequence,
                      case["past"], case["stack"] != "encoder", k, v)
        return {"hidden": hidden, "output": output, "k": k, "v": v}
    if kind == "dit":
        dit, config, mu, cond, noise, x, (t, dt, evaluate) = held
        if case["call"] == "velocity":
            return dit.velocity(mu, cond, noise, 0.63)
        x.copy_(noise)
        return dit.patch(mu, cond, x, t, dt, evaluate, config.cfg, config.zero_star)
    vae, latents, samples = held
    if case["reset"]:
        vae.reset()
    return vae.decode(latents, samples)


# ---- what a pass cannot do without -------------------------------------------

def _weight_bytes(n: int, k: int, weights: str) -> float:
    return n * k * (34 / 32 if weights == "q8" else 2)


def _layer_work(config, rows: int, pairs: int, weights: str) -> tuple[float, float]:
    """(weight bytes, flops) of one layer; `pairs`: attended (row, key)s."""
    matrices = ((config.qkv_width, config.hidden), (config.hidden, config.q_width),
                (2 * config.ffn, config.hidden), (config.hidden, config.ffn))
    return (sum(_weight_bytes(n, k, weights) for n, k in matrices),
            sum(2.0 * rows * n * k for n, k in matrices) + 4.0 * pairs * config.q_width)


def _pairs(case, causal: bool) -> int:
    per_sequence = case["rows"] // case["sequences"]
    own = per_sequence * (per_sequence + 1) // 2 if causal else per_sequence ** 2
    return case["sequences"] * own + case["rows"] * case["past"]


def work(case) -> dict:
    kind = case["kind"]
    if kind == "linear":
        m, k, n = case["m"], case["k"], case["n"]
        return {"bytes": 2 * m * k + _weight_bytes(n, k, case["weights"]) +
                (2 if case["out"] == "bf16" else 4) * m * n, "flops": 2.0 * m * n * k}
    if kind == "attention":
        width = case["heads"] * case["head_dim"]
        keys = case["past"] + case["rows"]
        return {"bytes": 6 * case["rows"] * width + 8 * keys * case["kv_heads"] * case["head_dim"],
                "flops": 4.0 * _pairs(case, case["causal"]) * width}
    if kind == "stack":
        config = _stack_config(case)
        weight_bytes, flops = _layer_work(config, case["rows"],
                                          _pairs(case, case["stack"] != "encoder"),
                                          case["weights"])
        cache = 8 * (case["past"] + case["rows"]) * config.kv_heads * config.head_dim
        return {"bytes": config.layers * (weight_bytes + cache) + 12 * case["rows"] * config.hidden,
                "flops": config.layers * flops}
    if kind == "dit":
        config = DITS[case["dit"]]
        branch = 3 + 2 * config.patch
        weight_bytes, flops = _layer_work(config, 2 * branch, 2 * branch ** 2, case["weights"])
        # The ten evaluations' weights fit no cache nearer than memory.
        calls = 1 if case["call"] == "velocity" else config.steps - int(config.skip)
        return {"bytes": calls * config.layers * weight_bytes,
                "flops": calls * config.layers * flops}
    t, weight_bytes, flops = case["frames"], 0.0, 0.0
    for b, s in enumerate(VAE.rates):
        c_in, c = VAE.channels(b)
        weight_bytes += 4 * (2 * s * c_in * c + 3 * (c * c + 7 * c))
        flops += 2.0 * t * s * c * 2 * c_in
        t *= s
        flops += 3 * 2.0 * t * c * (c + 7)
    return {"bytes": weight_bytes + 4 * (t + case["frames"] * VAE.latent), "flops": flops}


def tolerance(case) -> dict:
    """About four times the 2-norm errors measured against exact() over the
    listed and drawn cases (`max`: the largest of that many normal errors)."""
    kind = case["kind"]
    if kind == "linear":
        if case["weights"] == "q8" and case["m"] > 128:
            return {"rel": 7e-3, "max": 0.04}  # weights rounded to bf16 (1.7e-3)
        if case["out"] == "bf16":
            return {"rel": 7e-3, "max": 0.016}  # the output rounded to bf16 (1.6e-3)
        return {"rel": 5e-7, "max": 1e-5}      # float32 sums (1.4e-7)
    if kind == "attention":
        return {"rel": 7e-3, "max": 0.016}     # the output rounded to bf16 (1.7e-3)
    if kind in ("stack", "dit"):
        return {"rel": 1e-2, "max": 0.06}      # bf16 operands through the layers (2.5e-3)
    return {"rel": 2e-4, "max": 6e-3}          # float32, the Snakes amplifying (4.7e-5)


# ---- the same in 64 bits -------------------------------------------------------

def _values(blocks: torch.Tensor) -> torch.Tensor:
    """GGML Q8_0 blocks -> float64 [n][k]."""
    scale = blocks[..., :2].contiguous().view(torch.float16).double()
    return (blocks[..., 2:].view(torch.int8).double() * scale).flatten(1)


def _matrix(blocks: torch.Tensor, weights: str) -> torch.Tensor:
    values = _values(blocks)
    return values.bfloat16().double() if weights == "bf16" else values


def _vector(bits: torch.Tensor) -> torch.Tensor:
    return bits.view(torch.bfloat16).double()


def _rms(h, gamma, eps):
    return h * torch.rsqrt(h.square().mean(-1, keepdim=True) + eps) * _vector(gamma)


def _attend(q, k, v, past: int, causal: bool):
    """q [s][h][r][d], k and v [s][kv][keys][d] -> [s][r][h d]."""
    group = q.shape[1] // k.shape[1]
    k, v = (x.repeat_interleave(group, 1).contiguous() for x in (k, v))
    scores = torch.matmul(q, k.transpose(-1, -2).contiguous()) / math.sqrt(q.shape[-1])
    if causal:
        r, keys = scores.shape[-2:]
        later = torch.arange(keys, device="cuda") > past + torch.arange(r, device="cuda")[:, None]
        scores = scores.masked_fill(later, -math.inf)
    return torch.matmul(scores.softmax(-1), v).transpose(1, 2).flatten(2)


def _rotate(x, table):
    half = x.shape[-1] // 2
    c, s = table[:, :half], table[:, half:]
    a, b = x[..., :half], x[..., half:]
    return torch.cat((a * c - b * s, b * c + a * s), -1)


def _layer(config, layer, h, past_k, past_v, table, weights: str, causal: bool):
    """h [s][r][hidden] float64 through one layer: (h, k, v) with k and v
    [s][kv][r][d]; past_k and past_v [kv][past][d] (one sequence) or None."""
    s, r, _ = h.shape
    qkv = _rms(h, layer["input_norm"], config.eps) @ _matrix(layer["qkv"], weights).t()
    qkv = qkv.view(s, r, -1, config.head_dim).transpose(1, 2)
    q, k, v = qkv.split((config.heads, config.kv_heads, config.kv_heads), 1)
    if table is not None:
        q, k = _rotate(q, table), _rotate(k, table)
    past = 0 if past_k is None else past_k.shape[1]
    keys = k if past == 0 else torch.cat((past_k[None], k), 2)
    values = v if past == 0 else torch.cat((past_v[None], v), 2)
    h = h + _attend(q, keys, values, past, causal) @ _matrix(layer["o"], weights).t()
    gate, up = (_rms(h, layer["post_norm"], config.eps) @
                _matrix(layer["gate_up"], weights).t()).chunk(2, -1)
    h = h + (torch.nn.functional.silu(gate) * up) @ _matrix(layer["down"], weights).t()
    return h, k, v


def _rope(config, dtype) -> torch.Tensor:
    half = config.head_dim // 2
    factors = torch.tensor(config.rope_factors or [1.0] * half, dtype=torch.float64)
    inverse = config.rope_theta ** (-torch.arange(half, dtype=torch.float64) / half) / factors
    angle = torch.arange(ROPE_POSITIONS, dtype=torch.float64)[:, None] * inverse
    return (torch.cat((angle.cos(), angle.sin()), 1) * config.rope_scaling).to("cuda", dtype)


def exact(case, seed):
    torch.cuda.set_stream(_stream())
    return {"linear": _exact_linear, "attention": _exact_attention, "stack": _exact_stack,
            "dit": _exact_dit, "vae": _exact_vae}[case["kind"]](case, seed)


def _exact_linear(case, seed):
    x, w = _linear_inputs(case, seed)
    return x.double() @ (_values(w) if case["weights"] == "q8" else w.double()).t()


def _exact_attention(case, seed):
    q, k, v = (t.double() for t in _attention_inputs(case, seed))
    s, d = case["sequences"], case["head_dim"]
    q = q.view(s, -1, case["heads"], d).transpose(1, 2).contiguous()
    k, v = (t.view(case["kv_heads"], s, -1, d).transpose(0, 1).contiguous() for t in (k, v))
    return _attend(q, k, v, case["past"], case["causal"]).view(case["rows"], case["heads"], d)


def _exact_stack(case, seed):
    config, weights, hidden, k_cache, v_cache, positions, _ = _stack_inputs(case, seed)
    sequences, past = case["sequences"], case["past"]
    table = _rope(config, torch.float64)[positions[:case["rows"] // sequences].long()] \
        if config.rope else None
    h = hidden.double().view(sequences, -1, config.hidden)
    k_cache, v_cache = k_cache.double(), v_cache.double()
    for i, layer in enumerate(weights.layers):
        h, k, v = _layer(config, layer, h, k_cache[i, :, :past] if past else None,
                         v_cache[i, :, :past] if past else None, table, case["weights"],
                         case["stack"] != "encoder")
        for cache, new in ((k_cache, k), (v_cache, v)):
            cache[i, :, past:] = new.transpose(0, 1).flatten(1, 2)
    h = h.view(-1, config.hidden)
    return {"hidden": h, "output": _rms(h, weights.norm, config.eps), "k": k_cache, "v": v_cache}


def _exact_dit(case, seed):
    config, tensors, mu, cond, x = _dit_inputs(case, seed)
    branch = 3 + 2 * config.patch
    table = _rope(config, torch.float64)[:branch]
    silu = torch.nn.functional.silu

    def project(name, value):
        blocks, bias = tensors[name]
        return value @ _matrix(blocks, case["weights"]).t() + _vector(bias)

    def embed(t, first, second):
        half = config.time_in // 2
        frequency = torch.exp(torch.arange(half, dtype=torch.float64, device="cuda") *
                              (-math.log(10000.0) / (half - 1)))
        angle = 1000.0 * t * frequency
        return project(second, silu(project(first, torch.cat((angle.sin(), angle.cos())))))

    def velocity(x, t):
        time = embed(t, "time_1", "time_2")
        if config.has_delta:
            time = time + embed(0.0, "delta_1", "delta_2")
        head = mu.double().view(2, -1)
        h = torch.stack([torch.cat((m, time[None], project("cond_proj", cond.double()),
                                    project("in_proj", x))) for m in (head, 0 * head)])
        for layer in tensors["layers"]:
            h, _, _ = _layer(config, layer, h, None, None, table, case["weights"], False)
        return project("out_proj", _rms(h, tensors["norm"], config.eps)[:, 3 + config.patch:])

    x = x.double()
    if case["call"] == "velocity":
        return velocity(x, 0.63)
    for t, dt, evaluate in zip(*_schedule(config)):
        if evaluate:
            c, u = velocity(x, t)
            scale = (c * u).sum() / (u.square().sum() + 1e-8) if config.zero_star else 1.0
            x = x - dt * (u * scale + config.cfg * (c - u * scale))
    return x


def _schedule(config):
    """(t, dt, evaluate) of the Euler steps from t = 1 to 0."""
    span = [1.0 - i / config.steps for i in range(config.steps + 1)]
    span = [s + config.sway * (math.cos(math.pi / 2 * s) - 1.0 + s) for s in span]
    skipped = max(1, int((config.steps + 1) * 0.04)) if config.skip else 0
    return (span[:-1], [a - b for a, b in zip(span, span[1:])],
            [step >= skipped for step in range(config.steps)])


def _exact_vae(case, seed):
    weights, x = _vae_inputs(case, seed)
    t = weights.tensors

    def snake(y, alpha):
        return y + torch.sin(alpha.double() * y).square() / (alpha.double() + 1e-9)

    def depthwise(y, w, b, d):
        padded = torch.cat((y.new_zeros(6 * d, y.shape[1]), y))
        return b.double() + sum(padded[j * d:j * d + len(y)] * w[:, j].double() for j in range(7))

    y = depthwise(x.double(), t["in_depthwise"], t["in_depthwise_bias"], 1)
    y = y @ t["in_pointwise"].double().t() + t["in_pointwise_bias"].double()
    for block in t["blocks"]:
        s = block["stride"]
        u = snake(y * block["scale"].double() + block["bias"].double(), block["alpha"])
        before = torch.cat((u.new_zeros(1, u.shape[1]), u[:-1]))
        up = block["up"].double().permute(2, 0, 1)  # [2 s][in][out]
        y = torch.stack([u @ up[r].contiguous() + before @ up[r + s].contiguous()
                         for r in range(s)], 1).flatten(0, 1) + block["up_bias"].double()
        for unit, d in zip(block["units"], (1, 3, 9)):
            v = snake(depthwise(snake(y, unit["alpha_in"]), unit["depthwise"],
                                unit["depthwise_bias"], d), unit["alpha_out"])
            y = y + v @ unit["pointwise"].double().t() + unit["pointwise_bias"].double()
    y = snake(y, t["out_alpha"])
    padded = torch.cat((y.new_zeros(6, y.shape[1]), y))
    out = sum(padded[j:j + len(y)] @ t["out_conv"][:, j].double() for j in range(7))
    return torch.tanh(out + t["out_bias"])


# ---- kept by the program ---------------------------------------------------------

@functools.cache
def _stream() -> torch.cuda.Stream:
    return torch.cuda.Stream()


@functools.cache
def _scratch() -> ops.Scratch:
    return ops.Scratch(128, 16384)


def _host(tensor: torch.Tensor):
    array = tensor.cpu().numpy()
    return array.view("u2") if array.dtype == "int16" else array
