"""The work that a user of this package has it do, as cases with sizes: what a performance measurement runs.

Every case goes through the public entry points of the package.  Six kinds of work:

* ``linear``      one W4A4 linear layer (``FourOverSixLinear``): activation quantized on the fly, GEMM, bias;
* ``quantize``    ``quantize_to_fp4`` of a bf16 tensor (activations as they come, weights at bring-up);
* ``dequantize``  ``QuantizedTensor.dequantize`` (checkpoint export, inspection, comparison runs);
* ``kv_step``     what one layer does with one chunk: attention over [FP4 cache slots | chunk], then the chunk's K and V
                  written into their slot, with absolute or relative RoPE;
* ``block``       one transformer block of a denoising forward against a filled cache;
* ``generate``    the chunk loop of the streaming generator from noise to latents: denoising forwards, clean-context
                  pass, cache fill and roll, with either sampler and with or without guidance.

Sizes: dim 3072 / ffn 14336 / 24 heads, chunks of 3 latent frames of 22 x 40 tokens (2640), released chunks of 8 frames
(7040), 512 text tokens, and the dim 256 / ffn 512 / 2 heads model of the test suite span the range; a frame grid may have
any size, odd row counts included, and models between the two widths are as good as those.
"""
from __future__ import annotations

import math

import torch

from longlive_amd.dit import DiTBlock, DiTConfig, StreamingGenerator
from longlive_amd.fouroversix import ModelQuantizationConfig, QuantizationConfig, quantize_to_fp4
from longlive_amd.utils import kv_cache as kvc
from longlive_amd.utils.quant import quantize_model_with_filter
from longlive_amd.utils.rope import build_rope_angles, rope_cos_sin

DEVICE = "cuda"
HEAD_DIM = 128


def listed():
    return [
        # the projection of a test-sized model: the cost of the call itself
        dict(name="linear_tiny", kind="linear", m=48, k=256, n=512, rule="mse"),
        # a text key / value projection: 512 tokens, the smallest product of the full-width model
        dict(name="linear_text", kind="linear", m=512, k=3072, n=3072, rule="mse"),
        # FFN-down of a 3-frame chunk: the longest contraction
        dict(name="linear_ffn_down", kind="linear", m=2640, k=14336, n=3072, rule="mse"),
        # an activation of a mid-sized model: 3 frames of 23 x 17 tokens, the plain scale rule
        dict(name="quantize_odd", kind="quantize", m=1173, k=2048, rule="static_6"),
        # the FFN-down activation of a released 8-frame chunk: the largest activation that is quantized
        dict(name="quantize_large", kind="quantize", m=7040, k=14336, rule="mse"),
        # an FFN weight back to bf16, as the export of a merged checkpoint does
        dict(name="dequantize_weight", kind="dequantize", m=14336, k=3072, rule="mse", dtype="bfloat16"),
        # a one-frame chunk at a small resolution, relative RoPE over the window
        dict(name="kv_step_small_relative", kind="kv_step", frames=1, h=23, w=16, heads=16, cached=3, relative=True),
        # the benchmark chunk: sink block and three window blocks cached, 13200 keys
        dict(name="kv_step_chunk", kind="kv_step", frames=3, h=22, w=40, heads=24, cached=4, relative=False),
        # a block of a mid-sized model on a 2-frame chunk of a small grid, the prompt met for the first time
        dict(name="block_odd", kind="block", frames=2, h=23, w=16, heads=12, ffn=8960, cached=2, text_kept=False),
        # a block at the released shape: 8-frame chunks, sink block and two window blocks cached, 28160 keys
        dict(name="block_released", kind="block", frames=8, h=22, w=40, heads=24, ffn=14336, cached=3, text_kept=True),
        # the test suite's model end to end with the pipeline's own sampler: host work and launches
        dict(name="generate_small", kind="generate", layers=2, heads=2, ffn=512, text=16, frames=3, h=4, w=16, window=5, chunks=6,
             sampler="unipc", guidance=1.0),
        # the full width end to end, six chunks, so that the cache fills and rolls once (6 of the 30 equal layers)
        dict(name="generate_wide", kind="generate", layers=6, heads=24, ffn=14336, text=512, frames=3, h=22, w=40, window=5, chunks=6,
             sampler="euler", guidance=1.0),
    ]


# ------------------------------------------------------------------------------------------------- drawn cases
def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _width(rng):
    """(heads, ffn) of a model between the test suite's and the full one: ffn 2 to 4.7 times the width."""
    heads = rng.choice([2, 4, 6, 8, 12, 16, 20, 24])
    return heads, int(heads * HEAD_DIM * rng.uniform(2.0, 4.67)) // 128 * 128


def _grid(rng, lo, hi, frames, heads):
    """Rows and columns of a frame's token grid of about lo..hi tokens.  A cache slot holds whole groups of 128 rows
    (token, head), which the columns are made to fit; the rows may be odd."""
    tokens = _log(rng, lo, hi)
    h = max(3, int(math.sqrt(tokens * rng.uniform(0.4, 1.0))))
    unit = 128 // math.gcd(128, frames * h * heads)
    return h, max(1, int(tokens / h / unit + 0.5)) * unit


def draw(rng):
    kind = rng.choice(["linear", "linear", "quantize", "dequantize", "kv_step", "kv_step", "block", "block", "generate"])
    rule = rng.choice(["mse", "mse", "mse", "static_6", "mae", "static_4", "abs_max"])
    if kind in ("linear", "quantize", "dequantize"):
        heads, ffn = _width(rng)
        k, n = rng.choice([(heads * HEAD_DIM, heads * HEAD_DIM), (heads * HEAD_DIM, ffn), (ffn, heads * HEAD_DIM)])
        case = dict(kind=kind, m=_log(rng, 16, 7040), k=k, rule=rule)
        if kind == "linear":
            case["n"] = n
        if kind == "dequantize":
            case["dtype"] = rng.choice(["bfloat16", "float16", "float32"])
        return case
    if kind == "kv_step":
        heads, frames = _width(rng)[0], rng.randint(1, 4)
        h, w = _grid(rng, 40, 880, frames, heads)
        return dict(kind=kind, frames=frames, h=h, w=w, heads=heads, cached=rng.randint(0, 4), relative=rng.random() < 0.3)
    if kind == "block":
        (heads, ffn), frames = _width(rng), rng.randint(1, 4)
        h, w = _grid(rng, 40, 880, frames, heads)
        return dict(kind=kind, frames=frames, h=h, w=w, heads=heads, ffn=ffn, cached=rng.randint(0, 4), text_kept=rng.random() < 0.7)
    (heads, ffn), frames = _width(rng), rng.randint(1, 3)
    h, w = _grid(rng, 20, 880, frames, heads)
    return dict(kind=kind, layers=rng.randint(1, 3), heads=heads, ffn=ffn, text=rng.choice([64, 226, 512]), frames=frames, h=h, w=w,
                window=rng.randint(2, 5), chunks=rng.randint(2, 4), sampler=rng.choice(["euler", "unipc"]),
                guidance=rng.choice([1.0, 1.0, 2.0]))


# ------------------------------------------------------------------------------------------------- inputs
def _normal(shape, g, scale=1.0):
    return (torch.randn(shape, generator=g, device=DEVICE) * scale).bfloat16()


def _activations(shape, g):
    """N(0, 1) with one entry in a thousand twenty times as large: the outliers of transformer activations."""
    x = torch.randn(shape, generator=g, device=DEVICE)
    return torch.where(torch.rand(shape, generator=g, device=DEVICE) < 1e-3, x * 20, x).bfloat16()


def _quantized(module, rule="mse"):
    module, _ = quantize_model_with_filter(module, ModelQuantizationConfig(scale_rule=rule), use_default_filtered_modules=True,
                                           materialize_for_inference=True, verbose=False)
    return module


def _filled_cache(tokens, heads, cached, g):
    """A cache of cached + 1 slots of which the first ``cached`` hold chunks written by earlier steps and the last one the
    chunk at hand as its previous denoising forward left it: every further forward of the chunk rewrites that slot."""
    cfg = QuantizationConfig(scale_rule="mse")
    cache = kvc.initialize_kv_cache(1, tokens, cached + 1, heads, HEAD_DIM, cfg, DEVICE)[0]
    for chunk in range(cached + 1):
        k, v = (_normal((1, tokens, heads, HEAD_DIM), g) for _ in range(2))
        end, local_end, info = kvc.kv_cache_update_only(k, v, cache, chunk * tokens, tokens)
        kvc.apply_cache_update(cache, end, local_end, info, cfg)
    return cache, cfg


def prepare(case, seed):
    g = torch.Generator(device=DEVICE).manual_seed(seed)
    torch.manual_seed(seed)
    kind = case["kind"]
    state = dict(case=case)
    if kind == "linear":
        with torch.device(DEVICE):
            linear = torch.nn.Linear(case["k"], case["n"])
        with torch.no_grad():
            linear.weight.copy_(torch.randn(linear.weight.shape, generator=g, device=DEVICE) * 0.02)
            linear.bias.copy_(torch.randn(linear.bias.shape, generator=g, device=DEVICE) * 0.1)
        state.update(layer=_quantized(torch.nn.Sequential(linear), case["rule"])[0], x=_activations((case["m"], case["k"]), g))
    elif kind == "quantize":
        state.update(x=_activations((case["m"], case["k"]), g), config=QuantizationConfig(scale_rule=case["rule"]))
    elif kind == "dequantize":
        w = _normal((case["m"], case["k"]), g, 0.02)
        state.update(q=quantize_to_fp4(w, QuantizationConfig(scale_rule=case["rule"])), dtype=getattr(torch, case["dtype"]))
    elif kind == "kv_step":
        tokens, heads = case["frames"] * case["h"] * case["w"], case["heads"]
        cache, cfg = _filled_cache(tokens, heads, case["cached"], g)
        q, k, v = (_normal((1, tokens, heads, HEAD_DIM), g) for _ in range(3))
        state.update(cache=cache, config=cfg, q=q, k=k, v=v, tokens=tokens)
        if case["relative"]:
            angles, tables = build_rope_angles(HEAD_DIM), {}

            def rope_fn(frames, first):   # the position tables a program keeps per (frames, first frame)
                if (frames, first) not in tables:
                    tables[frames, first] = rope_cos_sin(angles, frames, case["h"], case["w"], first, torch.device(DEVICE))
                return tables[frames, first]

            for at in ((1, 0), (case["frames"] * (case["cached"] + 1), 0), (case["frames"], case["frames"] * case["cached"])):
                rope_fn(*at)
            state["rope_fn"] = rope_fn
    elif kind == "block":
        tokens, heads, dim = case["frames"] * case["h"] * case["w"], case["heads"], case["heads"] * HEAD_DIM
        cache, _ = _filled_cache(tokens, heads, case["cached"], g)
        with torch.device(DEVICE):
            block = DiTBlock(dim, case["ffn"], heads)
        block = _quantized(block)
        cos, sin = rope_cos_sin(build_rope_angles(HEAD_DIM), case["frames"], case["h"], case["w"], case["frames"] * case["cached"],
                                torch.device(DEVICE))
        # the conditioning of a trained model opens its gates a few tenths
        state.update(block=block, cache=cache, cos=cos, sin=sin, tokens=tokens, x=_normal((1, tokens, dim), g),
                     e=_normal((1, case["frames"], 6, dim), g, 0.3), context=_normal((1, 512, dim), g), text_kv=None)
        if case["text_kept"]:   # the prompt's projected keys and values, kept by the program between forwards
            state["text_kv"] = dict(is_init=False)
            run(state)
    else:
        dim = case["heads"] * HEAD_DIM
        cfg = DiTConfig(dim=dim, ffn_dim=case["ffn"], num_heads=case["heads"], num_layers=case["layers"], text_len=case["text"],
                        num_frame_per_block=case["frames"], local_attn_size=case["frames"] * case["window"], sink_size=case["frames"])
        gen = StreamingGenerator(cfg, DEVICE, seed=seed, sampler=case["sampler"], guidance_scale=case["guidance"])
        # A trained model's flow contracts towards the data; the flow of random weights does not.  The random head is scaled
        # down so that the loop answers to a rounding somewhere in the model as mildly as a trained model's does.
        gen.model.head.head.weight.data.mul_(0.1)
        noise = _normal((1, case["frames"] * case["chunks"], cfg.in_dim, 2 * case["h"], 2 * case["w"]), g)
        prompt, negative = (_normal((case["text"], cfg.text_dim), g) for _ in range(2))
        state.update(generator=gen, noise=noise, prompt=prompt, negative=negative if case["guidance"] != 1.0 else None)
    return state


# ------------------------------------------------------------------------------------------------- one pass
@torch.no_grad()
def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "linear":
        return state["layer"](state["x"])
    if kind == "quantize":
        q = quantize_to_fp4(state["x"], state["config"])
        return [q.values, q.scale_factors.view(torch.uint8), q.amax]
    if kind == "dequantize":
        return state["q"].dequantize(state["dtype"])
    if kind == "kv_step":
        cache, tokens = state["cache"], state["tokens"]
        start = case["cached"] * tokens
        if case["relative"]:
            out, update = kvc.kv_cache_attention_relative(state["q"], state["k"], state["v"], cache, start, tokens, state["rope_fn"])
        else:
            out, update = kvc.kv_cache_attention(state["q"], state["k"], state["v"], cache, start, tokens)
        kvc.apply_cache_update(cache, *update, state["config"])
        written = [cache[name][case["cached"]] for name in ("k", "v")]
        return [out] + [t for s in written for t in (s.values, s.scale_factors.view(torch.uint8), s.amax)]
    if kind == "block":
        out, _ = state["block"](state["x"], state["e"], state["cos"], state["sin"], state["context"], state["cache"],
                                case["cached"] * state["tokens"], state["tokens"], crossattn_cache=state["text_kv"],
                                collect_kv_amax=False)
        return out
    gen = state["generator"]
    gen.kv_cache = None   # a video of its own
    return gen.generate(state["noise"], state["prompt"], negative_context=state["negative"])


# ------------------------------------------------------------------------------------------------- what a pass cannot do without
def _fp4(rows, cols):
    return rows * cols * (0.5 + 1.0 / 16)


def _kv_work(tokens, heads, cached):
    row = heads * HEAD_DIM
    return (2 * _fp4(cached * tokens, row) + 4 * 2.0 * tokens * row,             # cached K and V, the chunk's q / k / v / out
            4.0 * tokens * (cached + 1) * tokens * row)


def _block_work(tokens, heads, ffn, cached, text, text_kept):
    dim = heads * HEAD_DIM
    kv_bytes, kv_flops = _kv_work(tokens, heads, cached)
    n_text = 0 if text_kept else 2
    weights = _fp4(dim, (6 + n_text) * dim + 2 * ffn)
    flops = 2.0 * tokens * dim * (6 * dim + 2 * ffn) + n_text * 2.0 * text * dim * dim + kv_flops + 4.0 * tokens * text * dim
    # x in and out, the cached window; the prompt's K and V, or its context where they are projected anew
    return weights + 2 * 2.0 * tokens * dim + 2 * _fp4(cached * tokens, dim) + 2.0 * text * dim * (2 if text_kept else 1), flops


def work(case):
    kind = case["kind"]
    if kind == "linear":
        m, k, n = case["m"], case["k"], case["n"]
        return dict(bytes=2.0 * m * k + _fp4(n, k) + 2.0 * m * n + 2.0 * n, flops=2.0 * m * n * k)
    if kind == "quantize":
        return dict(bytes=2.0 * case["m"] * case["k"] + _fp4(case["m"], case["k"]), flops=0.0)
    if kind == "dequantize":
        size = 4 if case["dtype"] == "float32" else 2
        return dict(bytes=_fp4(case["m"], case["k"]) + size * case["m"] * case["k"], flops=0.0)
    tokens = case["frames"] * case["h"] * case["w"]
    if kind == "kv_step":
        nbytes, flops = _kv_work(tokens, case["heads"], case["cached"])
        return dict(bytes=nbytes + 2 * _fp4(tokens, case["heads"] * HEAD_DIM), flops=flops)
    if kind == "block":
        nbytes, flops = _block_work(tokens, case["heads"], case["ffn"], case["cached"], 512, case["text_kept"])
        return dict(bytes=nbytes, flops=flops)
    total_bytes = total_flops = 0.0
    passes = 5 * (2 if case["guidance"] != 1.0 else 1)   # four denoising forwards and the clean-context pass per chunk
    for chunk in range(case["chunks"]):
        nbytes, flops = _block_work(tokens, case["heads"], case["ffn"], min(chunk, case["window"] - 1), case["text"], True)
        total_bytes += passes * case["layers"] * nbytes
        total_flops += passes * case["layers"] * flops
    return dict(bytes=total_bytes, flops=total_flops)


# ------------------------------------------------------------------------------------------------- tolerance
def tolerance(case):
    """Measured: every kind against itself with the sums of the GEMM and of the attention in another order (the schedules and
    work divisions the package lets a caller choose), over the listed and some 40 drawn cases."""
    kind = case["kind"]
    if kind in ("quantize", "dequantize"):
        return "exact"
    if kind == "linear":
        # fp32 sums of exact products, rounded once to bf16: another order moves at most 0.5 % of the results by one bf16 step
        return {"rel": 5e-4, "max": 1e-2}
    if kind == "kv_step":
        # bf16 probabilities against another reference point of the softmax: 0.003 seen; the bytes of the slot are exact
        return {"rel": 1.2e-2, "max": 0.07, "differ": 0.0}
    if kind == "block":
        # four activations are quantized again inside, which turns a difference d into about 0.65 sqrt(d): 0.007 seen
        return {"rel": 2.7e-2, "max": 0.35}
    # the same through every layer, step and chunk: 0.012 seen, most of it where guidance doubles a difference
    return {"rel": 3e-2, "max": 0.3}
