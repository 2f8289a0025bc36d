"""What a user of this package has it do, as cases that can be timed: decode steps over a stack of layers, prompt
passes, the reference's operators called by themselves, and a decoder around all of it.

The geometries are those of the benchmark workloads (``bench.py``) and of the two decoders the harness knows
(``llama.PRESETS``): 32 or 24 query heads on 8 KV heads of 128 dims, 4 sink tokens, a window of 512 to 1024 rows, 256
to 2048 coefficient rows, one to sixteen sequences of 2k to 128k tokens.  Queries, keys and values are N(0, 1) with
rotary embedding, weights are normal with a deviation of 0.02 (``llama.random_init``).

Kinds of case (``kind``):

* ``decode``: one decode step of ``layers`` layers, each ``fourier_attention`` on one new token per sequence (cache
  update, then attention over sink, window, coefficients and stored dims).  The cache grows by one token per pass, as it
  does in use.
* ``prompt``: a new cache, the prompt through ``layers`` layers (cache prefill and exact causal attention), then the
  first decode step behind it.
* ``operators``: spectral compression and both statistics of one tensor of a prompt, called as the reference names them.
* ``token_major``: the reference's decode operator on tensors in the reference's own layout.
* ``model``: one decode step of a decoder (projections, rotary embedding, attention, MLP, LM head) behind a long prompt.
* ``dialogue``: a decoder takes a short prompt into a new cache and then ``steps`` given tokens one by one.
"""
from __future__ import annotations

import math
import random

import torch

from fourierattention_amd import DynamicCache, ExtraConfig, masks, ops
from fourierattention_amd.attention import fourier_attention
from fourierattention_amd.llama import PRESETS, LlamaConfig, random_init, synthetic_prefill

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
MAX_POSITIONS = 131072     # both decoders' max_position_embeddings
MAX_NEW = 4096             # room for a long answer
SINK = 4

# Compressed dims per KV head, K and V, of three layers of the reference's own 8B mask at 1024 states (bench.py)
EVAL_COUNTS = (
    ([121, 124, 103, 127, 128, 117, 83, 118], [115, 122, 119, 126, 122, 125, 122, 121]),
    ([83, 116, 117, 96, 122, 88, 116, 81], [120, 128, 110, 111, 8, 122, 128, 92]),
    ([47, 86, 44, 60, 75, 64, 69, 67], [82, 127, 124, 61, 114, 1, 81, 126]),
)


def listed():
    decode = dict(kind="decode", Hq=32, Hkv=8, D=128, W=1024, M=1024, mask="half", dtype="bf16")
    return [
        # the reference's evaluation settings: one sequence, a window of 1020, its own mask (ragged from head to head)
        dict(decode, name="decode_1x32k_eval", B=1, ctx=32768, W=1020, mask="eval", layers=8),
        # the smallest benchmark configuration, in single precision as it is defined there
        dict(decode, name="decode_1x2k_fp32", B=1, ctx=2048, Hq=24, W=512, M=256, dtype="fp32", layers=8),
        # the headline benchmark configuration: a batch of eight at 32k
        dict(decode, name="decode_8x32k", B=8, ctx=32768, layers=4),
        # the largest caches: sixteen sequences of 64k, and four of 128k with 2048 states (two passes over the pages)
        dict(decode, name="decode_16x64k", B=16, ctx=65536, layers=2),
        dict(decode, name="decode_4x128k_m2048", B=4, ctx=131072, Hq=24, M=2048, layers=2),
        # an ordinary serving batch of odd size: ragged mask, half precision, 512 states
        dict(decode, name="decode_3x12k_fp16", B=3, ctx=12345, Hq=24, W=1020, M=512, mask="eval", dtype="fp16", layers=8),
        # prompts: one long one (the quadratic part leads), and a few short ones of odd length (compression leads)
        dict(decode, name="prompt_1x32k", kind="prompt", B=1, ctx=32768, layers=1),
        dict(decode, name="prompt_4x3k_fp16", kind="prompt", B=4, ctx=3001, Hq=24, W=1020, mask="eval", dtype="fp16", layers=2),
        # spectral compression and statistics of one 32k tensor by the reference's operator names
        dict(name="operators_1x32k", kind="operators", B=1, rows=32768, C=512, M=1024, dtype="bf16"),
        # the decode operator alone, on tensors as the reference's own cache holds them
        dict(decode, name="token_major_2x16k", kind="token_major", B=2, ctx=16384),
        # a decoder at work: a decode step behind a long prompt, and a short prompt with the tokens that follow it
        # (everything still fits the window there, so no layer is compressed)
        dict(name="model_1x32k", kind="model", preset="llama-3.1-8b", layers=8, B=1, ctx=32768, W=1020, M=1024, mask="half",
             dtype="bf16"),
        dict(name="dialogue_2x700", kind="dialogue", preset="llama-3.2-3b", layers=8, B=2, ctx=700, steps=16, W=1024,
             M=1024, mask="half", dtype="bf16"),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _heads(rng):
    return rng.choice([(32, 8, 128), (24, 8, 128), (32, 8, 128), (24, 8, 128), (16, 8, 128), (64, 8, 128), (32, 8, 64)])


def _mask(rng):
    return rng.choice(["half", "eval", "ragged-%d" % rng.randrange(1000), "uniform-%d" % rng.randrange(16, 113)])


def draw(rng):
    """One more case of the same ranges.  Batch times context stays below the largest listed cache, prompts below the
    longest one, so that no drawn case costs more than the largest listed one."""
    kind = rng.choice(["decode"] * 9 + ["prompt"] * 4 + ["operators"] * 2 + ["token_major"] * 2 + ["model", "model", "dialogue"])
    states = rng.choice([256, 512, 1024, 1024, 2048])
    window = rng.choice([512, 1020, 1024])
    dtype = rng.choice(["bf16", "bf16", "fp16"])
    if kind == "decode":
        if rng.random() < 0.12:     # single precision: small models at short contexts
            Hq, Hkv, D = 24, 8, 128
            return dict(kind=kind, Hq=Hq, Hkv=Hkv, D=D, W=512, M=rng.choice([256, 512]), mask=_mask(rng), dtype="fp32",
                        B=rng.choice([1, 2]), ctx=_log_int(rng, 1400, 4096), layers=rng.randrange(4, 9))
        Hq, Hkv, D = _heads(rng)
        B = _log_int(rng, 1, 16)
        ctx = _log_int(rng, SINK + window + states + 64, min(MAX_POSITIONS, 786432 // B))
        layers = max(1, min(8, 2000000 // (B * ctx)))
        return dict(kind=kind, Hq=Hq, Hkv=Hkv, D=D, W=window, M=states, mask=_mask(rng), dtype=dtype, B=B, ctx=ctx, layers=layers)
    if kind == "prompt":
        Hq, Hkv, D = _heads(rng)
        Hq = min(Hq, 32)
        B = _log_int(rng, 1, 8)
        ctx = _log_int(rng, SINK + window + states + 64, min(24576, max(49152 // B, 3500)))
        return dict(kind=kind, Hq=Hq, Hkv=Hkv, D=D, W=window, M=states, mask=_mask(rng), dtype=dtype, B=B, ctx=ctx,
                    layers=1 if B * ctx > 12288 else 2)
    if kind == "operators":
        return dict(kind=kind, B=rng.choice([1, 1, 2]), rows=_log_int(rng, 1024, 65536), C=rng.randrange(64, 901), M=states, dtype=dtype)
    if kind == "token_major":
        Hq, Hkv, D = rng.choice([(32, 8, 128), (24, 8, 128)])
        B = rng.choice([1, 2, 4])
        return dict(kind=kind, Hq=Hq, Hkv=Hkv, D=D, W=window, M=states, mask=_mask(rng), dtype=dtype, B=B,
                    ctx=_log_int(rng, 4200, 98304 // B))
    preset = rng.choice(sorted(PRESETS))
    if kind == "model":
        B = _log_int(rng, 1, 16)
        return dict(kind=kind, preset=preset, layers=rng.randrange(4, 9), B=B, ctx=_log_int(rng, SINK + window + states + 64, 131072 // B + 2000),
                    W=window, M=states, mask=_mask(rng), dtype="bf16")
    return dict(kind=kind, preset=preset, layers=rng.randrange(4, 9), B=rng.choice([1, 2, 3, 4]), ctx=_log_int(rng, 64, 1400),
                steps=rng.randrange(8, 17), W=1024, M=1024, mask=_mask(rng), dtype="bf16")


# ---------------------------------------------------------------------------------------------- inputs
def _counts(mask, Hkv, D):
    """Compressed dims per KV head of one layer of the mask, ``[(K counts, V counts)]`` of the layers it cycles through."""
    scale = lambda lists: [(v * D + 64) // 128 for v in lists]
    if mask == "half":
        return [([D // 2] * Hkv, [D // 2] * Hkv)]
    if mask == "eval":
        return [(scale((k * 8)[:Hkv]), scale((v * 8)[:Hkv])) for k, v in EVAL_COUNTS]
    kind, number = mask.split("-")
    if kind == "uniform":
        return [([int(number) * D // 128] * Hkv, [int(number) * D // 128] * Hkv)]
    r = random.Random(int(number))
    return [([r.randrange(D // 4, D + 1) for _ in range(Hkv)], [r.randrange(D // 4, D + 1) for _ in range(Hkv)]) for _ in range(3)]


def _masks(mask, layers, Hkv, D):
    kinds = _counts(mask, Hkv, D)
    out = {}
    for i in range(layers):
        k, v = kinds[i % len(kinds)]
        out["Layer_%d" % i] = masks.synthetic_masks(1, Hkv, D, k, v, seed=i)["Layer_0"]
    return out


def _config(case, Hkv, D):
    return ExtraConfig(numinittokens=SINK, maxlocallen=case["W"], maxmidstates=case["M"],
                       non_critical_dims=_masks(case["mask"], case.get("layers", 1), Hkv, D), non_critical_dims_path=None,
                       max_position_embeddings=MAX_POSITIONS, num_key_value_heads=Hkv, max_new_tokens=MAX_NEW, model_type="llama")


def _rotated(x, first):
    """Rotary embedding (base 500000) of ``x (B, H, S, D)`` whose rows sit at positions ``first ..``, sequence by sequence."""
    S, D = x.shape[2], x.shape[3]
    inv = 500000.0 ** (-torch.arange(0, D, 2, dtype=torch.float64, device=x.device) / D)
    ang = torch.arange(first, first + S, dtype=torch.float64, device=x.device)[:, None] * inv[None, :]
    cos, sin = ang.cos().float(), ang.sin().float()
    out = torch.empty_like(x)
    for b in range(x.shape[0]):
        lo, hi = x[b, :, :, : D // 2].float(), x[b, :, :, D // 2:].float()
        out[b, :, :, : D // 2] = lo * cos - hi * sin
        out[b, :, :, D // 2:] = hi * cos + lo * sin
    return out


def _normal(shape, dtype, g):
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32).to(dtype)


def _prompt(case, g):
    shape = (case["B"], case["Hkv"], case["ctx"], case["D"])
    dt = DTYPES[case["dtype"]]
    return _rotated(_normal(shape, dt, g), 0), _normal(shape, dt, g)


def _token(case, g):
    B, D, dt, at = case["B"], case["D"], DTYPES[case["dtype"]], case["ctx"]
    return (_rotated(_normal((B, case["Hq"], 1, D), dt, g), at), _rotated(_normal((B, case["Hkv"], 1, D), dt, g), at),
            _normal((B, case["Hkv"], 1, D), dt, g))


def _llama(case):
    return LlamaConfig(**dict(PRESETS[case["preset"]], num_hidden_layers=case["layers"]))


@torch.no_grad()
def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    kind = case["kind"]
    state = {"case": case}
    if kind in ("decode", "prompt", "token_major"):
        layers = case.get("layers", 1)
        config = _config(case, case["Hkv"], case["D"])
        if kind == "prompt":
            state["config"] = config
            state["prompt"] = []
            for _ in range(layers):
                q = _rotated(_normal((case["B"], case["Hq"], case["ctx"], case["D"]), DTYPES[case["dtype"]], g), 0)
                state["prompt"].append((q,) + _prompt(case, g))
        else:
            cache = DynamicCache(config)
            for layer in range(layers):
                cache.update(*_prompt(case, g), layer)
            state["cache"] = cache
        state["token"] = [_token(case, g) for _ in range(layers)]
        if kind == "token_major":     # the parts as the reference keeps them, and its argument list
            c = state.pop("cache")
            k, v = c.key_cache[0], c.value_cache[0]
            q = state.pop("token")[0][0]
            local = [torch.cat([p[t + "_init"], p[t + "_local"]], dim=1).contiguous() for p, t in ((k, "k"), (v, "v"))]
            state["args"] = dict(
                q=q.transpose(1, 2).reshape(case["B"], 1, -1).contiguous(), k_il=local[0], v_il=local[1],
                k_mc=k["k_compressed"], v_mc=v["v_compressed"], k_mn=k["k_uncompressed"], v_mn=v["v_uncompressed"],
                avg_k_u=c.k_layer_average[0], avg_k_d=c.kd_layer_average[0], scale_k=c.k_scale[0],
                avg_v_u=c.v_layer_average[0], avg_v_d=c.vd_layer_average[0], scale_v=c.v_scale[0],
                kc_list=c.k_non_critical_dims[0], kc_h_list=c.k_non_critical_head_dims[0],
                kn_list=c.k_critical_dims[0], kn_h_list=c.k_critical_head_dims[0],
                vc_list=c.v_non_critical_dims[0], vc_h_list=c.v_non_critical_head_dims[0],
                vn_list=c.v_critical_dims[0], vn_h_list=c.v_critical_head_dims[0],
                num_head_q=case["Hq"], num_head_kv=case["Hkv"], seq_len_m=case["ctx"] - SINK - case["W"],
                T=c.maxtokens - c.numinittokens - c.maxlocallen)
    elif kind == "operators":
        # keys after rotary embedding: every column an oscillation of its own under noise
        B, rows, C = case["B"], case["rows"], case["C"]
        x = _normal((B, 1, rows, 2 * ((C + 1) // 2)), torch.float32, g)
        state["x"] = _rotated(x, 0)[:, 0, :, :C].to(DTYPES[case["dtype"]]).contiguous()
    else:
        llama = _llama(case)
        model = random_init(llama, DTYPES[case["dtype"]], "cuda:0", seed=seed)
        model.model.fuse_projections()
        model.model.pack_projections()
        state["model"] = model
        config = _config(case, llama.num_key_value_heads, llama.head_dim)
        ids = lambda n: torch.randint(0, llama.vocab_size, (case["B"], n), generator=g, device="cuda")
        if kind == "model":
            state["cache"] = DynamicCache(config)
            synthetic_prefill(state["cache"], llama, case["B"], case["ctx"], DTYPES[case["dtype"]], "cuda:0", seed=seed)
            state["ids"] = ids(1)
        else:
            state["config"], state["ids"], state["answer"] = config, ids(case["ctx"]), ids(case["steps"])
    return state


# ---------------------------------------------------------------------------------------------- one pass
def _coefficients(cache):
    return [p["%s_compressed" % t] for parts, t in ((cache.key_cache, "k"), (cache.value_cache, "v")) for p in parts]


@torch.no_grad()
def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "decode":
        cache = state["cache"]
        out = [fourier_attention(q, k, v, cache, i, case["Hq"], case["Hkv"]) for i, (q, k, v) in enumerate(state["token"])]
        return {"attention": out, "coefficients": _coefficients(cache)}
    if kind == "prompt":
        cache = DynamicCache(state["config"])
        out = [fourier_attention(q, k, v, cache, i, case["Hq"], case["Hkv"]) for i, (q, k, v) in enumerate(state["prompt"])]
        out += [fourier_attention(q, k, v, cache, i, case["Hq"], case["Hkv"]) for i, (q, k, v) in enumerate(state["token"])]
        return {"attention": out, "coefficients": _coefficients(cache)}
    if kind == "operators":
        x, n_f = state["x"], case["M"] // 2
        c = ops.mat_fourier_triton(x, n_f, case["rows"])
        return {"coefficients": c, "rows": ops.mat_avg_std_triton(x), "reconstruction": ops.mat_fourier_avg_std_triton(c, case["rows"], case["rows"])}
    if kind == "token_major":
        return ops.triton_fourier_attn(**state["args"])
    model = state["model"]
    if kind == "model":
        logits = model(input_ids=state["ids"], past_key_values=state["cache"], num_logits_to_keep=1).logits
        return {"logits": logits, "coefficients": _coefficients(state["cache"])}
    cache = DynamicCache(state["config"])
    logits = [model(input_ids=state["ids"], past_key_values=cache, num_logits_to_keep=1).logits]
    for t in range(case["steps"]):
        logits.append(model(input_ids=state["answer"][:, t:t + 1], past_key_values=cache, num_logits_to_keep=1).logits)
    windows = [p["%s_local" % t] for parts, t in ((cache.key_cache, "k"), (cache.value_cache, "v")) for p in parts]
    return {"logits": logits, "windows": windows}


# ---------------------------------------------------------------------------------------------- what a pass needs
def _attention_step(case, Hq, Hkv, D, layer, size):
    """Bytes and operations of one decode step of one compressed layer, per sequence: sink and window rows, stored dims
    of the mid rows, coefficients (read, and written by the update), the new token, query and output."""
    kinds = _counts(case["mask"], Hkv, D)
    k, v = kinds[layer % len(kinds)]
    comp, full = sum(k) + sum(v), 2 * Hkv * D
    near, mid = SINK + case["W"], case["ctx"] - SINK - case["W"]
    nbytes = near * full * size + mid * (full - comp) * size + 2 * case["M"] * comp * 4 + (full + 2 * Hq * D) * size
    flops = near * 4 * Hq * D + mid * (2 * (full - comp) * (Hq // Hkv) + 4 * case["M"] * Hq) + 4 * case["M"] * comp * (Hq // Hkv)
    return nbytes, flops


def work(case):
    kind, B = case["kind"], case["B"]
    size = 4 if case["dtype"] == "fp32" else 2
    if kind == "operators":
        # the contraction with the basis, and the reconstruction its statistics are taken from
        n = B * case["rows"] * case["C"]
        return {"bytes": n * size + B * case["M"] * case["C"] * 4, "flops": 4.0 * case["M"] * n}
    if kind in ("decode", "token_major"):
        steps = [_attention_step(case, case["Hq"], case["Hkv"], case["D"], i, size) for i in range(case.get("layers", 1))]
        return {"bytes": B * sum(s[0] for s in steps), "flops": B * sum(s[1] for s in steps)}
    if kind == "prompt":
        nbytes = flops = 0
        S, Hq, Hkv, D = case["ctx"], case["Hq"], case["Hkv"], case["D"]
        for i in range(case["layers"]):
            step = _attention_step(case, Hq, Hkv, D, i, size)
            kinds = _counts(case["mask"], Hkv, D)
            comp = sum(kinds[i % len(kinds)][0]) + sum(kinds[i % len(kinds)][1])
            nbytes += S * (2 * Hq + 2 * Hkv) * D * size + 2 * step[0]
            flops += 2 * Hq * D * S * S + 2 * case["M"] * (S - SINK - case["W"]) * comp + step[1]
        return {"bytes": B * nbytes, "flops": B * flops}
    llama = _llama(case)
    h, inter, D = llama.hidden_size, llama.intermediate_size, llama.head_dim
    Hq, Hkv = llama.num_attention_heads, llama.num_key_value_heads
    weights = llama.num_hidden_layers * (h * (2 * Hq + 2 * Hkv) * D + 3 * h * inter)
    head = h * llama.vocab_size
    if kind == "model":
        steps = [_attention_step(case, Hq, Hkv, D, i, size) for i in range(case["layers"])]
        return {"bytes": (weights + head) * size + B * (sum(s[0] for s in steps) + 4 * llama.vocab_size),
                "flops": 2 * B * (weights + head) + B * sum(s[1] for s in steps)}
    rows, steps = case["ctx"], case["steps"]
    kv = case["layers"] * 2 * Hkv * D * size
    return {"bytes": (weights + head) * size * (1 + steps) + B * (kv * rows * (1 + steps) + 4 * llama.vocab_size * (1 + steps)),
            "flops": 2 * B * (weights * (rows + steps) + head * (1 + steps)) + B * case["layers"] * 2 * Hq * D * rows * (rows + 2 * steps)}


def tolerance(case):
    """About four times what was measured: decode attention against the any-shape kernels (single precision throughout)
    and against float64 over the rebuilt rows, prompts against float32 attention, the operators against float64, the
    decoders against the chain of tensor ops with the library's projections."""
    kind, dtype = case["kind"], case["dtype"]
    if kind in ("model", "dialogue"):
        return {"rel": 7e-2}        # 1.85e-2 on the logits behind eight layers of bf16 rounding
    if dtype == "fp32":
        return {"rel": 1e-5}        # 8e-7 on the attention, 3.3e-6 on coefficients summed in single precision
    if kind == "token_major":
        return {"rel": 2.5e-3}      # 6.1e-4: 16-bit operands, the result in single precision
    return {"rel": 7e-3 if dtype == "bf16" else 1.2e-3}     # 1.75e-3 / 3.1e-4: the rounding of the result itself
