"""The work that a user of the W4A16 library has it do, as cases that can be
timed and checked one by one: linear layers through ``QuantizedLinear`` (one
token, small batches, prompts; group sizes 128 and below), the ``dequantize``
op, the quantizer, one layer's attention over a long cache, and the decoder's
decode step and prefill.

Sizes are those of this repository's benchmark and tests: the 1.1B Llama
(hidden 2048, intermediate 5632, 32/4 heads of 64, vocabulary 32000, 22
layers), the 8B class (4096 / 14336) and the 70B class (8192 / 28672).

``graph`` cases record their calls in a HIP graph in ``prepare`` and replay it
in ``run``, as the decoder and the reference's benchmark do; the ``copies``
layers of a case hold weights of their own, so that a pass reads them from
memory as a model's layers would be and not from a cache.
"""

from __future__ import annotations

import math

import torch
import torch.nn.functional as F

from nibble_amd import _lib
from nibble_amd.linear import QuantizedLinear
from nibble_amd.llama import LlamaConfig, LlamaDecoder
from nibble_amd.quantization import quantize_and_pack_weights

DEVICE = "cuda"
INIT_STD = 0.02


def listed() -> list[dict]:
    return [
        # the smallest call: one token, one attention projection of the 1.1B model, called eagerly
        {"name": "linear_m1_2048x2048_eager", "kind": "linear", "m": 1, "k": 2048, "n": 2048, "group": 128,
         "copies": 1, "graph": False},
        # single-stream decode of the 8B class: the gate / up projections of 16 layers
        {"name": "linear_m1_4096x14336", "kind": "linear", "m": 1, "k": 4096, "n": 14336, "group": 128,
         "copies": 16, "graph": True},
        # eight sequences decoded together: the down projections of 16 layers
        {"name": "linear_m8_14336x4096", "kind": "linear", "m": 8, "k": 14336, "n": 4096, "group": 128,
         "copies": 16, "graph": True},
        # decode on a checkpoint with finer groups
        {"name": "linear_m1_g64_4096x4096", "kind": "linear", "m": 1, "k": 4096, "n": 4096, "group": 64,
         "copies": 32, "graph": True},
        # a short prompt or a larger decode batch (a ragged row count) on the 1.1B model's gate / up
        {"name": "linear_m24_2048x5632", "kind": "linear", "m": 24, "k": 2048, "n": 5632, "group": 128,
         "copies": 32, "graph": True},
        # a prompt of 200 tokens through the 1.1B model's down projections
        {"name": "linear_m200_5632x2048", "kind": "linear", "m": 200, "k": 5632, "n": 2048, "group": 128,
         "copies": 32, "graph": True},
        # a long prompt through one 8B-class projection, called eagerly
        {"name": "linear_m2048_4096x14336", "kind": "linear", "m": 2048, "k": 4096, "n": 14336, "group": 128,
         "copies": 2, "graph": False},
        # fp16 weights of a 70B-class layer for a caller's own GEMM
        {"name": "dequantize_8192x28672", "kind": "dequantize", "k": 8192, "n": 28672, "group": 128},
        # a model being converted: one 8B-class layer from fp16 weights
        {"name": "quantize_14336x4096", "kind": "quantize", "k": 14336, "n": 4096, "group": 128, "dtype": "fp16"},
        # the attention of a decode step's 22 layers, 1500 tokens into a 2048-slot cache
        {"name": "decode_attention_1500", "kind": "decode_attention", "layers": 22, "heads": 32, "kv_heads": 4,
         "slots": 2048, "position": 1500},
        # one decoded token of the 1.1B model
        {"name": "decode_step_1.1b", "kind": "decode", "position": 40, "max_seq_len": 64},
        # a 700-token prompt of the 1.1B model
        {"name": "prefill_700_1.1b", "kind": "prefill", "tokens": 700, "max_seq_len": 1024},
    ]


def _log(rng, low: float, high: float) -> int:
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng) -> dict:
    kind = rng.choice(["linear"] * 9 + ["dequantize", "quantize", "quantize", "decode_attention", "decode_attention",
                                       "decode", "prefill"])
    if kind == "linear":
        group = rng.choice([128, 128, 128, 64, 32])
        m = rng.choice([1, _log(rng, 1, 16), _log(rng, 1, 2048)])
        k = 128 * _log(rng, 8, 112)
        n = _log(rng, 512, 16384)
        if rng.random() < 0.6:
            n = (n + 63) // 64 * 64
        graph = m <= 512
        copies = max(1, min(32, 300_000_000 // (n * k // 2), 40_000_000_000 // (2 * m * n * k))) if graph else 1
        return {"kind": kind, "m": m, "k": k, "n": n, "group": group, "copies": copies, "graph": graph}
    if kind == "dequantize":
        return {"kind": kind, "k": 128 * _log(rng, 8, 64), "n": _log(rng, 512, 28672),
                "group": rng.choice([128, 128, 64, 32])}
    if kind == "quantize":
        return {"kind": kind, "k": 128 * _log(rng, 8, 112), "n": _log(rng, 512, 8192),
                "group": rng.choice([128, 128, 64, 32]), "dtype": rng.choice(["fp16", "fp32"])}
    if kind == "decode_attention":
        slots = rng.choice([1024, 2048, 4096])
        heads, kv_heads = rng.choice([(32, 4), (32, 8), (16, 4), (64, 8)])
        return {"kind": kind, "layers": 22, "heads": heads, "kv_heads": kv_heads, "slots": slots,
                "position": _log(rng, 256, slots - 1)}
    if kind == "decode":
        max_seq_len = rng.choice([64, 64, 512, 1024, 2048])
        return {"kind": kind, "position": rng.randrange(1, max_seq_len), "max_seq_len": max_seq_len}
    return {"kind": "prefill", "tokens": _log(rng, 2, 700), "max_seq_len": 1024}


def _gen(seed: int) -> torch.Generator:
    return torch.Generator(device=DEVICE).manual_seed(seed)


def _weights(n: int, k: int, group: int, gen: torch.Generator) -> tuple[torch.Tensor, torch.Tensor]:
    """Packed codes and fp16 scales of N(0, 0.02) weights rounded to nearest
    by group, in plain torch (the file format: symmetric codes in [-7, 7],
    the even-k code in the low nibble, scale = amax / 7)."""
    w = torch.randn((n, k // group, group), device=DEVICE, generator=gen) * INIT_STD
    scale = w.abs().amax(dim=2, keepdim=True) / 7.0
    codes = torch.round(w / scale).clamp_(-7, 7).to(torch.int32).reshape(n, k // 2, 2)
    packed = ((codes[..., 0] & 15) | ((codes[..., 1] & 15) << 4)).to(torch.uint8)
    return packed, scale.reshape(n, k // group).to(torch.float16)


def _dense(packed: torch.Tensor, scales: torch.Tensor) -> torch.Tensor:
    """The weights that packed codes and scales stand for, in 64 bits."""
    n, half = packed.shape
    wide = packed.to(torch.int16)
    codes = torch.stack((((wide & 15) ^ 8) - 8, ((wide >> 4) ^ 8) - 8), dim=-1)
    return (codes.reshape(n, scales.shape[1], -1).double() * scales.double().unsqueeze(-1)).reshape(n, 2 * half)


def _rows(m: int, k: int, gen: torch.Generator) -> torch.Tensor:
    return torch.randn((m, k), device=DEVICE, generator=gen).to(torch.float16)


def _record(call) -> tuple[torch.cuda.CUDAGraph, object]:
    """A HIP graph of call() and the outputs that its replays write."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        call()   # a warm-up outside the capture
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = call()
    return graph, out


# ---------------------------------------------------------------- the decoder

def _decoder_weights(cfg: LlamaConfig, seed: int) -> dict[str, torch.Tensor]:
    """A random model's state dict, from the seed alone."""
    gen = _gen(seed)
    h, kv, inter = cfg.hidden_size, cfg.num_kv_heads * cfg.head_dim, cfg.intermediate_size
    state = {"embed": (torch.randn((cfg.vocab_size, h), device=DEVICE, generator=gen) * INIT_STD).to(torch.float16)}

    def linear(name, n, k):
        state[name + ".packed_weights"], state[name + ".scales"] = _weights(n, k, cfg.group_size, gen)

    def norm(name):
        state[name + ".weight"] = (1 + 0.1 * torch.randn((h,), device=DEVICE, generator=gen)).to(torch.float16)

    for i in range(cfg.num_layers):
        p = f"layers.{i}."
        norm(p + "input_norm")
        linear(p + "q_proj", h, h)
        linear(p + "k_proj", kv, h)
        linear(p + "v_proj", kv, h)
        linear(p + "o_proj", h, h)
        norm(p + "post_norm")
        linear(p + "gate_proj", inter, h)
        linear(p + "up_proj", inter, h)
        linear(p + "down_proj", h, inter)
    norm("norm")
    linear("lm_head", cfg.vocab_size, h)
    return state


def _decoder(cfg: LlamaConfig, seed: int) -> LlamaDecoder:
    decoder = LlamaDecoder(cfg, device=DEVICE, init="empty")
    decoder.load_state_dict(_decoder_weights(cfg, seed))
    return decoder


def _caches(layers: int, kv_heads: int, slots: int, used: int, gen: torch.Generator):
    """Key and value caches whose first `used` slots are filled."""
    out = []
    for _ in range(2):
        cache = torch.zeros((layers, kv_heads, slots, 64), dtype=torch.float16, device=DEVICE)
        cache[:, :, :used] = torch.randn((layers, kv_heads, used, 64), device=DEVICE, generator=gen).to(torch.float16)
        out.append(cache)
    return out


def _tables(slots: int) -> tuple[torch.Tensor, torch.Tensor]:
    inv = 1.0 / (10000.0 ** (torch.arange(0, 64, 2, device=DEVICE).float() / 64))
    angles = torch.outer(torch.arange(slots, device=DEVICE).float(), inv)
    return angles.cos(), angles.sin()


def _rotate(x: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor) -> torch.Tensor:
    """x [T, heads, 64], cos / sin [T, 32]: the half-split rotary embedding."""
    a, b = x[..., :32], x[..., 32:]
    c, s = cos.unsqueeze(1), sin.unsqueeze(1)
    return torch.cat((a * c - b * s, b * c + a * s), dim=-1)


def _attend(q, k, v, first: int) -> torch.Tensor:
    """q [T, heads, 64] at positions first .. first + T - 1 over k / v [kv_heads, S, 64], causal, in 64 bits."""
    t, heads, _ = q.shape
    group = heads // k.shape[0]
    s = first + t
    hidden = torch.arange(s, device=q.device).unsqueeze(0) > first + torch.arange(t, device=q.device).unsqueeze(1)
    out = torch.empty_like(q)
    for h in range(heads):
        scores = q[:, h] @ k[h // group, :s].t().contiguous() / 8.0
        out[:, h] = torch.softmax(scores.masked_fill(hidden, float("-inf")), dim=-1) @ v[h // group, :s]
    return out.reshape(t, heads * 64)


def _exact_model(cfg: LlamaConfig, w: dict[str, torch.Tensor], tokens: torch.Tensor, first: int, k_cache, v_cache):
    """Logits of the last of `tokens`, which stand at positions first .., and the caches after them, in 64 bits."""
    def linear(name, x):
        return x @ _dense(w[name + ".packed_weights"], w[name + ".scales"]).t().contiguous()

    def norm(name, x):
        return x * torch.rsqrt(x.pow(2).mean(dim=-1, keepdim=True) + cfg.rms_norm_eps) * w[name + ".weight"].double()

    t, h, kv = tokens.numel(), cfg.hidden_size, cfg.num_kv_heads
    cos, sin = (table[first:first + t].double() for table in _tables(cfg.max_seq_len))
    k_cache, v_cache = k_cache.double(), v_cache.double()
    x = w["embed"][tokens].double()
    for i in range(cfg.num_layers):
        p = f"layers.{i}."
        n = norm(p + "input_norm", x)
        q = _rotate(linear(p + "q_proj", n).reshape(t, cfg.num_heads, 64), cos, sin)
        k = _rotate(linear(p + "k_proj", n).reshape(t, kv, 64), cos, sin)
        v = linear(p + "v_proj", n).reshape(t, kv, 64)
        k_cache[i, :, first:first + t] = k.transpose(0, 1)
        v_cache[i, :, first:first + t] = v.transpose(0, 1)
        x = x + linear(p + "o_proj", _attend(q, k_cache[i], v_cache[i], first))
        n = norm(p + "post_norm", x)
        x = x + linear(p + "down_proj", F.silu(linear(p + "gate_proj", n)) * linear(p + "up_proj", n))
    return {"logits": linear("lm_head", norm("norm", x[-1:]))[0], "k": k_cache, "v": v_cache}


# ------------------------------------------------------------------ the inputs
# one function a kind, for prepare() and exact() alike

def _linear_inputs(case: dict, seed: int):
    gen = _gen(seed)
    x = _rows(case["m"], case["k"], gen)
    return x, [_weights(case["n"], case["k"], case["group"], gen) for _ in range(case["copies"])]


def _quantize_input(case: dict, seed: int) -> torch.Tensor:
    w = torch.randn((case["n"], case["k"]), device=DEVICE, generator=_gen(seed)) * INIT_STD
    return w.to(torch.float16) if case["dtype"] == "fp16" else w


def _attention_inputs(case: dict, seed: int):
    gen = _gen(seed)
    k, v = _caches(case["layers"], case["kv_heads"], case["slots"], case["position"], gen)
    return _rows(case["layers"], (case["heads"] + 2 * case["kv_heads"]) * 64, gen), k, v


def _decode_inputs(case: dict, seed: int):
    cfg = LlamaConfig(max_seq_len=case["max_seq_len"])
    gen = _gen(seed + 1)
    k, v = _caches(cfg.num_layers, cfg.num_kv_heads, cfg.max_seq_len, case["position"], gen)
    return cfg, torch.randint(0, cfg.vocab_size, (1,), device=DEVICE, generator=gen), k, v


def _prefill_inputs(case: dict, seed: int):
    cfg = LlamaConfig(max_seq_len=case["max_seq_len"])
    return cfg, torch.randint(0, cfg.vocab_size, (case["tokens"],), device=DEVICE, generator=_gen(seed + 1))


@torch.inference_mode()
def prepare(case: dict, seed: int) -> dict:
    kind = case["kind"]
    state: dict = {"kind": kind, "case": case}
    if kind == "linear":
        x, weights = _linear_inputs(case, seed)
        layers = [QuantizedLinear(p, s, group_size=case["group"]) for p, s in weights]
        state.update(x=x, layers=layers)
        if case["graph"]:
            state["graph"], state["out"] = _record(lambda: [layer(x) for layer in layers])
    elif kind == "dequantize":
        state["packed"], state["scales"] = _weights(case["n"], case["k"], case["group"], _gen(seed))
    elif kind == "quantize":
        state["weights"] = _quantize_input(case, seed)
    elif kind == "decode_attention":
        qkv, k, v = _attention_inputs(case, seed)
        cos, sin = _tables(case["slots"])
        heads, kv_heads = case["heads"], case["kv_heads"]
        splits = min(max(1, 256 // heads), max(1, case["slots"] // 128), 64)   # the decoder's own choice
        out = torch.empty((case["layers"], heads * 64), dtype=torch.float16, device=DEVICE)
        state.update(qkv=qkv, k=k, v=v, cos=cos, sin=sin, out=out,
                     position=torch.full((1,), case["position"], dtype=torch.int64, device=DEVICE),
                     workspace=torch.empty((heads * splits * 66,), dtype=torch.float32, device=DEVICE))

        def layers_():
            for i in range(case["layers"]):
                _lib.decode_attention_split_f16(qkv[i], k[i], v[i], cos, sin, state["position"], out[i], heads,
                                                kv_heads, splits, state["workspace"])

        state["graph"], _ = _record(layers_)
    elif kind == "decode":
        cfg, token, k, v = _decode_inputs(case, seed)
        decoder = _decoder(cfg, seed)
        decoder.k_cache.copy_(k)
        decoder.v_cache.copy_(v)
        decoder.host_position = case["position"]
        decoder.position.fill_(case["position"])
        decoder.token.copy_(token)
        decoder.capture()
        # capturing runs steps and puts the state back; the slots it may have written are as given again
        decoder.k_cache.copy_(k)
        decoder.v_cache.copy_(v)
        state.update(decoder=decoder, token=token)
    elif kind == "prefill":
        cfg, prompt = _prefill_inputs(case, seed)
        decoder = _decoder(cfg, seed)
        decoder.capture_prefill(case["tokens"])
        state.update(decoder=decoder, prompt=prompt)
    return state


@torch.inference_mode()
def run(state: dict):
    kind = state["kind"]
    if kind == "linear":
        if "graph" in state:
            state["graph"].replay()
            return state["out"]
        return [layer(state["x"]) for layer in state["layers"]]
    if kind == "dequantize":
        return torch.ops.w4a16.dequantize(state["packed"], state["scales"], state["case"]["group"])
    if kind == "quantize":
        return quantize_and_pack_weights(state["weights"], state["case"]["group"])
    if kind == "decode_attention":
        state["graph"].replay()
        return {"out": state["out"], "k": state["k"], "v": state["v"]}
    decoder = state["decoder"]
    if kind == "decode":
        # the given token at the given position (a forced token, as when a prompt's last one is decoded again)
        decoder.host_position = state["case"]["position"]
        decoder.position.fill_(state["case"]["position"])
        _lib.embedding_f16(decoder.embed, state["token"], decoder.x_buf)
        decoder.replay()
    else:
        decoder.prefill(state["prompt"])
    return {"logits": decoder.logits, "k": decoder.k_cache, "v": decoder.v_cache}


def work(case: dict) -> dict:
    kind = case["kind"]
    if kind == "linear":
        m, n, k = case["m"], case["n"], case["k"]
        one = n * k / 2 + 2 * n * (k // case["group"]) + 2 * m * k + 2 * m * n
        return {"bytes": case["copies"] * one, "flops": case["copies"] * 2.0 * m * n * k}
    if kind in ("dequantize", "quantize"):
        n, k = case["n"], case["k"]
        packed = n * k / 2 + 2 * n * (k // case["group"])
        wide = 4 if case.get("dtype") == "fp32" else 2
        return {"bytes": packed + wide * n * k, "flops": float(n * k)}
    if kind == "decode_attention":
        seen = case["position"] + 1
        one = 2 * 2 * case["kv_heads"] * 64 * seen + 2 * 64 * (2 * case["heads"] + 4 * case["kv_heads"])
        return {"bytes": case["layers"] * one, "flops": case["layers"] * 4.0 * case["heads"] * 64 * seen}
    cfg = LlamaConfig()
    h, kv, inter = cfg.hidden_size, cfg.num_kv_heads * cfg.head_dim, cfg.intermediate_size
    layer = h * (2 * h + 2 * kv) + 3 * h * inter
    weights = cfg.num_layers * layer + cfg.vocab_size * h
    t, first = (1, case["position"]) if kind == "decode" else (case["tokens"], 0)
    seen = sum(first + i + 1 for i in range(t))
    cache = 2 * 2 * cfg.num_layers * kv * (first + t)
    return {"bytes": weights * (0.5 + 2 / 128) + cache + 2 * t * h + 2 * cfg.vocab_size,
            "flops": 2.0 * (t * cfg.num_layers * layer + cfg.vocab_size * h)
            + 4.0 * cfg.num_layers * cfg.num_heads * cfg.head_dim * seen}


def tolerance(case: dict):
    """Bytes, codes and the fp16 product of one code and one scale are exact.
    The others state about four times the error against 64 bits."""
    kind = case["kind"]
    if kind in ("dequantize", "quantize"):
        return "exact"
    if kind == "linear":
        # measured 2.1e-4 (fp16 rounding of the output), 2.8e-4 with fp16 weights
        return {"rel": 1.1e-3 if case["m"] > 8 else 9e-4}
    if kind == "decode_attention":
        return {"rel": 1.2e-3}   # measured 3.0e-4
    return {"rel": 1.6e-2}       # measured 3.9e-3, 22 layers of fp16 roundings


@torch.inference_mode()
def exact(case: dict, seed: int):
    kind = case["kind"]
    if kind == "linear":
        x, weights = _linear_inputs(case, seed)
        return [x.double() @ _dense(p, s).t().contiguous() for p, s in weights]
    if kind == "dequantize":
        return _dense(*_weights(case["n"], case["k"], case["group"], _gen(seed)))
    if kind == "quantize":
        w, group = _quantize_input(case, seed).double(), case["group"]
        return None, w.reshape(case["n"], -1, group).abs().amax(dim=2) / 7.0
    if kind == "decode_attention":
        qkv, k, v = _attention_inputs(case, seed)
        heads, kv_heads, at = case["heads"], case["kv_heads"], case["position"]
        cos, sin = (table[at:at + 1].double() for table in _tables(case["slots"]))
        k, v, out = k.double(), v.double(), []
        for i in range(case["layers"]):
            row = qkv[i].double().reshape(1, heads + 2 * kv_heads, 64)
            k[i, :, at] = _rotate(row[:, heads:heads + kv_heads], cos, sin)[0]
            v[i, :, at] = row[0, heads + kv_heads:]
            out.append(_attend(_rotate(row[:, :heads], cos, sin), k[i], v[i], at)[0])
        return {"out": torch.stack(out), "k": k, "v": v}
    if kind == "decode":
        cfg, token, k, v = _decode_inputs(case, seed)
        return _exact_model(cfg, _decoder_weights(cfg, seed), token, case["position"], k, v)
    cfg, prompt = _prefill_inputs(case, seed)
    shape = (cfg.num_layers, cfg.num_kv_heads, cfg.max_seq_len, 64)
    empty = torch.zeros(shape, device=DEVICE, dtype=torch.float16)
    return _exact_model(cfg, _decoder_weights(cfg, seed), prompt, 0, empty, empty)
