"""The work a user has this framework do, as cases to time and compare.

Kinds of case, each through a public entry point:

    linear      one quantized linear (kernels.quantized_linear): the GEMV up to 8 rows, the matrix cores above
    mlp         the prefill MLP's three products (kernels.gemm_swiglu, then kernels.quantized_linear)
    attention   prefill attention (kernels.flash_attn_prefill, kernels.flash_attn_segments)
    decode      one greedy decode step replayed from a HIP graph, then its logits (Qwen3Decoder)
    prefill     a prompt through the chunked prefill, then its last token's logits (Qwen3Decoder.prefill_chunked)
    encoder     an utterance through the Qwen3-ASR audio tower (Qwen3AudioEncoder.run_audio_encoder)
    codec       codec frames to a waveform (OmniVoiceAudioDecoder.decode)
    quantize    one fp32 checkpoint matrix to GGUF rows (kernels.quantize)

Weights are packed GGUF blocks drawn at random with the code and scale distributions that quantizing N(0, 0.02)
gives; ``exact`` decodes the same bytes and repeats the mathematics in 64 bits with plain torch.
"""

from __future__ import annotations

import math
import random

import numpy as np
import torch
import torch.nn.functional as F

from torch2vk_amd import kernels
from torch2vk_amd.omnivoice.decoder import AudioDecoderConfig, OmniVoiceAudioDecoder, dense_shapes
from torch2vk_amd.qwen3.config import QWEN3_0_6B, QWEN3_1_7B, QWEN3_8B, Qwen3Config, tensor_types
from torch2vk_amd.qwen3.model import Qwen3Decoder
from torch2vk_amd.qwen3.weights import Qwen3Weights, matrix_shapes, norm_shapes, stack_qkv
from torch2vk_amd.qwen3_asr import preprocess
from torch2vk_amd.qwen3_asr.config import QWEN3_ASR_0_6B_AUDIO, AudioEncoderConfig
from torch2vk_amd.qwen3_asr.encoder import PREFIX, AudioEncoderWeights, Qwen3AudioEncoder, audio_tensor_shapes

DEVICE = "cuda"
MODELS = {"0.6b": QWEN3_0_6B, "1.7b": QWEN3_1_7B, "8b": QWEN3_8B}
WEIGHT_STD = 0.02
# the audio codec's decoder: 8 codebooks of 1024 codes, five upsampling blocks, 960 samples a frame
CODEC = AudioDecoderConfig(codebooks=8, vocab=1024, codebook_dim=64, latent=1024, hidden=256, channels=1024,
                           strides=(8, 5, 4, 2, 3))
CODEC_DILATIONS = (1, 3, 9)


# ------------------------------------------------------------------ cases --


def listed() -> list[dict]:
    return [
        # one projection of the 0.6B decode, called by itself: launch and latency are all it costs
        {"name": "linear_1x1024x3072_q4_k", "kind": "linear", "wtype": "q4_k", "m": 1, "k": 1024, "n": 3072,
         "residual": False},
        # o_proj of an 8B prompt's last, short chunk of a few tokens
        {"name": "linear_6x4096x4096_q4_k", "kind": "linear", "wtype": "q4_k", "m": 6, "k": 4096, "n": 4096,
         "residual": True},
        # a checkpoint's q_proj packed for export
        {"name": "quantize_4096x4096_q4_k", "kind": "quantize", "wtype": "q4_k", "rows": 4096, "k": 4096},
        # chat on the small model: Q4_K_M weights, a context of a few hundred tokens
        {"name": "decode_0.6b_200", "kind": "decode", "model": "0.6b", "layers": 28, "policy": "q4_k_m",
         "position": 200, "capacity": 512},
        # the headline workload: the 8B shape, int4, 4096 tokens of context, every layer
        {"name": "decode_8b_4096", "kind": "decode", "model": "8b", "layers": 36, "policy": "uniform",
         "position": 4096, "capacity": 4352},
        # a long document: past the persistent kernel's 8192 positions, one launch per operation
        {"name": "decode_8b_12000_4_layers", "kind": "decode", "model": "8b", "layers": 4, "policy": "q4_k_m",
         "position": 12000, "capacity": 16384},
        # a short chat prompt before the first token
        {"name": "prefill_0.6b_128_4_layers", "kind": "prefill", "model": "0.6b", "layers": 4, "policy": "q4_k_m",
         "tokens": 128, "past": 0},
        # a ragged long prompt of the 8B shape, one layer of it (Q6_K v and down, as its first layers have)
        {"name": "prefill_8b_1901_1_layer", "kind": "prefill", "model": "8b", "layers": 1, "policy": "q4_k_m",
         "tokens": 1901, "past": 0},
        # the MLP of the batched prefill, 8 sequences of 2048 tokens, int8 weights: the largest products there are
        {"name": "mlp_16384_8b_q8_0", "kind": "mlp", "wtype": "q8_0", "m": 16384, "k": 4096, "f": 12288},
        # the attention of the same prefill
        {"name": "attention_8x2048_causal", "kind": "attention", "mode": "causal", "batch": 8, "tokens": 2048,
         "past": 0, "heads": 32, "kv_heads": 8, "dim": 128},
        # 40 s of speech through the convolutions, three encoder layers and the head
        {"name": "encoder_4000_frames_3_layers", "kind": "encoder", "frames": 4000, "layers": 3},
        # 3 s of speech out of the codec
        {"name": "codec_75_frames", "kind": "codec", "frames": 75},
    ]


def _log(rng: random.Random, lo: int, hi: int) -> int:
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng: random.Random) -> dict:
    kind = rng.choice(("linear", "linear", "mlp", "attention", "decode", "prefill", "encoder", "codec", "quantize"))
    wtype = rng.choice(("q4_k", "q6_k", "q8_0"))
    if kind == "linear":
        m = _log(rng, 1, 8) if rng.random() < 0.5 else _log(rng, 9, 4096)
        n = rng.choice((1024, 2048, 3072, 4096, 6144, 12288)) if rng.random() < 0.7 else _log(rng, 100, 12288)
        return {"kind": kind, "wtype": wtype, "m": m, "k": rng.choice((1024, 2048, 3072, 4096, 6144, 12288)), "n": n,
                "residual": rng.random() < 0.5}
    if kind == "mlp":
        c = MODELS[rng.choice(tuple(MODELS))]
        return {"kind": kind, "wtype": wtype, "m": _log(rng, 9, 12000), "k": c.hidden, "f": c.mlp}
    if kind == "attention":
        mode = rng.choice(("causal", "causal", "mask", "segments"))
        if mode == "segments":  # the audio tower's windows
            return {"kind": kind, "mode": mode, "batch": 1, "tokens": _log(rng, 40, 6000), "past": 0, "heads": 14,
                    "kv_heads": 14, "dim": 64}
        heads = rng.choice((16, 32))
        return {"kind": kind, "mode": mode, "batch": rng.choice((1, 1, 2, 4)), "tokens": _log(rng, 20, 2048),
                "past": 0 if mode == "mask" or rng.random() < 0.6 else _log(rng, 16, 2048), "heads": heads,
                "kv_heads": 8, "dim": 128}
    if kind == "decode":
        model = rng.choice(tuple(MODELS))
        long = rng.random() < 0.3
        capacity = 16384 if long else rng.choice((512, 2048, 4352, 8192))
        return {"kind": kind, "model": model, "layers": rng.choice((2, 4, 8)),
                "policy": rng.choice(("uniform", "q4_k_m")),
                "position": _log(rng, 8000, 16000) if long else _log(rng, 16, capacity - 1), "capacity": capacity}
    if kind == "prefill":
        return {"kind": kind, "model": rng.choice(tuple(MODELS)), "layers": rng.choice((1, 2)),
                "policy": rng.choice(("uniform", "q4_k_m")), "tokens": _log(rng, 10, 2600),
                "past": 0 if rng.random() < 0.6 else _log(rng, 16, 1024)}
    if kind == "encoder":
        return {"kind": kind, "frames": _log(rng, 60, 4000), "layers": rng.choice((1, 2, 3))}
    if kind == "codec":
        return {"kind": kind, "frames": _log(rng, 5, 75)}
    return {"kind": kind, "wtype": wtype, "rows": _log(rng, 64, 8192), "k": rng.choice((1024, 2048, 3072, 4096))}


# ---------------------------------------------------- packed random weights --


def _gen(seed: int) -> torch.Generator:
    return torch.Generator(device=DEVICE).manual_seed(int(seed))


def _randn(g: torch.Generator, *shape: int) -> torch.Tensor:
    return torch.randn(*shape, generator=g, device=DEVICE, dtype=torch.float32)


def _rand_codes(g: torch.Generator, lo: int, hi: int, *shape: int) -> torch.Tensor:
    return torch.randint(lo, hi + 1, shape, generator=g, device=DEVICE, dtype=torch.int32)


def _f16_bytes(v: torch.Tensor) -> torch.Tensor:
    return v.to(torch.float16).unsqueeze(-1).contiguous().view(torch.uint8)


def _rows(g: torch.Generator, wtype: str, n: int, k: int, std: float = WEIGHT_STD) -> torch.Tensor:
    """uint8 GGUF rows [n, bytes] of n x k values of standard deviation about ``std`` (Q8_0 rows padded to 32)."""
    if wtype == "q8_0":
        nb = n * (-(-k // 32))
        q = (_randn(g, nb, 32) * 42.0).round_().clamp_(-127, 127).to(torch.int8)
        q[:, 0] = 127  # the quantizer's scale is the block's largest magnitude over 127
        d = (0.8 + 0.4 * torch.rand(nb, generator=g, device=DEVICE)) * (std / 42.0)
        return torch.cat([_f16_bytes(d), q.view(torch.uint8)], dim=1).view(n, -1)
    nb = n * k // 256
    if wtype == "q4_k":
        q = (_randn(g, nb, 4, 2, 32) * 2.9 + 7.5).round_().clamp_(0, 15).to(torch.uint8)
        nib = (q[:, :, 0] | (q[:, :, 1] << 4)).view(nb, 128)
        sc, mn = _rand_codes(g, 40, 63, nb, 8), _rand_codes(g, 40, 63, nb, 8)
        packed = torch.cat([(sc[:, :4] | ((sc[:, 4:] & 48) << 2)), (mn[:, :4] | ((mn[:, 4:] & 48) << 2)),
                            ((sc[:, 4:] & 15) | ((mn[:, 4:] & 15) << 4))], dim=1).to(torch.uint8)
        d = (0.8 + 0.4 * torch.rand(nb, generator=g, device=DEVICE)) * (std / (2.9 * 51.5))
        return torch.cat([_f16_bytes(d), _f16_bytes(7.5 * d), packed, nib], dim=1).view(n, -1)
    q = (_randn(g, nb, 2, 4, 32) * 11.0 + 32.0).round_().clamp_(0, 63).to(torch.uint8)  # [half, part, value]
    ql = torch.cat([(q[:, :, 0] & 15) | ((q[:, :, 2] & 15) << 4), (q[:, :, 1] & 15) | ((q[:, :, 3] & 15) << 4)], dim=2)
    qh = (q[:, :, 0] >> 4) | ((q[:, :, 1] >> 4) << 2) | ((q[:, :, 2] >> 4) << 4) | ((q[:, :, 3] >> 4) << 6)
    sc = _rand_codes(g, 50, 127, nb, 16).to(torch.int8).view(torch.uint8)
    d = (0.8 + 0.4 * torch.rand(nb, generator=g, device=DEVICE)) * (std / (11.0 * 88.5))
    return torch.cat([ql.reshape(nb, 128), qh.reshape(nb, 64), sc, _f16_bytes(d)], dim=1).view(n, -1)


def _f64(block: torch.Tensor) -> torch.Tensor:
    """float64 [blocks] of two fp16 bytes per block."""
    return block.contiguous().view(torch.float16).to(torch.float64).view(-1)


def _dense(rows: torch.Tensor, k: int) -> torch.Tensor:
    """float64 [n, k] of packed rows (the type follows from the row's width)."""
    n, width = rows.shape
    if k % 256 == 0 and width == k // 256 * 144:
        b = rows.reshape(-1, 144)
        s = b[:, 4:16].to(torch.int32)
        sc = torch.cat([s[:, :4] & 63, (s[:, 8:] & 15) | ((s[:, :4] >> 6) << 4)], dim=1).to(torch.float64)
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:] >> 4) | ((s[:, 4:8] >> 6) << 4)], dim=1).to(torch.float64)
        nib = b[:, 16:].reshape(-1, 4, 1, 32)
        q = torch.cat([nib & 15, nib >> 4], dim=2).reshape(-1, 8, 32).to(torch.float64)
        return ((_f64(b[:, :2])[:, None] * sc)[:, :, None] * q -
                (_f64(b[:, 2:4])[:, None] * mn)[:, :, None]).view(n, k)
    if k % 256 == 0 and width == k // 256 * 210:
        b = rows.reshape(-1, 210)
        ql, qh = b[:, :128].reshape(-1, 2, 2, 32), b[:, 128:192].reshape(-1, 2, 1, 32)
        q = torch.cat([ql & 15, ql >> 4], dim=2)  # parts 0, 1 then 2, 3
        hi = torch.cat([(qh >> s) & 3 for s in (0, 2, 4, 6)], dim=2)
        q = (q | (hi << 4)).to(torch.float64) - 32.0
        sc = b[:, 192:208].contiguous().view(torch.int8).to(torch.float64).view(-1, 16, 1)
        return (_f64(b[:, 208:])[:, None, None] * sc * q.reshape(-1, 16, 16)).view(n, k)
    b = rows.reshape(-1, 34)
    q = b[:, 2:].contiguous().view(torch.int8).to(torch.float64)
    return (_f64(b[:, :2])[:, None] * q).view(n, -1)[:, :k]


def _row_bytes(wtype: str, k: int) -> int:
    return {"q4_k": k // 256 * 144, "q6_k": k // 256 * 210, "q8_0": -(-k // 32) * 34}[wtype]


# ------------------------------------------------------------ Qwen3 models --


def _config(case: dict) -> Qwen3Config:
    c = MODELS[case["model"]]
    return Qwen3Config(f"{c.name}-{case['layers']}", c.hidden, case["layers"], c.heads, c.kv_heads, c.head_dim, c.mlp,
                       c.vocab, c.rope_theta, c.rms_eps, c.eos_token_ids)


def _model_inputs(case: dict, seed: int) -> dict:
    """A decoder's weights, cache rows and tokens, from the seed alone."""
    g, c = _gen(seed), _config(case)
    types = tensor_types(c, case["policy"])
    packed = {name: _rows(g, types[name], n, k) for name, (n, k) in matrix_shapes(c).items()}
    norms = {name: 1.0 + 0.1 * _randn(g, n) for name, n in norm_shapes(c).items()}
    past = case["position"] if case["kind"] == "decode" else case["past"]
    kv = [_randn(g, c.layers, past, c.kv_heads, c.head_dim).to(torch.bfloat16) for _ in range(2)]
    tokens = torch.randint(0, c.vocab - 300, (case.get("tokens", 1),), generator=g, device=DEVICE)
    return {"config": c, "types": types, "packed": packed, "norms": norms, "kv": kv, "tokens": tokens, "past": past}


def _prepare_model(case: dict, seed: int) -> dict:
    i = _model_inputs(case, seed)
    w = Qwen3Weights(config=i["config"], policy=case["policy"], packed=i["packed"], types=i["types"],
                     norms=i["norms"])
    stack_qkv(w)
    capacity = case["capacity"] if case["kind"] == "decode" else case["past"] + case["tokens"] + 64
    dec = Qwen3Decoder(w, max_positions=capacity, max_new_tokens=64)
    dec.stop_on_eos = False
    if case["kind"] == "decode":
        dec.graph(1)  # a serving loop replays captured steps
    dec.k_cache[:, :i["past"]] = i["kv"][0]
    dec.v_cache[:, :i["past"]] = i["kv"][1]
    return {"decoder": dec, "tokens": i["tokens"], "token": int(i["tokens"][0]), "past": i["past"]}


def _run_decode(state: dict) -> tuple:
    dec, past = state["decoder"], state["past"]
    dec.position.fill_(past)
    dec.next_token.fill_(state["token"])
    dec.run_steps(1, steps_per_graph=1)
    return dec.logits(), dec.k_cache[:, past], dec.v_cache[:, past]


def _run_prefill(state: dict) -> tuple:
    dec, past, n = state["decoder"], state["past"], state["tokens"].numel()
    dec.prefill_chunked(state["tokens"], start=past)
    return dec.logits(), dec.k_cache[:, past:past + n], dec.v_cache[:, past:past + n]


def _rms(x: torch.Tensor, w: torch.Tensor, eps: float) -> torch.Tensor:
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * w.double()


def _rope(x: torch.Tensor, pos: torch.Tensor, theta: float) -> torch.Tensor:
    """x [T, heads, 128] rotated by halves at positions pos."""
    half = x.shape[-1] // 2
    freq = theta ** (-torch.arange(half, device=x.device, dtype=torch.float64) / half)
    ang = pos.double()[:, None, None] * freq
    cos, sin = ang.cos(), ang.sin()
    a, b = x[..., :half], x[..., half:]
    return torch.cat([a * cos - b * sin, b * cos + a * sin], dim=-1)


def _sdpa(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, visible) -> torch.Tensor:
    """float64 q [T, NH, D], k / v [S, NK, D] -> [T, NH, D]; ``visible`` [T, S] is True, or the additive mask."""
    t, nh, d = q.shape
    group = nh // k.shape[1]
    out = torch.empty_like(q)
    for h in range(nh):
        s = q[:, h] @ k[:, h // group].T / math.sqrt(d)
        s = s.masked_fill(~visible, -math.inf) if visible.dtype == torch.bool else s + visible
        out[:, h] = torch.softmax(s, dim=-1) @ v[:, h // group]
    return out


def _exact_model(case: dict, seed: int) -> tuple:
    i = _model_inputs(case, seed)
    c, p, nrm, past, t = i["config"], i["packed"], i["norms"], i["past"], i["tokens"].numel()
    pos = torch.arange(past, past + t, device=DEVICE)
    visible = torch.arange(past + t, device=DEVICE)[None, :] <= pos[:, None]
    h = _dense(p["embed"][i["tokens"]], c.hidden)
    keys, values = [], []
    for layer in range(c.layers):
        def lin(x: torch.Tensor, name: str) -> torch.Tensor:
            return x @ _dense(p[f"layers.{layer}.{name}"], x.shape[-1]).T
        def nw(name: str) -> torch.Tensor:
            return nrm[f"layers.{layer}.{name}"]
        x = _rms(h, nw("input_norm"), c.rms_eps)
        q, k, v = (lin(x, n).view(t, -1, c.head_dim) for n in ("q", "k", "v"))
        q = _rope(_rms(q, nw("q_norm"), c.rms_eps), pos, c.rope_theta)
        k = _rope(_rms(k, nw("k_norm"), c.rms_eps), pos, c.rope_theta)
        keys.append(k)
        values.append(v)
        kk = torch.cat([i["kv"][0][layer].double(), k])
        vv = torch.cat([i["kv"][1][layer].double(), v])
        h = h + lin(_sdpa(q, kk, vv, visible).reshape(t, -1), "o")
        x = _rms(h, nw("post_norm"), c.rms_eps)
        h = h + lin(F.silu(lin(x, "gate")) * lin(x, "up"), "down")
    x = _rms(h[-1], nrm["norm"], c.rms_eps)
    logits = torch.cat([_dense(part, c.hidden) @ x for part in p["lm_head"].split(16384)])
    k, v = torch.stack(keys), torch.stack(values)
    return (logits, k[:, 0], v[:, 0]) if case["kind"] == "decode" else (logits, k, v)


# --------------------------------------------------------- linears and MLPs --


def _linear_inputs(case: dict, seed: int) -> dict:
    g = _gen(seed)
    x = _randn(g, case["m"], case["k"]).to(torch.bfloat16)
    w = _rows(g, case["wtype"], case["n"], case["k"])
    return {"x": x, "w": w, "residual": _randn(g, case["m"], case["n"]) if case["residual"] else None,
            "wtype": case["wtype"]}


def _run_linear(s: dict) -> torch.Tensor:
    return kernels.quantized_linear(s["x"], s["w"], s["wtype"], residual=s["residual"])


def _exact_linear(case: dict, seed: int) -> torch.Tensor:
    s = _linear_inputs(case, seed)
    y = s["x"].double() @ _dense(s["w"], case["k"]).T
    return y if s["residual"] is None else y + s["residual"].double()


def _mlp_inputs(case: dict, seed: int) -> dict:
    g, m, k, f = _gen(seed), case["m"], case["k"], case["f"]
    return {"x": _randn(g, m, k).to(torch.bfloat16), "gate": _rows(g, case["wtype"], f, k),
            "up": _rows(g, case["wtype"], f, k), "down": _rows(g, case["wtype"], k, f), "h": _randn(g, m, k),
            "wtype": case["wtype"]}


def _run_mlp(s: dict) -> torch.Tensor:
    act = kernels.gemm_swiglu(s["x"], s["gate"], s["up"], s["wtype"])
    return kernels.quantized_linear(act, s["down"], s["wtype"], residual=s["h"])


def _exact_mlp(case: dict, seed: int) -> torch.Tensor:
    s = _mlp_inputs(case, seed)
    gate, up, down = _dense(s["gate"], case["k"]), _dense(s["up"], case["k"]), _dense(s["down"], case["f"])
    parts = [F.silu(x.double() @ gate.T) * (x.double() @ up.T) @ down.T for x in s["x"].split(2048)]
    return torch.cat(parts) + s["h"].double()


# ---------------------------------------------------------------- attention --


def _window_bounds(tokens: int) -> list[int]:
    """The audio tower's windows: 104 tokens each, then the rest."""
    return list(range(0, tokens, 104)) + [tokens]


def _attention_inputs(case: dict, seed: int) -> dict:
    g, b, t = _gen(seed), case["batch"], case["tokens"]
    s = case["past"] + t
    q = _randn(g, b, t, case["heads"], case["dim"]).to(torch.bfloat16)
    k, v = (_randn(g, b, s, case["kv_heads"], case["dim"]).to(torch.bfloat16) for _ in range(2))
    out = {"q": q, "k": k, "v": v, "mode": case["mode"], "past": case["past"]}
    if case["mode"] == "mask":  # a generated span that only sees itself and a prompt that sees everything
        mask = torch.zeros(1, t, s, device=DEVICE)
        mask[:, :t // 3, t // 3:] = -math.inf
        out["mask"] = mask
    elif case["mode"] == "segments":
        out["cu"] = torch.tensor(_window_bounds(t), dtype=torch.int32, device=DEVICE)
    return out


def _run_attention(s: dict) -> torch.Tensor:
    if s["mode"] == "segments":
        return kernels.flash_attn_segments(s["q"], s["k"], s["v"], s["cu"])
    if s["mode"] == "mask":
        return kernels.flash_attn_prefill(s["q"], s["k"], s["v"], causal=False, mask=s["mask"])
    return kernels.flash_attn_prefill(s["q"], s["k"], s["v"], causal=True, causal_offset=s["past"])


def _visible(case: dict, s: dict) -> torch.Tensor:
    t, n = case["tokens"], case["past"] + case["tokens"]
    if case["mode"] == "mask":
        return s["mask"][0].double()
    if case["mode"] == "segments":
        seg = torch.arange(t, device=DEVICE) // 104
        return seg[:, None] == seg[None, :]
    return torch.arange(n, device=DEVICE)[None, :] <= case["past"] + torch.arange(t, device=DEVICE)[:, None]


def _exact_attention(case: dict, seed: int) -> torch.Tensor:
    s = _attention_inputs(case, seed)
    visible = _visible(case, s)
    return torch.stack([_sdpa(q.double(), k.double(), v.double(), visible)
                        for q, k, v in zip(s["q"], s["k"], s["v"])])


# ------------------------------------------------------------ audio encoder --


def _encoder_config(case: dict) -> AudioEncoderConfig:
    a = QWEN3_ASR_0_6B_AUDIO
    return AudioEncoderConfig(d_model=a.d_model, layers=case["layers"], heads=a.heads, ffn=a.ffn,
                              output_dim=a.output_dim)


def _encoder_inputs(case: dict, seed: int) -> dict:
    g, cfg = _gen(seed), _encoder_config(case)
    packed, vectors = {}, {}
    for name, shape in audio_tensor_shapes(cfg).items():
        if len(shape) == 1:
            norm = "norm.weight" in name or name.endswith("ln_post.weight")
            vectors[name] = _randn(g, *shape) * 0.05 + (1.0 if norm else 0.0)
            continue
        cols = math.prod(shape[1:])
        std = 1.0 / math.sqrt(cols) if len(shape) == 4 or "conv_out" in name else WEIGHT_STD
        packed[name] = _rows(g, "q8_0", shape[0], cols, std)
    mel = _randn(g, cfg.mel_bins, case["frames"]).cpu().numpy()
    inp = preprocess.preprocess_audio_inputs(np.zeros(0), mel, np.ones(case["frames"]), cfg)
    dev = {n: torch.from_numpy(inp[n].copy()).to(DEVICE) for n in ("padded_feature", "position_embedding", "compact_index")}
    return {"config": cfg, "packed": packed, "vectors": vectors, "cu": inp["cu_seqlens"], **dev}


def _prepare_encoder(case: dict, seed: int) -> dict:
    i = _encoder_inputs(case, seed)
    return {"encoder": Qwen3AudioEncoder(AudioEncoderWeights(i["config"], i["packed"], i["vectors"])), "inputs": i}


def _run_encoder(s: dict) -> torch.Tensor:
    i = s["inputs"]
    return s["encoder"].run_audio_encoder(i["padded_feature"], i["position_embedding"], i["compact_index"], i["cu"])


def _exact_encoder(case: dict, seed: int) -> torch.Tensor:
    i = _encoder_inputs(case, seed)
    cfg, shapes = i["config"], audio_tensor_shapes(i["config"])

    def w(name: str) -> torch.Tensor:
        return _dense(i["packed"][PREFIX + name], math.prod(shapes[PREFIX + name][1:]))

    def vec(name: str) -> torch.Tensor:
        return i["vectors"][PREFIX + name].double()

    def lin(x: torch.Tensor, name: str) -> torch.Tensor:
        return x @ w(name + ".weight").T + vec(name + ".bias")

    def norm(x: torch.Tensor, name: str) -> torch.Tensor:
        return F.layer_norm(x, x.shape[-1:], vec(name + ".weight"), vec(name + ".bias"), cfg.eps)

    x = i["padded_feature"].double()
    for n in ("conv2d1", "conv2d2", "conv2d3"):
        b, _, hh, ww = x.shape
        taps = F.unfold(x, 3, padding=1, stride=2)  # [B, C 9, positions]
        y = w(n + ".weight") @ taps + vec(n + ".bias")[:, None]
        x = F.gelu(y).view(b, -1, (hh - 1) // 2 + 1, (ww - 1) // 2 + 1)
    b, ch, f, t = x.shape
    x = x.reshape(b, ch * f, t).transpose(1, 2) @ w("conv_out.weight").T + i["position_embedding"].double()
    h = x.reshape(b * t, -1)[i["compact_index"]]
    n_tok, cu = h.shape[0], torch.from_numpy(np.asarray(i["cu"])).to(DEVICE)
    seg = torch.bucketize(torch.arange(n_tok, device=DEVICE), cu[1:], right=True)
    visible = seg[:, None] == seg[None, :]
    for layer in range(cfg.layers):
        p = f"layers.{layer}."
        x = norm(h, p + "self_attn_layer_norm")
        q, k, v = (lin(x, f"{p}self_attn.{n}").view(n_tok, cfg.heads, -1) for n in ("q_proj", "k_proj", "v_proj"))
        h = h + lin(_sdpa(q, k, v, visible).reshape(n_tok, -1), p + "self_attn.out_proj")
        h = h + lin(F.gelu(lin(norm(h, p + "final_layer_norm"), p + "fc1")), p + "fc2")
    return lin(F.gelu(lin(norm(h, "ln_post"), "proj1")), "proj2")


# -------------------------------------------------------------- audio codec --


def _codec_inputs(case: dict, seed: int) -> dict:
    """Dense weights whose every 32-value block is a whole multiple of an fp16 scale with its largest at 127, so
    that packing them as Q8_0 loses nothing; residual branches of small gain, as a trained decoder's are."""
    g, dense = _gen(seed), {}
    for name, shape in dense_shapes(CODEC).items():
        if len(shape) == 1:
            alpha = "alpha" in name or name.endswith((".a1", ".a2"))
            dense[name] = torch.exp(0.3 * _randn(g, *shape)) if alpha else 0.05 * _randn(g, *shape)
            continue
        fan = 2 * shape[0] if name.endswith("convt.w") else shape[1]
        std = 1.0 if name.startswith("cb") else (0.25 if name.endswith("c2.w") else 0.7) / math.sqrt(fan)
        rows = _rows(g, "q8_0", shape[0], shape[1], std)
        full = _dense(rows, -(-shape[1] // 32) * 32)
        full[:, shape[1]:] = 0.0
        dense[name] = full[:, :shape[1]].float()
    codes = torch.randint(0, CODEC.vocab, (CODEC.codebooks, case["frames"]), generator=g, device=DEVICE)
    return {"dense": dense, "codes": codes}


def _prepare_codec(case: dict, seed: int) -> dict:
    i = _codec_inputs(case, seed)
    return {"decoder": OmniVoiceAudioDecoder(CODEC, {n: t.cpu().numpy() for n, t in i["dense"].items()}, DEVICE),
            "codes": i["codes"]}


def _run_codec(s: dict) -> torch.Tensor:
    return s["decoder"].decode(s["codes"])


def _exact_codec(case: dict, seed: int) -> torch.Tensor:
    i = _codec_inputs(case, seed)
    w = {n: t.double() for n, t in i["dense"].items()}

    def conv(x: torch.Tensor, name: str, k: int, dil: int = 1) -> torch.Tensor:  # x [T, C], taps c * k + j
        pad = dil * (k - 1) // 2
        xp = F.pad(x, (0, 0, pad, pad))
        y = w[name + ".b"]
        for j in range(k):
            y = y + xp[j * dil:j * dil + x.shape[0]] @ w[name + ".w"][:, j::k].T
        return y

    def snake(x: torch.Tensor, name: str) -> torch.Tensor:
        return x + torch.sin(w[name] * x) ** 2 / (w[name] + 1e-9)

    x = sum(w[f"cb{c}"][i["codes"][c]] @ w[f"proj{c}.w"].T + w[f"proj{c}.b"] for c in range(CODEC.codebooks))
    x = conv(x @ w["fc2.w"].T + w["fc2.b"], "conv1", 7)
    for b, s in enumerate(CODEC.strides):
        x = snake(x, f"b{b}.alpha")
        t, co = x.shape[0], w[f"b{b}.convt.b"].numel()
        taps = (x @ w[f"b{b}.convt.w"]).view(t, co, 2 * s)
        y = torch.zeros((t + 2) * s, co, dtype=torch.float64, device=DEVICE)
        at = torch.arange(t, device=DEVICE) * s
        for j in range(2 * s):
            y.index_add_(0, at + j, taps[:, :, j])
        first = math.ceil(s / 2)
        x = y[first:first + t * s] + w[f"b{b}.convt.b"]
        for j, dil in enumerate(CODEC_DILATIONS):
            p = f"b{b}.r{j}."
            x = x + conv(snake(conv(snake(x, p + "a1"), p + "c1", 7, dil), p + "a2"), p + "c2", 1)
    return conv(snake(x, "final.alpha"), "conv2", 7).view(-1)


# ---------------------------------------------------------------- quantizers --


def _prepare_quantize(case: dict, seed: int) -> dict:
    return {"x": _randn(_gen(seed), case["rows"], case["k"]) * WEIGHT_STD, "wtype": case["wtype"]}


def _run_quantize(s: dict) -> torch.Tensor:
    return kernels.quantize(s["x"], s["wtype"])


# ------------------------------------------------------------- the interface --

_PREPARE = {"linear": _linear_inputs, "mlp": _mlp_inputs, "attention": _attention_inputs, "decode": _prepare_model,
            "prefill": _prepare_model, "encoder": _prepare_encoder, "codec": _prepare_codec,
            "quantize": _prepare_quantize}
_RUN = {"linear": _run_linear, "mlp": _run_mlp, "attention": _run_attention, "decode": _run_decode,
        "prefill": _run_prefill, "encoder": _run_encoder, "codec": _run_codec, "quantize": _run_quantize}
_EXACT = {"linear": _exact_linear, "mlp": _exact_mlp, "attention": _exact_attention, "decode": _exact_model,
          "prefill": _exact_model, "encoder": _exact_encoder, "codec": _exact_codec}


def prepare(case: dict, seed: int) -> dict:
    return {"kind": case["kind"], **_PREPARE[case["kind"]](case, seed)}


def run(state: dict):
    return _RUN[state["kind"]](state)


def exact(case: dict, seed: int):
    fn = _EXACT.get(case["kind"])  # packed bytes have no 64-bit value
    return None if fn is None else fn(case, seed)


def tolerance(case: dict):
    """About four times the distance to ``exact`` that was measured for the kind (whole models: what 16-bit
    activations leave after every layer, 0.5 % to 2 % measured, with no room for four times that)."""
    kind = case["kind"]
    if kind == "quantize":
        return "exact"
    if kind == "linear" and case["m"] <= 8 and case["n"] % 16 == 0:
        # exact products and 32-bit sums: 7e-6 measured for Q4_K (its offset cancels in the sum), 8e-7 for the others
        return {"rel": 3e-5 if case["wtype"] == "q4_k" else 5e-6}
    if kind in ("decode", "prefill"):
        return {"rel": 0.03}
    # weights and activations rounded to bf16 once per product: 1.7e-3, 3.2e-3, 2.3e-3, 5.7e-3 and 3.1e-3 measured
    return {"rel": {"linear": 7e-3, "mlp": 1.3e-2, "attention": 1e-2, "encoder": 2.3e-2, "codec": 1.3e-2}[kind]}


def _attention_pairs(t: int, past: int, causal: bool) -> int:
    return t * past + (t * (t + 1) // 2 if causal else t * t)


def _work_model(case: dict) -> dict:
    c = _config(case)
    types = tensor_types(c, case["policy"])
    past = case["position"] if case["kind"] == "decode" else case["past"]
    t = case.get("tokens", 1)
    weights, products = 0, 0
    for name, (n, k) in matrix_shapes(c).items():
        if name == "embed":
            weights += t * _row_bytes(types[name], k)
            continue
        weights += n * _row_bytes(types[name], k)
        products += n * k * (1 if name == "lm_head" else t)
    kv_row = 2 * c.layers * c.kv_dim * 2
    pairs = _attention_pairs(t, past, True)
    return {"bytes": weights + kv_row * (past + t) + 4 * c.vocab,
            "flops": 2 * products + 4 * c.layers * c.q_dim * pairs}


def work(case: dict) -> dict:
    kind = case["kind"]
    if kind in ("decode", "prefill"):
        return _work_model(case)
    if kind == "linear":
        m, k, n = case["m"], case["k"], case["n"]
        return {"bytes": n * _row_bytes(case["wtype"], k) + 2 * m * k + (8 if case["residual"] else 4) * m * n,
                "flops": 2 * m * n * k}
    if kind == "mlp":
        m, k, f = case["m"], case["k"], case["f"]
        return {"bytes": 2 * f * _row_bytes(case["wtype"], k) + k * _row_bytes(case["wtype"], f) + 10 * m * k,
                "flops": 6 * m * k * f}
    if kind == "attention":
        b, t, past, d = case["batch"], case["tokens"], case["past"], case["dim"]
        if case["mode"] == "segments":
            pairs = sum((hi - lo) ** 2 for lo, hi in zip(_window_bounds(t), _window_bounds(t)[1:]))
        elif case["mode"] == "mask":
            pairs = t * t - (t // 3) * (t - t // 3)
        else:
            pairs = _attention_pairs(t, past, True)
        mask = 4 * t * t if case["mode"] == "mask" else 0
        return {"bytes": 2 * b * d * (2 * t * case["heads"] + 2 * (past + t) * case["kv_heads"]) + mask,
                "flops": 4 * b * case["heads"] * d * pairs}
    if kind == "quantize":
        n = case["rows"] * case["k"]
        return {"bytes": 4 * n + case["rows"] * _row_bytes(case["wtype"], case["k"]), "flops": 0}
    if kind == "encoder":
        cfg = _encoder_config(case)
        tokens = int(preprocess.feat_extract_output_lengths(case["frames"]))
        chunks = -(-case["frames"] // cfg.chunk_frames)
        weights, flops = 0, 0
        spots = {"conv2d1": 64 * 50, "conv2d2": 32 * 25, "conv2d3": 16 * 13, "conv_out": 13}
        for name, shape in audio_tensor_shapes(cfg).items():
            if len(shape) == 1:
                weights += 4 * shape[0]
                continue
            cols, stem = math.prod(shape[1:]), name[len(PREFIX):].split(".")[0]
            weights += shape[0] * _row_bytes("q8_0", cols)
            flops += 2 * shape[0] * cols * (chunks * spots[stem] if stem in spots else tokens)
        flops += cfg.layers * 4 * cfg.d_model * tokens * min(tokens, 104)
        return {"bytes": weights + 4 * chunks * cfg.mel_bins * cfg.chunk_frames + 4 * tokens * cfg.output_dim,
                "flops": flops}
    t, ch, weights, flops = case["frames"], CODEC.channels, 0, 0
    length, block = t, -1
    for name, shape in dense_shapes(CODEC).items():
        if name.startswith("b") and name.split(".")[0] != f"b{block}":
            block = int(name.split(".")[0][1:])
        if len(shape) == 1:
            weights += 4 * shape[0]
            continue
        if name.startswith("cb"):
            weights += t * _row_bytes("q8_0", shape[1])
            continue
        weights += shape[0] * _row_bytes("q8_0", shape[1])
        flops += 2 * shape[0] * shape[1] * length
        if name.endswith("convt.w"):
            length *= CODEC.strides[block]
    return {"bytes": weights + 8 * CODEC.codebooks * t + 4 * length, "flops": flops}
