"""OmniVoice's acoustic decoder (run_audio_decode, src/models/quantized_omnivoice/dispatch/audio_decode.py:
60-760) on this library's kernels, activations channels-last [T, C] throughout:

    per codebook c: EMBEDDING_Q8_0 -> LINEAR_BIAS (project_out), summed      (lines 66-141)
    LINEAR_BIAS fc2                                                          (line 145)
    CONV1D conv1 (k 7, pad 3)                                                (line 149)
    per block (stride s): snake -> CONV_TRANSPOSE1D (k 2s, pad ceil(s/2), s outputs per input)
                          -> 3 residual units (dilation 1, 3, 9):
                             x + conv_k1(snake(conv_k7,dil(snake(x))))       (lines 151-740)
    snake -> CONV1D conv2 (k 7, pad 3, one output channel)                   (lines 741-755)

Q8_0 weights are the reference's rows as stored: [out, in * k] for conv1d and linears, [in, out * k] for
conv_transpose1d (each row padded to whole 32-value blocks).
"""

from __future__ import annotations

import ctypes
import math
from dataclasses import dataclass

import numpy as np
import torch

from torch2vk_amd import _lib, kernels
from torch2vk_amd._lib import call, ptr, stream_handle

DILATIONS = (1, 3, 9)


@dataclass(frozen=True)
class AudioDecoderConfig:
    codebooks: int
    vocab: int
    codebook_dim: int
    latent: int
    hidden: int
    channels: int              # conv1's output channels; each block halves them
    strides: tuple[int, ...]


def out_len(cfg: AudioDecoderConfig, t: int) -> int:
    """Waveform samples for t codec frames: each block's transposed conv (kernel 2s, padding ceil(s/2), output
    padding s % 2) writes s outputs per input, as the reference's tensors are sized (target_len * 8, * 40, * 160,
    * 320, * 960 for strides 8, 5, 4, 2, 3: src/models/quantized_omnivoice/tensors/audio_decode.py)."""
    for s in cfg.strides:
        t = (t - 1) * s - 2 * math.ceil(s / 2) + 2 * s + s % 2
    return t


def dense_shapes(cfg: AudioDecoderConfig) -> dict[str, tuple[int, ...]]:
    """Logical fp32 shapes: matrices as the rows the reference quantizes, vectors [n]."""
    s = {}
    for c in range(cfg.codebooks):
        s[f"cb{c}"] = (cfg.vocab, cfg.codebook_dim)
        s[f"proj{c}.w"] = (cfg.latent, cfg.codebook_dim)
        s[f"proj{c}.b"] = (cfg.latent,)
    s["fc2.w"], s["fc2.b"] = (cfg.hidden, cfg.latent), (cfg.hidden,)
    s["conv1.w"], s["conv1.b"] = (cfg.channels, cfg.hidden * 7), (cfg.channels,)
    ch = cfg.channels
    for i, st in enumerate(cfg.strides):
        co = ch // 2
        s[f"b{i}.alpha"] = (ch,)
        s[f"b{i}.convt.w"], s[f"b{i}.convt.b"] = (ch, co * 2 * st), (co,)
        for j in range(len(DILATIONS)):
            p = f"b{i}.r{j}."
            s[p + "a1"], s[p + "a2"] = (co,), (co,)
            s[p + "c1.w"], s[p + "c1.b"] = (co, co * 7), (co,)
            s[p + "c2.w"], s[p + "c2.b"] = (co, co), (co,)
        ch = co
    s["final.alpha"] = (ch,)
    s["conv2.w"], s["conv2.b"] = (1, ch * 7), (1,)
    return s


def synthetic_dense(cfg: AudioDecoderConfig, seed: int = 0) -> dict[str, np.ndarray]:
    rng = np.random.default_rng(seed)
    out = {}
    for name, shape in dense_shapes(cfg).items():
        if "alpha" in name or name.endswith(".a1") or name.endswith(".a2"):
            out[name] = (np.abs(rng.standard_normal(shape)) + 0.3).astype(np.float32)
        elif len(shape) == 1:
            out[name] = (rng.standard_normal(shape) * 0.05).astype(np.float32)
        else:
            fan_in = shape[1] if not name.endswith("convt.w") else shape[0]
            out[name] = (rng.standard_normal(shape) / math.sqrt(fan_in)).astype(np.float32)
    return out


def quantize_rows(w: np.ndarray, device) -> torch.Tensor:
    """Q8_0 rows of w [R, K], zero-padded to whole 32-value blocks as the reference stores them."""
    r, k = w.shape
    kp = (k + 31) // 32 * 32
    full = np.zeros((r, kp), np.float32)
    full[:, :k] = w
    return kernels.quantize(torch.from_numpy(full).to(device), "q8_0")


def conv_fragments(rows: list[torch.Tensor], cin: int, taps: int) -> torch.Tensor:
    """Q8_0 conv rows [n, cin * taps] (element c * taps + k), several matrices' inputs side by side, as the bf16
    fragments t2h_codec_decode reads: [tap][step of 16 inputs][tile of 32 columns][64][8]."""
    n, steps = int(rows[0].shape[0]), -(-cin // 32) * 2
    out = torch.empty(taps, steps * len(rows), -(-n // 64) * 2, 64, 8, dtype=torch.bfloat16, device=rows[0].device)
    for i, r in enumerate(rows):
        call("t2h_conv_fragments_q8_0", ptr(r), n, cin, taps, steps * len(rows), steps * i, ptr(out), stream_handle())
    return out


class OmniVoiceAudioDecoder:
    """``w`` holds the packed weights.  The convolutions are also laid out as bf16 fragments when the decoder is
    made (t2h_codec_decode then runs a whole decode as about 40 launches); channel counts that path is not built
    for run operator by operator."""

    def __init__(self, cfg: AudioDecoderConfig, dense: dict[str, np.ndarray], device) -> None:
        self.cfg = cfg
        self.device = torch.device(device)
        self.w = {n: (quantize_rows(a, self.device) if a.ndim == 2 else torch.from_numpy(a).to(self.device))
                  for n, a in dense.items()}
        self._dims = (ctypes.c_uint32 * (6 + len(cfg.strides)))(cfg.codebooks, cfg.codebook_dim, cfg.latent, cfg.hidden,
                                                                cfg.channels, len(cfg.strides), *cfg.strides)
        fused = cfg.codebook_dim % 32 == 0 and cfg.latent % 64 == 0 and cfg.hidden % 64 == 0 and \
            self._workspace_bytes(1) > 0 and self._weights_fit()
        self._plan = self._lay_out() if fused else None

    def _weights_fit(self) -> bool:
        """Whether every weight is as t2h_codec_decode reads it through its pointer: Q8_0 rows of dense_shapes' sizes (a
        codebook of any number of rows) and fp32 vectors.  Other weights run operator by operator, where each operator
        takes or refuses them."""
        for name, shape in dense_shapes(self.cfg).items():
            t = self.w.get(name)
            if not isinstance(t, torch.Tensor) or not t.is_cuda or not t.is_contiguous():
                return False
            if len(shape) == 1:
                if t.dtype != torch.float32 or t.shape != shape or t.data_ptr() % 16:
                    return False
                continue
            rows = t.shape[0] if name.startswith("cb") and t.dim() == 2 else shape[0]
            if t.dtype != torch.uint8 or t.shape != (rows, -(-shape[1] // 32) * kernels.Q8_0_BYTES) or t.data_ptr() % 2:
                return False
        return True

    def _lay_out(self) -> list[torch.Tensor]:
        """t2h_codec_decode's operands in its order."""
        cfg, w = self.cfg, self.w
        bias = w["proj0.b"]
        for c in range(1, cfg.codebooks):
            bias = bias + w[f"proj{c}.b"]
        plan = [w[f"cb{c}"] for c in range(cfg.codebooks)]
        plan += [conv_fragments([w[f"proj{c}.w"] for c in range(cfg.codebooks)], cfg.codebook_dim, 1), bias]
        plan += [conv_fragments([w["fc2.w"]], cfg.latent, 1), w["fc2.b"]]
        plan += [conv_fragments([w["conv1.w"]], cfg.hidden, 7), w["conv1.b"], w["b0.alpha"]]
        ch, blocks, units = cfg.channels, len(cfg.strides), len(DILATIONS)
        for i in range(blocks):
            ch //= 2
            plan += [w[f"b{i}.convt.w"], w[f"b{i}.convt.b"], w[f"b{i}.r0.a1"]]
            for j in range(units):
                p = f"b{i}.r{j}."
                if j + 1 < units:
                    after = f"b{i}.r{j + 1}.a1"
                else:
                    after = f"b{i + 1}.alpha" if i + 1 < blocks else "final.alpha"
                plan += [conv_fragments([w[p + "c1.w"]], ch, 7), w[p + "c1.b"], w[p + "a2"],
                         conv_fragments([w[p + "c2.w"]], ch, 1), w[p + "c2.b"], w[after]]
        return plan + [conv_fragments([w["conv2.w"]], ch, 7), w["conv2.b"]]

    def _workspace_bytes(self, frames: int) -> int:
        """Bytes t2h_codec_decode needs (0: more frames than it takes)."""
        return int(_lib.lib().t2h_codec_decode_workspace_bytes(ctypes.addressof(self._dims), frames))

    def _decode_fused(self, codes: torch.Tensor, nbytes: int, stages: list | None) -> torch.Tensor:
        cfg, t = self.cfg, int(codes.shape[1])
        codes = codes[:cfg.codebooks].contiguous()
        space = torch.empty(nbytes, dtype=torch.uint8, device=self.device)
        out = torch.empty(out_len(cfg, t), dtype=torch.float32, device=self.device)
        operands = (ctypes.c_void_p * len(self._plan))(*[x.data_ptr() for x in self._plan])
        rows = (ctypes.c_uint32 * cfg.codebooks)(*[x.shape[0] for x in self._plan[:cfg.codebooks]])
        stage_ptrs = None
        if stages is not None:
            ch, length = cfg.channels, t
            new = [torch.empty(1, t, ch, dtype=torch.float32, device=self.device)]
            for s in cfg.strides:
                ch, length = ch // 2, length * s
                new += [torch.empty(1, length, ch, dtype=torch.float32, device=self.device)
                        for _ in range(1 + len(DILATIONS))]
            stages.extend(new)
            stage_arr = (ctypes.c_void_p * len(new))(*[x.data_ptr() for x in new])
            stage_ptrs = ctypes.addressof(stage_arr)
        call("t2h_codec_decode", ctypes.addressof(self._dims), ctypes.addressof(operands), len(self._plan),
             ctypes.addressof(rows), ptr(codes), t, kernels.SNAKE_EPS, ptr(out), stage_ptrs, ptr(space), nbytes,
             stream_handle())
        return out

    def _unit(self, x: torch.Tensor, p: str, dil: int) -> torch.Tensor:
        w = self.w
        r = kernels.snake(x, w[p + "a1"])
        r = kernels.conv1d_q8_0(r, w[p + "c1.w"], w[p + "c1.b"], 7, padding=3 * dil, dilation=dil)
        r = kernels.snake(r, w[p + "a2"])
        return kernels.conv1d_q8_0(r, w[p + "c2.w"], w[p + "c2.b"], 1, residual=x)

    def decode(self, codes: torch.Tensor, stages: list | None = None) -> torch.Tensor:
        """codes int64 [C, T] -> waveform fp32 [out_len(T)].  ``stages``: a list that receives the fp32
        channels-last activation [T, C] after conv1, after each block's transposed conv and after each of its
        residual units."""
        cfg, w = self.cfg, self.w
        codes = codes.to(device=self.device, dtype=torch.int64)
        t = int(codes.shape[1])
        if self._plan is not None and 0 < t < 1 << 31 and codes.dim() == 2 and codes.shape[0] >= cfg.codebooks:
            nbytes = self._workspace_bytes(t)
            if nbytes:
                return self._decode_fused(codes, nbytes, stages)
        acc = torch.zeros(t, cfg.latent, dtype=torch.float32, device=self.device)
        for c in range(cfg.codebooks):
            e = kernels.embedding_q8_0(w[f"cb{c}"], codes[c].contiguous(), cfg.codebook_dim)
            cols = kernels.im2col_1d(e.view(1, t, -1), 1)
            kernels.q8_0_linear(cols, w[f"proj{c}.w"], bias=w[f"proj{c}.b"], out=acc, out_dtype=torch.float32,
                                residual=acc)
        h = kernels.q8_0_linear(kernels.im2col_1d(acc.view(1, t, -1), 1), w["fc2.w"], bias=w["fc2.b"],
                                out_dtype=torch.float32)
        x = kernels.conv1d_q8_0(h.view(1, t, -1), w["conv1.w"], w["conv1.b"], 7, padding=3)
        if stages is not None:
            stages.append(x)
        ch = cfg.channels
        for i, s in enumerate(cfg.strides):
            x = kernels.snake(x, w[f"b{i}.alpha"])
            x = kernels.conv_transpose1d_q8_0(x, w[f"b{i}.convt.w"], w[f"b{i}.convt.b"], ch // 2, 2 * s, stride=s,
                                              padding=math.ceil(s / 2), output_padding=s % 2)
            if stages is not None:
                stages.append(x)
            for j, d in enumerate(DILATIONS):
                x = self._unit(x, f"b{i}.r{j}.", d)
                if stages is not None:
                    stages.append(x)
            ch //= 2
        x = kernels.snake(x, w["final.alpha"])
        return kernels.conv1d_q8_0(x, w["conv2.w"], w["conv2.b"], 7, padding=3).view(-1)
