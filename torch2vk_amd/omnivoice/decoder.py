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
from functools import reduce
from operator import attrgetter, itemgetter, or_

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


_dtype, _is_cuda, _size = attrgetter("dtype"), attrgetter("is_cuda"), torch.Tensor.size


class _Operands:
    """What t2h_codec_decode reads through its pointers for parts ``part`` .. ``part + parts - 1`` of a decode: the names
    of dense_shapes from index ``first``, their dtypes and their packed sizes."""

    def __init__(self, cfg: AudioDecoderConfig, part: int, parts: int) -> None:
        def at(q: int) -> int:  # where part q's operands start; a part also reads the alpha that follows it
            return 0 if q == 0 else 3 * cfg.codebooks + 4 + 21 * (q - 1)

        every = list(dense_shapes(cfg).items())
        self.part, self.parts, self.first = part, parts, at(part)
        shapes = every[self.first:at(part + parts) + 1 if part + parts < len(cfg.strides) + 2 else len(every)]
        self.last = self.first + len(shapes)
        self.tensors = itemgetter(*(name for name, _ in shapes))
        self.dtypes = [torch.float32 if len(s) == 1 else torch.uint8 for _, s in shapes]
        self.sizes = [s if len(s) == 1 else (s[0], -(-s[1] // 32) * kernels.Q8_0_BYTES) for _, s in shapes]
        self.tables = [i for i, (name, _) in enumerate(shapes) if name.startswith("cb")]  # of any number of rows
        self.vectors = itemgetter(*(i for i, (_, s) in enumerate(shapes) if len(s) == 1))

    def pointers(self, w: dict[str, torch.Tensor]) -> tuple[list[int], list[int]] | None:
        """(pointers, rows of the codebooks), or None where a weight is not as the chain reads it.  Looked at on every
        call (about 0.4 us a weight): entries of ``w`` can be replaced, resized or cast at any time."""
        try:
            ts = self.tensors(w)
        except KeyError:
            return None
        if not all(issubclass(t, torch.Tensor) for t in set(map(type, ts))) or list(map(_dtype, ts)) != self.dtypes:
            return None
        sizes = list(map(_size, ts))
        rows = []
        for i in self.tables:
            if len(sizes[i]) != 2:
                return None
            rows.append(sizes[i][0])
            sizes[i] = (self.sizes[i][0], sizes[i][1])
        if sizes != self.sizes or not all(map(_is_cuda, ts)) or not all(map(torch.Tensor.is_contiguous, ts)):
            return None
        ptrs = list(map(torch.Tensor.data_ptr, ts))
        if reduce(or_, ptrs) & 1 or reduce(or_, self.vectors(ptrs)) & 15 or 0 in ptrs:
            return None
        return ptrs, rows


class OmniVoiceAudioDecoder:
    """``w`` holds the packed weights; a decode reads them as they are when it is called.  Where they have the configured
    shapes it is one chain of about 40 launches (t2h_codec_decode); other shapes, and channel counts that chain is not
    built for, run operator by operator."""

    def __init__(self, cfg: AudioDecoderConfig, dense: dict[str, np.ndarray], device) -> None:
        self.cfg = cfg
        self.device = torch.device(device)
        self.w = {n: (quantize_rows(a, self.device) if a.ndim == 2 else torch.from_numpy(a).to(self.device))
                  for n, a in dense.items()}
        blocks = len(cfg.strides)
        self._dims = (ctypes.c_uint32 * (6 + blocks))(cfg.codebooks, cfg.codebook_dim, cfg.latent, cfg.hidden,
                                                      cfg.channels, blocks, *cfg.strides)
        fused = cfg.codebook_dim % 32 == 0 and cfg.latent % 64 == 0 and cfg.hidden % 64 == 0 and \
            self._workspace_bytes(1) > 0
        # in two calls: the host looks at the later blocks' weights while the GPU runs the first part
        self._plan = [_Operands(cfg, 0, 2), _Operands(cfg, 2, blocks)] if fused else None

    def _workspace_bytes(self, frames: int) -> int:
        """Bytes t2h_codec_decode needs (0: more frames than it takes)."""
        return int(_lib.lib().t2h_codec_decode_workspace_bytes(ctypes.addressof(self._dims), frames))

    def _decode_fused(self, codes: torch.Tensor, nbytes: int, stages: list | None) -> torch.Tensor | None:
        """The decode as t2h_codec_decode's chain, or None where a weight does not fit it."""
        cfg, t = self.cfg, int(codes.shape[1])
        found = self._plan[0].pointers(self.w)
        if found is None:
            return None
        n = self._plan[-1].last
        operands, rows = (ctypes.c_void_p * n)(), (ctypes.c_uint32 * cfg.codebooks)(*found[1])
        codes = codes[:cfg.codebooks].contiguous()
        space = torch.empty(nbytes, dtype=torch.uint8, device=self.device)
        out = torch.empty(out_len(cfg, t), dtype=torch.float32, device=self.device)
        new, stage_ptrs = [], None
        if stages is not None:
            ch, length = cfg.channels, t
            new = [torch.empty(1, t, ch, dtype=torch.float32, device=self.device)]
            for s in cfg.strides:
                ch, length = ch // 2, length * s
                new += [torch.empty(1, length, ch, dtype=torch.float32, device=self.device)
                        for _ in range(1 + len(DILATIONS))]
            stage_arr = (ctypes.c_void_p * len(new))(*[x.data_ptr() for x in new])
            stage_ptrs = ctypes.addressof(stage_arr)
        for group in self._plan:
            found = found or group.pointers(self.w)
            if found is None:
                return None  # what is enqueued writes only this call's own buffers
            operands[group.first:group.last] = found[0]
            found = None
            call("t2h_codec_decode", ctypes.addressof(self._dims), group.part, group.parts, ctypes.addressof(operands), n,
                 ctypes.addressof(rows), ptr(codes), t, kernels.SNAKE_EPS, ptr(out), stage_ptrs, ptr(space), nbytes,
                 stream_handle())
        if stages is not None:
            stages.extend(new)
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
            out = self._decode_fused(codes, nbytes, stages) if nbytes else None
            if out is not None:
                return out
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
