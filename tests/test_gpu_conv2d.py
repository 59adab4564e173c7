"""conv2d without a patch matrix against torch's conv2d in 64 bits on the operands the kernels multiply (bf16 inputs,
d * q weights rounded to bf16).  Sizes sit at the edges of tiles: rows and columns past the last whole tile, a K that
ends inside a 64-deep stage, every tile, patches over the border on every side, and the launch's own choice.

Tolerance per value: one bf16 rounding of the result (2^-9 of it; twice that where the result sits at a power of two),
plus K fp32 roundings of the accumulated magnitudes (K 2^-24 sum |x| |w|), plus 2e-6 for the GELU's erf (1.5e-7) and
its slope of at most 1.13."""

from __future__ import annotations

import pytest
import torch

from torch2vk_amd import kernels

pytestmark = pytest.mark.gpu


def _rows(g: torch.Generator, n: int, k: int) -> torch.Tensor:
    w = torch.randn(n, -(-k // 32) * 32, generator=g) / k ** 0.5
    w[:, k:] = 0.0
    return kernels.quantize(w.cuda(), "q8_0")


def _weights(packed: torch.Tensor, k: int) -> torch.Tensor:
    blocks = packed.cpu().view(packed.shape[0], -1, 34)
    d = blocks[..., :2].contiguous().view(torch.float16).float()
    q = blocks[..., 2:].contiguous().view(torch.int8).float()
    return (d * q).view(packed.shape[0], -1)[:, :k].to(torch.bfloat16).double()


def _check(out, x, w, bias, stride, pad, act):
    conv = torch.nn.functional.conv2d
    want = conv(x, w, bias, stride, pad)
    size = conv(x.abs(), w.abs(), bias.abs(), stride, pad)
    if act:
        want = want * 0.5 * (1.0 + torch.erf(want * 0.5 ** 0.5))
    tol = want.abs() * 2.0 ** -8 + size * (w[0].numel() + 1) * 2.0 ** -24 * 1.13 + 2e-6
    err = (out.cpu().double().permute(0, 3, 1, 2) - want).abs()
    assert out.shape[1:3] == want.shape[2:] and bool((err <= tol).all()), float((err - tol).max())


@pytest.mark.parametrize("shape,kernel,stride,pad,tile,act", [
    ((1, 5, 7, 64), (3, 3), 2, 1, -1, "gelu"),       # 12 rows of a 64-row tile
    ((2, 13, 11, 72), (3, 3), 2, 1, 0, "gelu"),      # K 648: taps end inside stages, the last stage has 8 values
    ((3, 17, 9, 480), (3, 3), 2, 1, 1, "gelu"),      # 135 rows: one past a 128-row tile
    ((2, 16, 13, 480), (3, 3), 1, 1, 2, None),
    ((2, 33, 25, 136), (3, 3), 2, 1, 3, "gelu"),     # 442 rows of 256-row tiles
    ((1, 9, 8, 64), (3, 1), 1, 0, -1, None),         # one column of taps
    ((1, 6, 30, 64), (2, 12), 3, 5, -1, "gelu"),     # 24 taps, padding wider than the stride
    ((1, 3, 3, 64), (3, 3), 1, 0, 3, None),          # one output pixel
])
@pytest.mark.parametrize("n", [36, 288])
def test_conv2d_matches_reference(shape, kernel, stride, pad, tile, act, n):
    g = torch.Generator().manual_seed(7)
    c, taps = shape[3], kernel[0] * kernel[1]
    x = torch.randn(shape, generator=g).to(torch.bfloat16)
    packed = _rows(g, n, c * taps)
    bias = torch.randn(n, generator=g)
    out = kernels.conv2d(x.cuda(), kernels.conv2d_rows(packed, c, kernel), bias.cuda(), kernel, stride, pad, act=act,
                         tile=tile)
    w = _weights(packed, c * taps).view(n, c, *kernel)
    _check(out, x.double().permute(0, 3, 1, 2), w, bias.double(), stride, pad, act)


@pytest.mark.parametrize("shape,kernel,stride,pad,n", [
    ((1, 1, 4, 5), (3, 3), 2, 1, 8), ((2, 1, 33, 17), (3, 3), 2, 1, 72), ((1, 1, 128, 100), (3, 3), 2, 1, 480),
    ((3, 1, 19, 23), (4, 4), 1, 2, 64), ((1, 1, 40, 3), (5, 1), 3, 0, 136),
])
def test_conv2d_1ch_matches_reference(shape, kernel, stride, pad, n):
    g = torch.Generator().manual_seed(8)
    taps = kernel[0] * kernel[1]
    x = torch.randn(shape, generator=g)
    packed = _rows(g, n, taps)
    bias = torch.randn(n, generator=g)
    out = kernels.conv2d_1ch(x.cuda(), packed, bias.cuda(), kernel, stride, pad, act="gelu")
    w = _weights(packed, taps).view(n, 1, *kernel)
    _check(out, x.to(torch.bfloat16).double(), w, bias.double(), stride, pad, "gelu")


# a whole stage of K and one that ends inside it; channels past one block's 512; channel counts off 8 and 32
@pytest.mark.parametrize("n,c,taps", [(3, 64, 9), (5, 480, 9), (2, 1096, 24), (4, 36, 6), (3, 517, 3), (1, 8, 1)])
def test_conv2d_rows_are_the_weights_tap_major(n, c, taps):
    packed = _rows(torch.Generator().manual_seed(n + c), n, c * taps)
    rows = kernels.conv2d_rows(packed, c, (1, taps)).cpu()
    want = _weights(packed, c * taps).view(n, c, taps).transpose(1, 2).reshape(n, -1)
    assert rows.shape == (n, -(-c * taps // 64) * 64)
    assert torch.equal(rows[:, :c * taps].double(), want) and not rows[:, c * taps:].any()


def test_encoder_front_end_reads_the_weights_of_the_call():
    """Convolution weights written in place or replaced after an encoder was made are the ones that it uses."""
    from torch2vk_amd.qwen3_asr.config import AudioEncoderConfig
    from torch2vk_amd.qwen3_asr.encoder import Qwen3AudioEncoder, quantize_audio_weights, synthetic_audio_dense

    cfg = AudioEncoderConfig(d_model=128, layers=1, heads=2, ffn=256, output_dim=128, conv_channels=64)
    a, b = (Qwen3AudioEncoder(quantize_audio_weights(synthetic_audio_dense(cfg, seed=s), cfg, torch.device("cuda")))
            for s in (1, 2))
    g = torch.Generator().manual_seed(3)
    mel = torch.randn(2, 1, cfg.mel_bins, 100, generator=g).cuda()
    tokens = 100
    for _ in range(3):
        tokens = (tokens - 1) // 2 + 1
    pos = torch.randn(2, tokens, cfg.d_model, generator=g).cuda()
    want = b.frontend(mel, pos)
    assert not torch.equal(a.frontend(mel, pos), want)
    for name, t in b.weights.packed.items():
        if "conv" in name and name.endswith("2.weight"):
            a.weights.packed[name].copy_(t)
        elif "conv" in name:
            a.weights.packed[name] = t.clone()
    for name, t in b.weights.vectors.items():
        if "conv" in name:
            a.weights.vectors[name].copy_(t)
    assert torch.equal(a.frontend(mel, pos), want)
