"""The audio codec's kernels against the float64 oracle at the edges of their tiles."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle
from oracle import omnivoice as O

pytestmark = pytest.mark.gpu


# 31 useful rows a tile at kernel 2 stride: one row, a whole tile, one past it; channels below, at and past an LDS
# stage of 32; 7 column tiles (k 7, rows of G reaching 6 back); sizes of the per-output kernel (k 9; k 40 stride 1)
@pytest.mark.parametrize("length,ci,co,k,stride,pad,opad", [
    (1, 64, 8, 16, 8, 4, 0), (31, 32, 16, 8, 4, 2, 0), (32, 36, 40, 4, 2, 1, 0), (95, 65, 24, 6, 3, 2, 1),
    (40, 48, 20, 10, 5, 3, 1), (33, 30, 33, 7, 1, 3, 0), (64, 32, 3, 2, 2, 0, 1), (20, 16, 9, 9, 3, 0, 2),
    (50, 8, 4, 40, 1, 0, 0), (12, 40, 70, 1, 1, 0, 0), (9, 12, 5, 3, 7, 2, 6)])
@pytest.mark.parametrize("layout", ["rows", "channel_major"])
def test_conv_transpose1d_tiles_match_oracle(device, length, ci, co, k, stride, pad, opad, layout):
    from torch2vk_amd import kernels

    rng = np.random.default_rng(length + 7 * k)
    kk = co * k
    w = np.zeros((ci, (kk + 31) // 32 * 32), np.float32)
    w[:, :kk] = rng.standard_normal((ci, kk)) * 0.05
    packed = kernels.quantize(torch.from_numpy(w).to(device), "q8_0")
    dense = oracle.dequant_q8_0(packed.cpu().numpy(), w.shape[1])[:, :kk]
    bias = rng.standard_normal(co).astype(np.float32)
    x = torch.from_numpy(rng.standard_normal((2, length, ci)).astype(np.float32)).to(device)
    xd = x if layout == "rows" else x.transpose(1, 2).contiguous().transpose(1, 2)
    y = kernels.conv_transpose1d_q8_0(xd, packed, torch.from_numpy(bias).to(device), co, k, stride=stride, padding=pad,
                                      output_padding=opad).cpu().numpy()
    ref = O.conv_transpose1d_ref(x.cpu().numpy().transpose(0, 2, 1), dense, bias, k, stride, pad, opad)
    ref = ref.transpose(0, 2, 1)
    assert y.shape == ref.shape
    # fp32 sums of ci ceil(k / stride) products: (n + 2) 2^-24 of the sum of magnitudes bounds each output
    n = ci * -(-k // stride)
    mag = O.conv_transpose1d_ref(np.abs(x.cpu().numpy()).transpose(0, 2, 1), np.abs(dense), np.abs(bias), k, stride,
                                 pad, opad).transpose(0, 2, 1)
    assert (np.abs(y - ref) <= (n + 2) * 2.0 ** -24 * mag).all()
