"""Quantizers and the bf16 dequantizer where their last thread blocks are part full."""

from __future__ import annotations

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

BLOCK = {"q4_k": 256, "q6_k": 256, "q8_0": 32}


# blocks a launch: 1, one short of and one past a thread block's 8 (4 for Q6_K), and an odd number of them
@pytest.mark.parametrize("wtype", ["q4_k", "q6_k", "q8_0"])
@pytest.mark.parametrize("rows,blocks", [(1, 1), (1, 7), (3, 3), (1, 9), (5, 5), (33, 17)])
def test_quantize_tails_bit_exact(device, wtype, rows, blocks):
    import oracle
    from torch2vk_amd import kernels

    rng = np.random.default_rng(rows * 100 + blocks)
    x = (rng.standard_normal((rows, blocks * BLOCK[wtype])) * 0.02).astype(np.float32)
    x[0, :32] = np.abs(x[0, :32])  # a sub-block without negative values, one constant and one of zeros
    x[-1, -16:] = 0.0
    x[-1, :16] = 0.5
    got = kernels.quantize(torch.from_numpy(x).to(device), wtype).cpu().numpy()
    assert np.array_equal(got, getattr(oracle, f"quantize_{wtype}")(x))


# rows past a 256-row tile, and fewer; Q8_0 blocks past a thread block's 256
@pytest.mark.parametrize("wtype,rows,k", [("q4_k", 3, 256), ("q4_k", 257, 512), ("q6_k", 300, 256), ("q8_0", 5, 64),
                                          ("q8_0", 257, 192), ("q8_0", 64, 256)])
def test_dequantize_bf16_tails(device, wtype, rows, k):
    """The fp32 dequantizer's values rounded once (within one bf16 step for the K types, whose fp32 products round in a
    different order), and nothing written past the last row."""
    from torch2vk_amd import _lib, kernels

    g = torch.Generator(device=device)
    g.manual_seed(rows)
    w = kernels.quantize(torch.randn(rows, k, generator=g, device=device) * 0.05, wtype)
    buf = torch.full((rows + 1, k), 3.0, dtype=torch.bfloat16, device=device)
    kernels.dequantize_bf16(w, wtype, k, out=buf[:rows])
    f32 = torch.empty(rows, k, device=device)
    _lib.call("t2h_dequantize", kernels.WTYPES[wtype], _lib.ptr(w), rows, k, _lib.ptr(f32), _lib.stream_handle())
    diff = (buf[:rows].float() - f32.to(torch.bfloat16).float()).abs()
    assert (diff <= (0.0 if wtype == "q8_0" else 2.0 ** -7) * f32.abs()).all()
    assert (buf[rows] == 3.0).all()
