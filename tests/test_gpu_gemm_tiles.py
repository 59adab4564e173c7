"""The small-tile GEMM (t2h_gemm_tiles) against the one-pass kernel: the same products, another fp32 order."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


def _call(tile, wtype, x, w, w_up, out, n, w_k, bias=None, act=0, residual=None):
    from torch2vk_amd import kernels
    from torch2vk_amd._lib import call, ptr, stream_handle

    m, k = x.shape
    call("t2h_gemm_tiles", kernels.WTYPES[wtype], ptr(x), ptr(w), ptr(w_up), ptr(bias), act, ptr(out),
         0 if out.dtype == torch.float32 else 1, ptr(residual), m, k, n, w_k, tile, stream_handle())
    return out


# rows at, below and past a tile (32, 64, 128), one row; columns that are no multiple of 4 (single stores), of a tile, or
# less than one; K of half a stage, one, an odd number of them, fewer than the K groups, and more than the ring
@pytest.mark.parametrize("tile", [0, 1, 2, 3])
@pytest.mark.parametrize("wtype,m,k,n", [
    ("q8_0", 1, 64, 7), ("q8_0", 33, 192, 129), ("q8_0", 128, 1088, 64), ("q8_0", 65, 4096, 30), ("q4_k", 32, 256, 96),
    ("q4_k", 127, 2048, 68), ("q6_k", 64, 256, 33), ("q6_k", 129, 2304, 132), ("bf16", 31, 128, 100),
    ("bf16", 200, 1600, 65)])
def test_gemm_tiles_equal_one_pass(device, tile, wtype, m, k, n):
    from torch2vk_amd import kernels

    print(f"tile {tile} {wtype} M={m} K={k} N={n}", flush=True)
    g = torch.Generator(device=device)
    g.manual_seed(m + k + n)
    x = torch.randn(m, k, generator=g, device=device).to(torch.bfloat16)

    def weights():
        d = torch.randn(n, k, generator=g, device=device) * 0.05
        return d.to(torch.bfloat16) if wtype == "bf16" else kernels.quantize(d, wtype)

    w, w_up = weights(), weights()
    dense = [(a if wtype == "bf16" else kernels.dequantize_bf16(a, wtype, k)).double() for a in (w, w_up)]
    # two fp32 sums of the same k products, in any order: (k + 8) 2^-24 of the sum of magnitudes each
    bound = [2 * (k + 8) * 2.0 ** -24 * (x.double().abs() @ d.abs().T) for d in dense]
    one = kernels.gemm(x, w, wtype, out_dtype=torch.float32, splits=1)
    got = _call(tile, wtype, x, w, None, torch.full((m, n), 7.0, device=device), n, k)
    assert ((got - one).double().abs() <= bound[0]).all()
    half = _call(tile, wtype, x, w, None, torch.empty(m, n, dtype=torch.bfloat16, device=device), n, k)
    assert torch.equal(half, got.to(torch.bfloat16))  # the same sums, rounded once
    # bias, GELU and an fp32 residual in place
    bias, res = torch.randn(n, generator=g, device=device), torch.randn(m, n, generator=g, device=device)
    r = res.clone()
    _call(tile, wtype, x, w, None, r, n, k, bias=bias, act=1, residual=r)
    want = torch.nn.functional.gelu(got.double() + bias.double()) + res.double()
    # gelu's slope is below 1.13, its erf within 1.5e-7 (times |v| / 2); three fp32 roundings of the result's terms
    v = (got + bias).double().abs()
    assert ((r.double() - want).abs() <= 1.13 * 2.0 ** -23 * v + 1e-6 * v + 2.0 ** -22 * (v + res.double().abs())).all()
    if tile >= 2:
        s = _call(tile, wtype, x, w, w_up, torch.empty(m, n, dtype=torch.bfloat16, device=device), n, k).double()
        gate, up = got.double(), _call(tile, wtype, x, w_up, None, torch.empty(m, n, device=device), n, k).double()
        want = torch.nn.functional.silu(gate) * up  # the same sums; fp32 exp2 and reciprocal, then one bf16 rounding
        assert ((s - want).abs() <= 2.0 ** -8 * want.abs() + 1e-6 * up.abs()).all()


def test_gemm_tiles_short_weight_rows(device):
    """Q8_0 rows shorter than x's (padded) rows: the columns past them multiply zeros."""
    from torch2vk_amd import kernels

    g = torch.Generator(device=device)
    g.manual_seed(3)
    x = torch.randn(70, 320, generator=g, device=device).to(torch.bfloat16)
    for w_k in (32, 160, 288):
        w = kernels.quantize(torch.randn(66, w_k, generator=g, device=device) * 0.05, "q8_0")
        want = kernels.q8_0_linear(x, w, out_dtype=torch.float32, splits=1)
        for tile in range(4):
            got = _call(tile, "q8_0", x, w, None, torch.empty(70, 66, device=device), 66, w_k)
            assert (got - want).abs().max().item() <= 2 * (w_k + 8) * 2.0 ** -24 * 66, (w_k, tile)


def test_gemm_tile_rule(device):
    """The rule's tiles fit the chip and their K limit, and the gated form only gets whole 64-column groups."""
    from torch2vk_amd import kernels

    for m in (1, 9, 33, 128, 300, 520, 1024, 4095, 4096, 16384):
        for n in (7, 896, 1024, 4096, 6144, 24576):
            for k in (64, 896, 4096, 6144, 12288):
                for gated in (False, True):
                    t = kernels.gemm_tile(m, n, k, gated)
                    if t is None:
                        continue
                    rows, cols, k_max = kernels.GEMM_TILES[t]
                    blocks = -(-m // rows) * -(-n // cols)
                    assert m < 4096 and k <= k_max and (blocks <= 256 or (t == 3 and blocks <= 512))
                    assert not gated or cols >= 64
