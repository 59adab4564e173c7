"""The GEMVs over several tokens (one launch) against the same tokens one call at a time: the same bits."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", [2, 5, 8, 19])
@pytest.mark.parametrize("wtype,k,n", [("q4_k", 256, 48), ("q4_k", 1024, 3072), ("q4_k", 4096, 1024), ("q4_k", 8192, 96),
                                       ("q4_k", 12288, 512), ("q6_k", 1024, 1028), ("q6_k", 6144, 40),
                                       ("q8_0", 512, 36), ("q8_0", 4096, 130)])
def test_matvec_rows_equal_single_calls(device, wtype, m, k, n):
    from torch2vk_amd import kernels

    fn = kernels.q4k_matvec if wtype == "q4_k" else lambda *a, **kw: kernels.qx_matvec(*a, wtype, **kw)
    g = torch.Generator(device=device)
    g.manual_seed(m * k + n)
    x = torch.randn(m, k, generator=g, device=device).to(torch.bfloat16)
    w = kernels.quantize(torch.randn(n, k, generator=g, device=device) * 0.05, wtype)
    res = torch.randn(m, n, generator=g, device=device)
    for out_dtype, residual in ((torch.float32, None), (torch.bfloat16, None), (torch.float32, res)):
        got = fn(x, w, out_dtype=out_dtype, residual=residual)
        one = torch.stack([fn(x[i], w, out_dtype=out_dtype, residual=None if residual is None else residual[i])
                           for i in range(m)])
        assert torch.equal(got, one)
