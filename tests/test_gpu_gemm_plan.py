"""The prefill GEMM below 4096 rows by gemm_plan (K parts, weights dequantised first or in the loop) against the
one-pass kernel over packed rows: the same bf16 operands, another fp32 order where K is split."""

from __future__ import annotations

import pytest
import torch


@pytest.mark.parametrize("wtype", ["q4_k", "q6_k", "q8_0", "bf16"])
@pytest.mark.parametrize("gated", [False, True])
def test_plan_stays_in_the_kernels_limits(wtype, gated):
    """Every part has at least two stages of K, splits stay in two rounds of blocks, and only packed rows are
    dequantised."""
    from torch2vk_amd import kernels

    for m in (0, 1, 9, 128, 129, 520, 1024, 1901, 4095):
        for n in (1, 7, 896, 4096, 12288, 151936):
            for k in (64, 256, 896, 4096, 12288):
                splits, dequant = kernels.gemm_plan(m, n, k, wtype, gated)
                tiles = -(-m // 128) * -(-n * (2 if gated else 1) // 256)
                assert splits == 1 or (splits <= min(16, k // 128) and tiles * splits <= 512)
                assert not (dequant and wtype == "bf16")
                assert kernels.gemm_plan(m, n, k, wtype, gated, False)[1] is False


# each route past gemm_tile's tiles: in the loop and dequantised, one pass and split, ragged rows and columns
@pytest.mark.gpu
@pytest.mark.parametrize("wtype,m,n,k,gated,want", [
    ("q4_k", 33, 4096, 6144, False, (16, False)), ("q4_k", 1037, 4099, 4096, False, None),
    ("q4_k", 1900, 6000, 2048, True, (1, True)), ("q6_k", 735, 4096, 4096, False, (2, True)),
    ("q6_k", 2049, 2050, 6144, False, (3, True)), ("q6_k", 300, 1030, 8192, True, None),
    ("q8_0", 548, 4096, 4096, False, (3, False)), ("q8_0", 3000, 4100, 2048, False, (1, True)),
    ("bf16", 548, 4096, 4096, False, (3, False))])
def test_planned_gemm_equals_one_pass(device, wtype, m, n, k, gated, want):
    from torch2vk_amd import kernels

    plan = kernels.gemm_plan(m, n, k, wtype, gated)
    print(f"{wtype} M={m} N={n} K={k} gated={gated} plan={plan}", flush=True)
    assert kernels.gemm_tile(m, 2 * n if gated else n, k, gated) is None and plan == (want or plan)
    g = torch.Generator(device=device)
    g.manual_seed(m + n)
    x = torch.randn(m, k, generator=g, device=device).to(torch.bfloat16)

    def weights():
        d = torch.randn(n, k, generator=g, device=device) * 0.05
        return d.to(torch.bfloat16) if wtype == "bf16" else kernels.quantize(d, wtype)

    w, w_up = weights(), weights()
    def bound(a):  # two fp32 sums of the same k products, in any order: (k + 8) 2^-24 of their magnitudes each
        dense = (a if wtype == "bf16" else kernels.dequantize_bf16(a, wtype, k)).double()
        return 2 * (k + 8) * 2.0 ** -24 * (x.double().abs() @ dense.abs().T)

    if gated:
        got, one = kernels.gemm_swiglu(x, w, w_up, wtype), kernels.gemm_swiglu(x, w, w_up, wtype, splits=1)
        if plan[0] == 1:
            assert torch.equal(got, one)
        else:  # silu's slope is below 1.1, its value below its argument's; then one bf16 rounding each
            gate, up = (kernels.gemm(x, a, wtype, out_dtype=torch.float32, splits=1).double().abs() for a in (w, w_up))
            allowed = 1.1 * bound(w) * (up + bound(w_up)) + gate * bound(w_up)
            assert ((got.double() - one.double()).abs() <= 2.0 ** -7 * one.double().abs() + allowed).all()
        return
    bound = bound(w)
    res = torch.randn(m, n, generator=g, device=device)
    one = kernels.gemm(x, w, wtype, out_dtype=torch.float32, splits=1)
    got = kernels.gemm(x, w, wtype, out_dtype=torch.float32)
    summed = kernels.gemm(x, w, wtype, out=res.clone(), residual=res)
    half = kernels.gemm(x, w, wtype)
    if plan[0] == 1:
        assert torch.equal(got, one) and torch.equal(half, one.to(torch.bfloat16))
    assert ((got - one).double().abs() <= bound).all()
    assert torch.equal(half, got.to(torch.bfloat16))
    assert ((summed.double() - res.double() - one.double()).abs() <= bound + 2.0 ** -23 * (res.abs() + one.abs())).all()
    if wtype == "q8_0":
        bias = torch.randn(n, generator=g, device=device)
        y = kernels.q8_0_linear(x, w, bias=bias, act="gelu", out_dtype=torch.float32)
        ref = kernels.q8_0_linear(x, w, bias=bias, act="gelu", out_dtype=torch.float32, splits=1)
        # gelu's slope is below 1.13; its own fp32 roundings are those of values a few units apart
        assert ((y - ref).double().abs() <= 1.13 * bound + 2.0 ** -21 * (one.abs() + bias.abs())).all()


@pytest.mark.gpu
def test_planned_linear_keeps_unaligned_rows(device):
    """Q8_0 rows that start at any even address: not dequantised first (that needs 16 bytes), the same result."""
    from torch2vk_amd import kernels

    g = torch.Generator(device=device)
    g.manual_seed(5)
    m, n, k = 3000, 4100, 2048
    assert kernels.gemm_plan(m, n, k, "q8_0") == (1, True)
    x = torch.randn(m, k, generator=g, device=device).to(torch.bfloat16)
    w = kernels.quantize(torch.randn(n, k, generator=g, device=device) * 0.05, "q8_0")
    buf = torch.empty(w.numel() + 16, dtype=torch.uint8, device=device)
    odd = buf[2:2 + w.numel()].view(n, -1)
    odd.copy_(w)
    assert torch.equal(kernels.q8_0_linear(x, odd), kernels.q8_0_linear(x, w))


def _room_cases(kernels, device):
    """(name, calls of one planned GEMM each into its own output, one-pass output or None where K is not split)."""
    g = torch.Generator(device=device)
    g.manual_seed(6)

    def weights(n, k, wtype):
        return kernels.quantize(torch.randn(n, k, generator=g, device=device) * 0.05, wtype)

    def x(m, k):
        return torch.randn(m, k, generator=g, device=device).to(torch.bfloat16)

    m, n, k = 3000, 4100, 2048
    assert kernels.gemm_plan(m, n, k, "q8_0") == (1, True)
    x0, w0, y0 = x(m, k), weights(n, k, "q8_0"), torch.empty(m, n, device=device)
    yield "linear", lambda splits=None: kernels.q8_0_linear(x0, w0, out=y0, out_dtype=torch.float32, splits=splits)
    yield "gemm", lambda splits=None: kernels.gemm(x0, w0, "q8_0", out=y0, out_dtype=torch.float32, splits=splits)
    m, n, k = 1900, 6000, 2048
    assert kernels.gemm_plan(m, n, k, "q4_k", True) == (1, True)
    x1, w1, w2 = x(m, k), weights(n, k, "q4_k"), weights(n, k, "q4_k")
    y1 = torch.empty(m, n, dtype=torch.bfloat16, device=device)
    yield "swiglu", lambda splits=None: kernels.gemm_swiglu(x1, w1, w2, "q4_k", out=y1, splits=splits)
    m, n, k = 735, 4096, 4096
    assert kernels.gemm_plan(m, n, k, "q6_k") == (2, True)
    x3, w3, y3 = x(m, k), weights(n, k, "q6_k"), torch.empty(m, n, device=device)
    yield "split", lambda splits=None: kernels.gemm(x3, w3, "q6_k", out=y3, out_dtype=torch.float32, splits=splits)


@pytest.mark.gpu
def test_no_room_for_dequantised_rows(device, monkeypatch):
    """A GEMM whose dequantised rows find no room multiplies the packed rows: the same bits."""
    from torch2vk_amd import kernels

    def no_room(*args, **kwargs):
        raise torch.OutOfMemoryError("no room")

    for name, call in _room_cases(kernels, device):
        want = call().clone()
        with monkeypatch.context() as m:
            m.setattr(kernels, "dequantize_bf16", no_room)
            assert torch.equal(call(), want), name


@pytest.mark.gpu
@pytest.mark.parametrize("captured", [False, True])
def test_no_room_for_any_scratch(device, captured):
    """With no memory left for a scratch of its size a planned GEMM takes none: one pass over packed rows, eagerly
    and inside a graph that is replayed."""
    from torch2vk_amd import kernels

    total = torch.cuda.mem_get_info()[1]
    cases = list(_room_cases(kernels, device))
    wants = [call(splits=1).clone() for _, call in cases]  # compiled, and what one pass gives
    torch.cuda.synchronize()
    for (name, call), want in zip(cases, wants):
        planned = call().clone()
        assert name != "split" or not torch.equal(planned, want)
        out = call()
        torch.cuda.empty_cache()
        filled = []
        try:
            torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + (4 << 20)) / total)
            with pytest.raises(torch.OutOfMemoryError):
                while len(filled) < 1000:
                    filled.append(torch.empty(4 << 20, dtype=torch.uint8, device=device))
            torch.cuda.reset_peak_memory_stats()
            before = torch.cuda.memory_allocated()
            if captured:
                graph = torch.cuda.CUDAGraph()
                with torch.cuda.graph(graph):
                    call()
            else:
                call()
        finally:
            torch.cuda.set_per_process_memory_fraction(1.0)
        assert torch.cuda.max_memory_allocated() - before < 4 << 20, name
        for _ in range(3 if captured else 0):
            out.zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, want), name
        assert torch.equal(out, want), name


def test_plan_below_the_dequantising_rows(monkeypatch):
    """DEQUANT_FIRST_ROWS is the one limit between the rules, wherever it is set."""
    from torch2vk_amd import kernels

    n, k = 12288, 4096
    planned = {m: kernels.gemm_plan(m, n, k, "q4_k") for m in (300, 4095, 6000)}
    assert kernels._gemm_plan(4095, n, k, "q4_k", None) == planned[4095]
    assert kernels._gemm_plan(4096, n, k, "q4_k", None) == (1, True)
    monkeypatch.setattr(kernels, "DEQUANT_FIRST_ROWS", 256)
    assert kernels._planned(255) and not kernels._planned(256)
    assert planned[300] != (1, True)
    assert kernels._gemm_plan(300, n, k, "q4_k", None) == (kernels.gemm_splits(300, n, k), kernels.gemm_splits(300, n, k) == 1)
    monkeypatch.setattr(kernels, "DEQUANT_FIRST_ROWS", 8192)
    assert kernels._gemm_plan(6000, n, k, "q4_k", None) == planned[6000]
    assert kernels._gemm_plan(8192, n, k, "q4_k", None) == (1, True)
    monkeypatch.setattr(kernels, "DEQUANT_FIRST_ROWS", 0)
    assert kernels._gemm_plan(300, n, k, "q4_k", None) == (planned[300][0], False)
    assert kernels._gemm_plan(6000, n, k, "q4_k", None) == (kernels.gemm_splits(6000, n, k), False)


def test_tiles_leave_long_chains_to_split_k():
    """Few blocks of 64 x 64 or 128 x 64 over a long K are slower than splits over the idle CUs (up to 1.5 times)."""
    from torch2vk_amd import kernels

    for m, n_cols, k in ((118, 2 * 2688, 6144), (350, 2 * 1024, 5120), (69, 2 * 4035, 4096), (92, 2 * 4608, 3328),
                         (27, 2 * 2048, 1792), (42, 2 * 2048, 2048)):
        assert kernels.gemm_tile(m, n_cols, k, True) is None, (m, n_cols, k)
    assert kernels.gemm_tile(128, 2 * 3072, 1024, True) == 2 and kernels.gemm_tile(115, 2 * 6144, 2048, True) == 3
    assert kernels.gemm_tile(64, 2048, 4096) == 0 and kernels.gemm_tile(520, 896, 3584) == 1
