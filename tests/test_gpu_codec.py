"""The audio codec's kernels against the float64 oracle at the edges of their tiles."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle
from oracle import omnivoice as O
from oracle import reference as R
from tests.conftest import assert_close

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


def _check_stages(dec, cfg, dense, frames):
    """Every stage of a decode against the float64 oracle over the stage's own input, and the waveform of the run that
    keeps no stages against the run that does (the same arithmetic, so the same bits)."""
    from torch2vk_amd.omnivoice.decoder import out_len

    deq = {}
    for n, a in dense.items():
        if a.ndim != 2:
            deq[n] = a.astype(np.float64)
            continue
        kp = (a.shape[1] + 31) // 32 * 32
        deq[n] = oracle.dequant_q8_0(dec.w[n].cpu().numpy(), kp)[:, :a.shape[1]].astype(np.float64)
        if not (n.startswith("cb") or n.endswith("convt.w")):
            deq[n] = R.bf16_round(deq[n].astype(np.float32)).astype(np.float64)
    bf = lambda a: R.bf16_round(np.asarray(a, np.float32)).astype(np.float64)  # noqa: E731
    codes = np.random.default_rng(8).integers(-1, cfg.vocab + 1, (cfg.codebooks, frames)).astype(np.int64)
    stages = []
    y = dec.decode(torch.from_numpy(codes), stages=stages)
    assert torch.equal(y, dec.decode(torch.from_numpy(codes)))
    y = y.cpu().numpy()
    assert y.shape == (out_len(cfg, frames),)
    got = [a.cpu().numpy().astype(np.float64)[0].T[None] for a in stages]
    # ids outside the table embed as zeros: one zero row after the table
    ref_deq = {n: (np.concatenate([a, np.zeros((1, a.shape[1]))]) if n.startswith("cb") else a) for n, a in deq.items()}
    ids = np.where((codes >= 0) & (codes < cfg.vocab), codes, cfg.vocab)
    checks = [("front", got[0], O.audio_decode_front_ref(cfg, ref_deq, ids, bf))]
    k = 1
    for i in range(len(cfg.strides)):
        checks.append((f"block {i} upsample", got[k], O.audio_decode_upsample_ref(cfg, deq, got[k - 1], i)))
        k += 1
        for j, d in enumerate((1, 3, 9)):
            checks.append((f"block {i} unit {j}", got[k],
                           O.audio_decode_unit_ref(deq, got[k - 1], f"b{i}.r{j}.", d, bf)))
            k += 1
    checks.append(("final", y, O.audio_decode_final_ref(deq, got[-1], bf)))
    # a stage holds up to two convolutions (the front three products): an fp32 sum that lands on the other side of
    # a bf16 boundary moves one staged input by 2^-8 of itself, so the stage by 2^-8 of one product of its sums
    for what, a, b in checks:
        assert a.shape == b.shape, what
        assert_close(a, b, max_abs=2.0 ** -8 * float(np.abs(b).max()), min_cos=0.99999, what=what)


# channels down to 8 (padded column tiles and channel steps), one frame, a frame count past a row tile,
# channel slabs split over 1, 2 and 4 waves (wide first layers, few rows), more rows than one block takes
@pytest.mark.parametrize("books,dim,latent,hidden,channels,strides,frames", [
    (3, 32, 64, 64, 64, (3, 2, 2), 1), (1, 64, 192, 128, 256, (2, 3), 33), (2, 32, 128, 320, 512, (8, 5, 4, 2, 3), 3),
    (4, 32, 64, 64, 96, (5, 7), 70)])
def test_codec_decode_stages_match_oracle(device, books, dim, latent, hidden, channels, strides, frames):
    """Every stage of the fused decode against the float64 oracle."""
    from torch2vk_amd.omnivoice.decoder import AudioDecoderConfig, OmniVoiceAudioDecoder, synthetic_dense

    cfg = AudioDecoderConfig(codebooks=books, vocab=16, codebook_dim=dim, latent=latent, hidden=hidden,
                             channels=channels, strides=strides)
    dense = synthetic_dense(cfg, seed=frames)
    dec = OmniVoiceAudioDecoder(cfg, dense, device)
    assert dec._plan is not None
    _check_stages(dec, cfg, dense, frames)


# latent, hidden and channel sizes that the chain is not built for, more codebooks than it takes, and sizes that it takes
@pytest.mark.parametrize("fields,fused", [({"latent": 96}, False), ({"hidden": 96}, False), ({"codebooks": 33}, False),
                                          ({"channels": 48, "strides": (4, 3)}, False), ({"strides": (8, 5)}, True)])
def test_codec_operators_match_oracle(device, fields, fused):
    """The decode operator by operator, which runs wherever the chain does not: the same stages, the same oracle."""
    dec, cfg, dense, _ = _small_codec(device, 41, **fields)
    assert (dec._plan is not None) == fused
    dec._plan = None
    _check_stages(dec, cfg, dense, 11)


# a 4-column group of an epilogue with one alpha whose argument passes the polynomial's range: the whole group takes
# the general form, each column its own value
@pytest.mark.parametrize("column", range(4))
def test_codec_epilogue_large_arguments(device, column):
    from torch2vk_amd.omnivoice.decoder import OmniVoiceAudioDecoder

    _, cfg, dense, _ = _small_codec(device, 51)
    for name in ("b0.alpha", "b0.r0.a2", "b0.r1.a1", "b1.r2.a2", "final.alpha"):
        dense[name][column::8] = 1e30  # sin^2 / alpha vanishes beside the value
    dense["b1.r0.a2"][column::8] = 3e9
    _check_stages(OmniVoiceAudioDecoder(cfg, dense, device), cfg, dense, 13)


def _small_codec(device, seed, **fields):
    """A decoder whose shapes the fused chain takes, its dense weights, and codes of one id past its vocab."""
    from torch2vk_amd.omnivoice.decoder import AudioDecoderConfig, OmniVoiceAudioDecoder, synthetic_dense

    cfg = AudioDecoderConfig(**{**dict(codebooks=2, vocab=16, codebook_dim=32, latent=64, hidden=64, channels=64,
                                       strides=(3, 2)), **fields})
    dense = synthetic_dense(cfg, seed=seed)
    codes = torch.from_numpy(np.random.default_rng(seed).integers(0, cfg.vocab + 1, (cfg.codebooks, 9)))
    codes[0, 0] = cfg.vocab
    return OmniVoiceAudioDecoder(cfg, dense, device), cfg, dense, codes


@pytest.mark.parametrize("extra", [1, -5])
def test_codec_tables_have_their_own_row_counts(device, extra):
    """A codebook with more rows than cfg.vocab (a mask row) is looked up by its own row count, and ids past a shorter
    one embed as zeros: the same samples as with a table padded with zeros to the ids used."""
    from torch2vk_amd.omnivoice.decoder import OmniVoiceAudioDecoder

    dec, cfg, dense, codes = _small_codec(device, 11)
    rng = np.random.default_rng(12)
    rows = cfg.vocab + extra
    tables = {n: (rng.standard_normal((rows, cfg.codebook_dim)) * 0.2).astype(np.float32)
              for n in dense if n.startswith("cb")}
    full = {n: np.concatenate([t, np.zeros((max(0, cfg.vocab + 1 - rows), cfg.codebook_dim), np.float32)])
            for n, t in tables.items()}
    got = OmniVoiceAudioDecoder(cfg, {**dense, **tables}, device).decode(codes)
    want = OmniVoiceAudioDecoder(type(cfg)(**{**vars(cfg), "vocab": cfg.vocab + 1}), {**dense, **full}, device)
    assert torch.equal(got, want.decode(codes))
    if extra > 0:
        assert not torch.equal(got, dec.decode(codes))


# what the operators refuse of each kind of weight is refused by a decode that would run as one chain, too
@pytest.mark.parametrize("name,change,error", [
    ("b0.r0.a1", "half", TypeError), ("proj0.b", "double", TypeError), ("conv2.b", "half", TypeError),
    ("b1.alpha", "longer", ValueError), ("b0.convt.b", "shorter", ValueError), ("fc2.b", "longer", ValueError),
    ("cb1", "wider", ValueError), ("b0.r1.c1.w", "rows", ValueError), ("proj1.w", "wider", ValueError),
    ("b1.convt.w", "rows", ValueError), ("conv2.w", "wider", ValueError)])
def test_codec_refuses_weights_that_do_not_fit(device, name, change, error):
    from torch2vk_amd.omnivoice.decoder import OmniVoiceAudioDecoder

    _, cfg, dense, codes = _small_codec(device, 21)
    a = dense[name]
    a = {"half": lambda: a.astype(np.float16), "double": lambda: a.astype(np.float64),
         "longer": lambda: np.concatenate([a, a]), "shorter": lambda: a[:a.shape[0] // 2].copy(),
         "wider": lambda: np.concatenate([a] * 5, axis=1), "rows": lambda: np.concatenate([a, a])}[change]()
    dec = OmniVoiceAudioDecoder(cfg, {**dense, name: a}, device)
    with pytest.raises(error):
        dec.decode(codes)


# 32 codebooks: more matrices than one layout launch takes; channels 48 and 24: steps and tiles that end inside
@pytest.mark.parametrize("fields", [{}, {"codebooks": 32}, {"channels": 96, "hidden": 320}])
def test_codec_decode_reads_the_weights_of_the_call(device, fields):
    """Weights written in place or replaced between decodes are the ones that the next decode uses: the samples of a
    decoder made with them."""
    a, _, _, codes = _small_codec(device, 31, **fields)
    b, _, _, _ = _small_codec(device, 32, **fields)
    assert not torch.equal(a.decode(codes), b.decode(codes))
    kept = {n: t.clone() for n, t in a.w.items()}
    for i, (n, t) in enumerate(b.w.items()):
        if i % 2:
            a.w[n].copy_(t)
        else:
            a.w[n] = t.clone()
    assert torch.equal(a.decode(codes), b.decode(codes))
    for n in a.w:  # one at a time: each of them counts
        before, a.w[n] = a.w[n], kept[n]
        changed = a.decode(codes)
        assert not torch.equal(changed, b.decode(codes)), n
        a.w[n] = before
    assert torch.equal(a.decode(codes), b.decode(codes))
    a.w["b1.r2.a2"] = a.w["b1.r2.a2"].half()
    with pytest.raises(TypeError):
        a.decode(codes)


def test_snake_matches_64_bits(device):
    """x + sin(alpha x)^2 / (alpha + eps) at the bounds stated for sin^2 (1.2e-7, and 2.8e-7 of its value), alpha a
    power of two so that its argument is exact.  eps leaves a divisor of 2^-24 alpha, which lifts sin^2 as far above x
    as 24 bits allow; x's own rounding is what is left at large arguments (2^-18 of sin^2 at 2^30)."""
    from torch2vk_amd import kernels

    rng = np.random.default_rng(3)
    near = np.arange(1, 4000) * (np.pi / 2)                    # where the reduced argument is smallest
    y = np.concatenate([2.0 ** rng.uniform(-20, 30, 20000), near, rng.integers(1, 2 ** 29, 4000) * (np.pi / 2),
                        [2.0 ** 30, 2.0 ** 30 * (1 + 2.0 ** -23), 1e10, 1e20, 3e38]]).astype(np.float32)
    y = np.concatenate([y, -y, [0.0]]).astype(np.float32)
    for alpha in (1.0, 2.0 ** 12, 2.0 ** -6):
        with np.errstate(over="ignore"):
            x = (y / np.float32(alpha)).astype(np.float32)
        ok = np.isfinite(x)
        x, args = x[ok], y[ok].astype(np.float64)
        step = 2.0 ** -24 * alpha
        got = kernels.snake(torch.from_numpy(x).to(device)[:, None].contiguous(),
                            torch.full((1,), alpha, device=device), eps=-(alpha - step)).cpu().numpy()[:, 0]
        s2 = np.sin(args) ** 2
        want = x.astype(np.float64) + s2 / step
        tol = np.minimum(1.2e-7, 2.8e-7 * s2) / step + 2.0 ** -23 * (np.abs(x.astype(np.float64)) + s2 / step)
        large = np.abs(args) > 2.0 ** 30
        tol[large] += 2e-7 / step
        err = np.abs(got.astype(np.float64) - want)
        assert (err <= tol).all(), (alpha, args[np.argmax(err - tol)], float((err / tol).max()))
    bad = torch.tensor([[float("nan")], [float("inf")], [-float("inf")], [1.0]], device=device)
    out = kernels.snake(bad, torch.ones(1, device=device)).cpu().numpy()[:, 0]
    assert np.isnan(out[:3]).all() and np.isfinite(out[3])
