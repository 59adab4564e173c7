// The audio codec's decoder (run_audio_decode, src/models/quantized_omnivoice/dispatch/audio_decode.py:60-760)
// as one enqueue of fused launches, activations channels-last [T, C]:
//
//   codes -> bf16 embedding rows of all codebooks side by side        (one gather)
//   project_out of every codebook, summed: one product over C D       (conv, 1 tap)
//   fc2, conv1 (7 taps)                                                (conv)
//   per block: transposed conv, then 3 residual units of 2 launches   (conv 7 taps dilated, conv 1 tap)
//   conv2 (7 taps, one channel)                                       (conv)
//
// Every snake runs once, in the epilogue of the launch that produces its argument: a convolution's input is
// bf16(snake(x)), so the epilogue writes it as such beside the fp32 value the residual (or the transposed
// convolution, which stays fp32) needs.  Rounding is where the operator-by-operator path has it: weights and
// convolution inputs to bf16, everything else fp32.  Measured at 75 frames (1024 channels, strides 8, 5, 4, 2, 3):
// 1806 us as about 200 launches of embedding, im2col, GEMM, snake and transposed convolution, bound by their
// host work, by im2col's writes and by 256-wide GEMM tiles over 32 to 512 columns; 447 us as these 39, of
// which the transposed convolutions take 161.
//
// Convolution weights are laid out once by the caller as bf16 fragments of v_mfma_f32_32x32x16_bf16,
// [tap][channel step of 16][column tile of 32][lane][8]: lane l holds column l % 32, channels 8 (l / 32) + 0..7,
// so a wave loads a fragment as one contiguous KB (channels padded with zeros to 32, columns to 64).
#include "codec.h"

namespace t2h {

typedef __bf16 cd_bf16x8_t __attribute__((ext_vector_type(8)));
typedef float cd_f32x16_t __attribute__((ext_vector_type(16)));

constexpr uint32_t CD_MAX_DIL = 9;  // the residual units' dilations are 1, 3 and 9
constexpr uint32_t CD_TAPS = 7;

struct CdConvArgs {
    const uint16_t* x;    // bf16 [len, cin], cin % 8 == 0
    const uint16_t* w;    // fragments
    const float* bias;    // [n]
    const float* res;     // fp32 [len, n] added last (may be `raw`), or null
    float* raw;           // fp32 [len, n] of the result, or null
    uint16_t* bf;         // bf16 [len, n] of the result, snaked when alpha is given, or null
    float* snaked;        // fp32 [len, n] of snake(result), or null
    const float* alpha;   // [n] or null
    float eps;
    uint32_t len, cin, n;
    uint32_t dil;         // TAPS 7: tap j reads row t + (j - 3) dil
    uint32_t ksteps;      // 16-channel steps per tap in w
    uint32_t ntiles;      // 32-column tiles in w
};

// A block of 4 waves: 32 (4 / WK) rows x 32 NJ columns, WK waves sharing a row tile and splitting the channels.
// Rows (with the taps' halo) go through LDS in slabs of SC channels a wave, loaded once for all taps, the next
// slab in flight meanwhile; LDS rows are 16 bytes past a power of two, so a fragment read of 16 rows hits 16
// distinct 4-bank groups.  Weight fragments come straight from L2 into registers, each reloaded for the next
// slab as soon as its MFMA has issued.  The codec's layers are small (0.1 to 2.2 GFLOP): what bounds them is
// latency and filling the chip, hence the split of the channels within a block where rows are few, with the
// partial tiles summed in LDS.
template <int TAPS, int SC, int WK, int NJ>
__global__ __launch_bounds__(256) void codec_conv_kernel(const CdConvArgs a) {
    constexpr int WM = 4 / WK, BM = 32 * WM;
    constexpr int LROWS = BM + (TAPS - 1) * (int)CD_MAX_DIL;
    constexpr int RS = SC + 8;              // LDS row, bf16
    constexpr int KQ = SC / 16;             // channel steps per slab
    constexpr int FR = TAPS * KQ;           // fragments per slab and column tile
    constexpr int CPR = WK * SC / 8;        // 16-B chunks per row and slab
    constexpr int APT = (LROWS * CPR + 255) / 256;
    constexpr int SLAB = WK * LROWS * RS;   // bf16 per buffer
    constexpr int TS = 32 * NJ + 8;         // row of the result tile in LDS: the half-waves' rows, 4 apart, use
                                            // distinct banks
    constexpr int TILE_BYTES = 4 * 32 * TS * 4;
    constexpr int LDS_BYTES = 2 * SLAB * 2 > TILE_BYTES ? 2 * SLAB * 2 : TILE_BYTES;
    __shared__ __align__(16) uint8_t lds[LDS_BYTES];
    uint16_t* ls = reinterpret_cast<uint16_t*>(lds);

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / WK, wk = wave % WK;
    const int r32 = lane & 31, h = lane >> 5;
    const uint32_t nt0 = blockIdx.y * NJ;
    const int64_t t0 = (int64_t)blockIdx.x * BM;
    const int pad = (TAPS / 2) * (int)a.dil;
    const int rows = BM + 2 * pad;
    const uint32_t slabs = (a.ksteps * 16 + WK * SC - 1) / (WK * SC);

    uint4 ra[APT];
    auto load_rows = [&](uint32_t s) {
#pragma unroll
        for (int i = 0; i < APT; ++i) {
            const int idx = tid + 256 * i, row = idx / CPR;
            const uint32_t c = s * (WK * SC) + 8u * (uint32_t)(idx % CPR);
            const int64_t t = t0 + row - pad;
            ra[i] = make_uint4(0u, 0u, 0u, 0u);
            if (row < rows && t >= 0 && t < (int64_t)a.len && c < a.cin)
                ra[i] = load_u4(a.x + (size_t)t * a.cin + c);
        }
    };
    auto store_rows = [&](int buf) {
#pragma unroll
        for (int i = 0; i < APT; ++i) {
            const int idx = tid + 256 * i, row = idx / CPR, j = idx % CPR;
            if (row < rows)
                *reinterpret_cast<uint4*>(&ls[buf * SLAB + ((j / (SC / 8)) * LROWS + row) * RS + 8 * (j % (SC / 8))]) =
                    ra[i];
        }
    };
    // fragment f (tap f / KQ, step f % KQ) of slab s; a split past the last channels re-reads the last step
    // (its rows are zero)
    auto load_w = [&](uint32_t s, int f, int nj) {
        const uint32_t ks = min((s * WK + wk) * KQ + (uint32_t)(f % KQ), a.ksteps - 1);
        const size_t tile = ((size_t)(f / KQ) * a.ksteps + ks) * a.ntiles + nt0 + nj;
        return *reinterpret_cast<const cd_bf16x8_t*>(a.w + (tile * 64 + lane) * 8);
    };

    cd_f32x16_t acc[NJ];
#pragma unroll
    for (int nj = 0; nj < NJ; ++nj)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[nj][e] = 0.0f;
    cd_bf16x8_t wf[FR][NJ];
    load_rows(0);
#pragma unroll
    for (int f = 0; f < FR; ++f)
#pragma unroll
        for (int nj = 0; nj < NJ; ++nj) wf[f][nj] = load_w(0, f, nj);
    store_rows(0);
    __syncthreads();
    for (uint32_t s = 0; s < slabs; ++s) {
        const uint32_t sn = min(s + 1, slabs - 1);
        if (s + 1 < slabs) load_rows(s + 1);
        const uint16_t* base = ls + (s & 1) * SLAB + (wk * LROWS + wm * 32 + r32) * RS + 8 * h;
#pragma unroll
        for (int f = 0; f < FR; ++f) {
            const cd_bf16x8_t fa =
                *reinterpret_cast<const cd_bf16x8_t*>(base + (f / KQ) * (int)a.dil * RS + 16 * (f % KQ));
#pragma unroll
            for (int nj = 0; nj < NJ; ++nj) {
                acc[nj] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa, wf[f][nj], acc[nj], 0, 0, 0);
                wf[f][nj] = load_w(sn, f, nj);
            }
        }
        if (s + 1 < slabs) store_rows((s + 1) & 1);
        __syncthreads();
    }

    // The tile goes through LDS (the channel splits' partial tiles are summed there), then each thread finishes 4
    // columns of a row at a time: + bias, + residual (the next row's in flight), snake, and the forms the next
    // launches read, as 16- and 8-byte stores.  With a guarded residual load and the library's sinf per element
    // instead, the one-tap convolution of 12000 x 128 took 26 us, and takes 9.
    float* tile = reinterpret_cast<float*>(lds);
#pragma unroll
    for (int nj = 0; nj < NJ; ++nj)
#pragma unroll
        for (int e = 0; e < 16; ++e)
            tile[(wave * 32 + 8 * (e >> 2) + 4 * h + (e & 3)) * TS + 32 * nj + r32] = acc[nj][e];
    __syncthreads();
    constexpr int GROUPS = 8 * NJ;  // 4-column groups per row; 256 is a multiple, so a thread keeps its columns
    const int cg = tid % GROUPS;
    const uint32_t col = nt0 * 32 + 4 * cg;
    const uint32_t left = a.len - (uint32_t)t0;  // rows of the tile inside the activation
    if (a.n % 4 != 0) {
        // a row that is not whole 16-byte groups (the waveform's one channel): only the fp32 result
        for (uint32_t r = tid / GROUPS; r < min(left, (uint32_t)BM); r += 256 / GROUPS)
            for (uint32_t j = 0; j < 4 && col + j < a.n; ++j) {
                float v = a.bias[col + j];
#pragma unroll
                for (int p = 0; p < WK; ++p) v += tile[((r / 32 * WK + p) * 32 + r % 32) * TS + 4 * cg + j];
                a.raw[((uint32_t)t0 + r) * a.n + col + j] = v;
            }
        return;
    }
    if (col >= a.n) return;
    const float4 bias = *reinterpret_cast<const float4*>(a.bias + col);
    float4 alpha = make_float4(0.f, 0.f, 0.f, 0.f);
    if (a.alpha) alpha = *reinterpret_cast<const float4*>(a.alpha + col);
    const float al[4] = {alpha.x, alpha.y, alpha.z, alpha.w};
    float inv[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) inv[j] = 1.0f / (al[j] + a.eps);
    const uint32_t rows_here = min(left, (uint32_t)BM);
    uint32_t r = tid / GROUPS;
    // (32-bit element offsets: an activation has fewer than 2^31)
    float4 res = make_float4(0.f, 0.f, 0.f, 0.f);
    if (a.res && r < rows_here) res = *reinterpret_cast<const float4*>(a.res + ((uint32_t)t0 + r) * a.n + col);
#pragma unroll 1
    for (; r < rows_here; r += 256 / GROUPS) {
        const uint32_t at = ((uint32_t)t0 + r) * a.n + col;
        float4 next = res;  // the next row's residual is in flight while this one is finished
        if (a.res && r + 256 / GROUPS < rows_here)
            next = *reinterpret_cast<const float4*>(a.res + at + (256 / GROUPS) * a.n);
        float o[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int p = 0; p < WK; ++p) {
            const float4 v = *reinterpret_cast<const float4*>(&tile[((r / 32 * WK + p) * 32 + r % 32) * TS + 4 * cg]);
            o[0] += v.x;
            o[1] += v.y;
            o[2] += v.z;
            o[3] += v.w;
        }
        o[0] = res.x + (o[0] + bias.x);
        o[1] = res.y + (o[1] + bias.y);
        o[2] = res.z + (o[2] + bias.z);
        o[3] = res.w + (o[3] + bias.w);
        res = next;
        if (a.raw) *reinterpret_cast<float4*>(a.raw + at) = make_float4(o[0], o[1], o[2], o[3]);
        if (a.alpha) {
            bool large = false;
            float sv[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float y = al[j] * o[j];
                large |= !(fabsf(y) <= SIN_SQUARED_MAX);
                sv[j] = o[j] + inv[j] * sin_squared(y);
            }
            if (large) {  // one rolled copy of the general form (large arguments, infinities and NaN)
#pragma unroll 1
                for (int j = 0; j < 4; ++j) {
                    const float x = j < 2 ? (j == 0 ? o[0] : o[1]) : (j == 2 ? o[2] : o[3]);
                    const float xa = j < 2 ? (j == 0 ? al[0] : al[1]) : (j == 2 ? al[2] : al[3]);
                    const float y = snake_f32(x, xa, a.eps);
                    sv[0] = j == 0 ? y : sv[0];
                    sv[1] = j == 1 ? y : sv[1];
                    sv[2] = j == 2 ? y : sv[2];
                    sv[3] = j == 3 ? y : sv[3];
                }
            }
#pragma unroll
            for (int j = 0; j < 4; ++j) o[j] = sv[j];
        }
        if (a.bf) *reinterpret_cast<uint2*>(a.bf + at) = make_uint2(pack_bf16x2(o[0], o[1]), pack_bf16x2(o[2], o[3]));
        if (a.snaked) *reinterpret_cast<float4*>(a.snaked + at) = make_float4(o[0], o[1], o[2], o[3]);
    }
}

// Q8_0 rows [n, cin * taps] (element c taps + tap) -> fragments, channel steps kstep0 .. of `ksteps` per tap: thread
// (tap, step, column tile, lane) converts its 8 weights, zero past the last channel and column.
__global__ __launch_bounds__(256) void codec_fragments_kernel(const uint8_t* __restrict__ w, uint32_t n, uint32_t cin,
                                                              uint32_t taps, uint32_t steps, uint32_t ntiles,
                                                              uint32_t ksteps, uint32_t kstep0,
                                                              uint16_t* __restrict__ out) {
    const uint64_t idx = (uint64_t)blockIdx.x * 256 + threadIdx.x;
    if (idx >= (uint64_t)taps * steps * ntiles * 64) return;
    const uint32_t lane = (uint32_t)(idx % 64), tile = (uint32_t)(idx / 64 % ntiles);
    const uint32_t step = (uint32_t)(idx / 64 / ntiles % steps), tap = (uint32_t)(idx / 64 / ntiles / steps);
    const uint32_t col = tile * 32 + (lane & 31), c0 = step * 16 + 8 * (lane >> 5);
    const uint8_t* row = w + (size_t)col * ((cin * taps + 31) / 32 * 34);
    float v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        v[j] = 0.0f;
        if (col < n && c0 + j < cin) {
            const uint32_t e = (c0 + j) * taps + tap;
            const uint8_t* b = row + (size_t)(e / 32) * 34;
            v[j] = f16_bits_to_f32(load_u16(b)) * (float)(int8_t)b[2 + e % 32];
        }
    }
    *reinterpret_cast<uint4*>(out + ((((size_t)tap * ksteps + kstep0 + step) * ntiles + tile) * 64 + lane) * 8) =
        make_uint4(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]), pack_bf16x2(v[4], v[5]), pack_bf16x2(v[6], v[7]));
}

// codes -> bf16 [T, codebooks * dim]: codebook c's Q8_0 row of code [c, t] at columns c dim .. (an id outside that
// table gives zeros), rounded to bf16 as the project_out product reads it.  One thread per 8 values.
struct CdTables {
    const uint8_t* rows[32];
    uint32_t count[32];  // rows of each table
};
__global__ __launch_bounds__(256) void codec_embed_kernel(const CdTables tables, const int64_t* __restrict__ codes,
                                                          uint32_t books, uint32_t dim, uint32_t len,
                                                          uint16_t* __restrict__ out) {
    const uint32_t per = dim / 8;
    const uint64_t idx = (uint64_t)blockIdx.x * 256 + threadIdx.x;
    if (idx >= (uint64_t)len * books * per) return;
    const uint32_t j = (uint32_t)(idx % per), c = (uint32_t)(idx / per % books);
    const uint64_t t = idx / per / books;
    const int64_t id = codes[(uint64_t)c * len + t];
    uint4 o = make_uint4(0u, 0u, 0u, 0u);
    if (id >= 0 && id < (int64_t)tables.count[c]) {
        const uint8_t* p = tables.rows[c] + (size_t)id * ((dim + 31) / 32 * 34) + (size_t)(j / 4) * 34;
        const float d = f16_bits_to_f32(load_u16(p));
        const uint2 q = load_u2_ua(p + 2 + 8 * (j % 4));
        uint32_t w[2] = {q.x, q.y};
        uint32_t r[4];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            r[2 * i] = pack_bf16x2(d * (float)(int8_t)(w[i] & 0xffu), d * (float)(int8_t)((w[i] >> 8) & 0xffu));
            r[2 * i + 1] = pack_bf16x2(d * (float)(int8_t)((w[i] >> 16) & 0xffu), d * (float)(int8_t)(w[i] >> 24));
        }
        o = make_uint4(r[0], r[1], r[2], r[3]);
    }
    *reinterpret_cast<uint4*>(out + (size_t)t * books * dim + (size_t)c * dim + 8 * j) = o;
}

template <int TAPS, int SC, int WK, int NJ>
static void cd_launch(const CdConvArgs& a, hipStream_t s) {
    constexpr uint32_t BM = 32 * (4 / WK);
    const dim3 grid((a.len + BM - 1) / BM, (a.n + 32 * NJ - 1) / (32 * NJ));
    hipLaunchKernelGGL((codec_conv_kernel<TAPS, SC, WK, NJ>), grid, dim3(256), 0, s, a);
}

// The fewest waves per row tile (the most rows per weight fragment) that still gives about a block per CU, at
// most one per slab of channels; one column tile per block only where there is one, or too few blocks of two.
template <int TAPS, int SC>
static void cd_dispatch(const CdConvArgs& a, hipStream_t s) {
    const uint32_t slabs = (a.ksteps * 16 + SC - 1) / SC;
    auto blocks = [&](uint32_t wk, uint32_t nj) {
        const uint32_t bm = 32 * (4 / wk);
        return (uint64_t)((a.n + 32 * nj - 1) / (32 * nj)) * ((a.len + bm - 1) / bm);
    };
    uint32_t nj = a.n <= 32 ? 1 : 2, wk = 1;
    while (wk < 4 && 2 * wk <= slabs && blocks(wk, nj) < 192) wk *= 2;
    if (nj == 2 && blocks(wk, 2) < 96) nj = 1;
    switch (wk * 10 + nj) {
        case 11: cd_launch<TAPS, SC, 1, 1>(a, s); break;
        case 12: cd_launch<TAPS, SC, 1, 2>(a, s); break;
        case 21: cd_launch<TAPS, SC, 2, 1>(a, s); break;
        case 22: cd_launch<TAPS, SC, 2, 2>(a, s); break;
        case 41: cd_launch<TAPS, SC, 4, 1>(a, s); break;
        default: cd_launch<TAPS, SC, 4, 2>(a, s); break;
    }
}

static void cd_conv(const CdConvArgs& a, uint32_t taps, hipStream_t s) {
    if (taps == CD_TAPS) cd_dispatch<CD_TAPS, 32>(a, s);
    else if (a.ksteps >= 8) cd_dispatch<1, 128>(a, s);
    else cd_dispatch<1, 32>(a, s);
}

// dims: codebooks, codebook_dim, latent, hidden, channels, blocks, then the blocks' strides
struct CdDims {
    uint32_t books, dim, latent, hidden, channels, blocks;
    uint32_t strides[16];
    uint64_t len(uint32_t frames, uint32_t b) const {  // positions after b blocks
        uint64_t l = frames;
        for (uint32_t i = 0; i < b; ++i) l *= strides[i];
        return l;
    }
};

static int cd_dims(const uint32_t* d, CdDims& o) {
    o.books = d[0];
    o.dim = d[1];
    o.latent = d[2];
    o.hidden = d[3];
    o.channels = d[4];
    o.blocks = d[5];
    if (o.books == 0 || o.books > 32 || o.blocks == 0 || o.blocks > 16) return T2H_ERR_UNSUPPORTED;
    if (o.dim == 0 || o.latent == 0 || o.hidden == 0 || o.channels == 0) return T2H_ERR_SHAPE;
    if (o.channels > (1u << 20) || o.latent > (1u << 20) || o.hidden > (1u << 20) || o.dim > (1u << 20))
        return T2H_ERR_UNSUPPORTED;
    if (o.dim % 8 || o.latent % 8 || o.hidden % 8 || (o.channels >> o.blocks) % 8 ||
        (o.channels >> o.blocks) == 0 || (o.channels & ((1u << o.blocks) - 1)))
        return T2H_ERR_UNSUPPORTED;
    for (uint32_t i = 0; i < o.blocks; ++i) {
        o.strides[i] = d[6 + i];
        if (o.strides[i] < 2) return T2H_ERR_UNSUPPORTED;  // an output padding of stride % 2 needs stride > 1
        if (o.strides[i] > 1024) return T2H_ERR_UNSUPPORTED;
    }
    return T2H_OK;
}

// workspace: bf16 gathered rows, bf16 sums, bf16 hidden, then per position and channel of the widest point two
// fp32 and two bf16 activations
struct CdSpace {
    uint64_t gather, latent, hidden, act, total;  // byte sizes; act: elements of the widest activation
};
static int cd_space(const CdDims& d, uint32_t frames, CdSpace& s) {
    auto up = [](uint64_t v) { return (v + 255) / 256 * 256; };
    s.gather = up(2ull * frames * d.books * d.dim);
    s.latent = up(2ull * frames * d.latent);
    s.hidden = up(2ull * frames * d.hidden);
    s.act = (uint64_t)frames * d.channels;
    for (uint32_t b = 1; b <= d.blocks; ++b) {
        // 2^31 outputs a layer at most, and positions a row tile can index
        const uint64_t l = d.len(frames, b);
        if (l > 0x3fffffffull) return T2H_ERR_SHAPE;
        const uint64_t n = l * (d.channels >> b);
        s.act = n > s.act ? n : s.act;
    }
    if (s.act > 0x7fffffffull || (uint64_t)frames * d.books * d.dim > 0x7fffffffull) return T2H_ERR_SHAPE;
    s.act = up(s.act);
    s.total = s.gather + s.latent + s.hidden + s.act * (4 + 4 + 2 + 2);
    return T2H_OK;
}

}  // namespace t2h

using namespace t2h;

extern "C" int t2h_conv_fragments_q8_0(const void* w, uint32_t n, uint32_t cin, uint32_t taps, uint32_t ksteps,
                                       uint32_t kstep0, void* out, void* stream) {
    if (!w || !out) return T2H_ERR_NULL;
    if (n == 0 || cin == 0 || taps == 0) return T2H_ERR_SHAPE;
    if ((uint64_t)cin * taps > 0x7fffffffu || n > 0x7fffff00u) return T2H_ERR_SHAPE;
    const uint32_t steps = (cin + 31) / 32 * 2, ntiles = (n + 63) / 64 * 2;
    if (kstep0 > ksteps || steps > ksteps - kstep0) return T2H_ERR_ARG;
    if (reinterpret_cast<uintptr_t>(w) % 2 != 0 || reinterpret_cast<uintptr_t>(out) % 16 != 0) return T2H_ERR_ALIGN;
    const uint64_t threads = (uint64_t)taps * steps * ntiles * 64;
    if (threads / 256 >= 0x7fffffffu) return T2H_ERR_SHAPE;
    hipLaunchKernelGGL(codec_fragments_kernel, dim3((uint32_t)((threads + 255) / 256)), dim3(256), 0,
                       reinterpret_cast<hipStream_t>(stream), reinterpret_cast<const uint8_t*>(w), n, cin, taps, steps,
                       ntiles, ksteps, kstep0, reinterpret_cast<uint16_t*>(out));
    T2H_LAUNCH_CHECK();
    return T2H_OK;
}

extern "C" size_t t2h_codec_decode_workspace_bytes(const uint32_t* dims, uint32_t frames) {
    CdDims d;
    CdSpace s;
    if (!dims || frames == 0 || cd_dims(dims, d) != T2H_OK || cd_space(d, frames, s) != T2H_OK) return 0;
    return s.total;
}

extern "C" int t2h_codec_decode(const uint32_t* dims, const void* const* ptrs, uint32_t n_ptrs,
                                const uint32_t* table_rows, const int64_t* codes, uint32_t frames, float eps,
                                float* out, float* const* stages, void* workspace, size_t workspace_bytes,
                                void* stream) {
    if (!dims || !ptrs || !table_rows || !codes || !out || !workspace) return T2H_ERR_NULL;
    CdDims d;
    int st = cd_dims(dims, d);
    if (st) return st;
    if (n_ptrs != d.books + 6 + d.blocks * 21 + 3) return T2H_ERR_ARG;
    for (uint32_t i = 0; i < n_ptrs; ++i)
        if (!ptrs[i]) return T2H_ERR_NULL;
    if (frames == 0) return T2H_ERR_SHAPE;
    if (reinterpret_cast<uintptr_t>(workspace) % 256 != 0) return T2H_ERR_ALIGN;
    CdSpace sp;
    st = cd_space(d, frames, sp);
    if (st) return st;
    if (workspace_bytes < sp.total) return T2H_ERR_WORKSPACE;
    if (stages)
        for (uint32_t i = 0; i < 1 + 4 * d.blocks; ++i)
            if (!stages[i]) return T2H_ERR_NULL;
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    uint8_t* ws = reinterpret_cast<uint8_t*>(workspace);
    auto take = [&](uint64_t bytes) {
        uint8_t* p = ws;
        ws += bytes;
        return p;
    };
    uint16_t* gathered = reinterpret_cast<uint16_t*>(take(sp.gather));
    uint16_t* latent = reinterpret_cast<uint16_t*>(take(sp.latent));
    uint16_t* hidden = reinterpret_cast<uint16_t*>(take(sp.hidden));
    float* xs = reinterpret_cast<float*>(take(4 * sp.act));   // snaked input of the next transposed conv
    float* xr = reinterpret_cast<float*>(take(4 * sp.act));   // residual stream of a block
    uint16_t* s1 = reinterpret_cast<uint16_t*>(take(2 * sp.act));
    uint16_t* s2 = reinterpret_cast<uint16_t*>(take(2 * sp.act));

    const void* const* p = ptrs;
    auto f32 = [&]() { return reinterpret_cast<const float*>(*p++); };
    auto frag = [&]() { return reinterpret_cast<const uint16_t*>(*p++); };
    // one convolution: alpha null leaves the result as it is
    auto conv = [&](const uint16_t* x, const uint16_t* w, const float* bias, uint64_t len, uint32_t cin, uint32_t n,
                    uint32_t taps, uint32_t dil, const float* res, float* raw, uint16_t* bf, float* snaked,
                    const float* alpha) {
        CdConvArgs a = {};
        a.x = x;
        a.w = w;
        a.bias = bias;
        a.res = res;
        a.raw = raw;
        a.bf = bf;
        a.snaked = snaked;
        a.alpha = alpha;
        a.eps = eps;
        a.len = (uint32_t)len;
        a.cin = cin;
        a.n = n;
        a.dil = dil;
        a.ksteps = (cin + 31) / 32 * 2;
        a.ntiles = (n + 63) / 64 * 2;
        cd_conv(a, taps, s);
    };

    CdTables tables = {};
    for (uint32_t c = 0; c < d.books; ++c) {
        tables.rows[c] = reinterpret_cast<const uint8_t*>(*p++);
        tables.count[c] = table_rows[c];
    }
    const uint64_t work = (uint64_t)frames * d.books * (d.dim / 8);
    hipLaunchKernelGGL(codec_embed_kernel, dim3((uint32_t)((work + 255) / 256)), dim3(256), 0, s, tables, codes, d.books,
                       d.dim, frames, gathered);
    T2H_LAUNCH_CHECK();
    const uint16_t* w = frag();
    conv(gathered, w, f32(), frames, d.books * d.dim, d.latent, 1, 0, nullptr, nullptr, latent, nullptr, nullptr);
    w = frag();
    conv(latent, w, f32(), frames, d.latent, d.hidden, 1, 0, nullptr, nullptr, hidden, nullptr, nullptr);
    w = frag();
    const float* b1 = f32();
    const float* alpha = f32();  // block 0's
    conv(hidden, w, b1, frames, d.hidden, d.channels, CD_TAPS, 1, nullptr, stages ? stages[0] : nullptr, nullptr, xs,
         alpha);
    T2H_LAUNCH_CHECK();
    uint64_t len = frames;
    static const uint32_t dils[3] = {1, 3, 9};
    for (uint32_t b = 0; b < d.blocks; ++b) {
        const uint32_t ch = d.channels >> b, co = ch / 2, stride = d.strides[b];
        const void* wt = *p++;
        const float* bt = f32();
        float* x = stages ? stages[1 + 4 * b] : xr;
        const int64_t strides[3] = {(int64_t)(len * ch), 1, (int64_t)ch};
        const uint64_t lo = len * stride;
        const float* a1 = f32();
        st = conv_transpose1d_q8_0_launch(xs, strides, wt, bt, x, 1, ch, (uint32_t)len, co, 2 * stride, stride,
                                          (stride + 1) / 2, (uint32_t)lo, s1, a1, eps, stream);
        if (st) return st;
        len = lo;
        for (uint32_t u = 0; u < 3; ++u) {
            const uint16_t* w1 = frag();
            const float* bias1 = f32();
            const float* a2 = f32();
            const uint16_t* w2 = frag();
            const float* bias2 = f32();
            const float* next = f32();  // the next unit's, the next block's, or the final alpha
            conv(s1, w1, bias1, len, co, co, CD_TAPS, dils[u], nullptr, nullptr, s2, nullptr, a2);
            const bool last = u == 2, end = last && b + 1 == d.blocks;
            float* raw = stages ? stages[2 + 4 * b + u] : (last ? nullptr : xr);
            conv(s2, w2, bias2, len, co, co, 1, 0, x, raw, last && !end ? nullptr : s1, last && !end ? xs : nullptr,
                 next);
            x = raw;
            T2H_LAUNCH_CHECK();
        }
    }
    w = frag();
    conv(s1, w, f32(), len, d.channels >> d.blocks, 1, CD_TAPS, 1, nullptr, out, nullptr, nullptr, nullptr);
    T2H_LAUNCH_CHECK();
    return T2H_OK;
}
