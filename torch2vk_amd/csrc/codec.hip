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
// host work, by im2col's writes and by 256-wide GEMM tiles over 32 to 512 columns; 462 us as these 40 and two that
// lay the weights out (8 + 5 us), of which the transposed convolutions take 160.
//
// Convolution weights are read as bf16 fragments of v_mfma_f32_32x32x16_bf16, [tap][channel step of 16][column tile
// of 32][lane][8]: lane l holds column l % 32, channels 8 (l / 32) + 0..7, so a wave loads a fragment as one contiguous
// KB (channels padded with zeros to 32, columns to 64).  Each call lays them out from the packed rows into its workspace
// (codec_layout_kernel), so a weight written between calls, by whatever means, is the one that the next call uses.
#include "codec.h"
#include "gemm_formats.h"

#include <algorithm>

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

// Weight rows -> fragments, all matrices of a call in one launch (Q8_0 rows [n, cin taps], element c taps + tap; several
// matrices may lie side by side in one operand, each at its own channel steps).  A block converts 32 columns x 32
// channels x 7 taps, or x 256 channels of one tap: 32 channels of a row are `taps` whole Q8_0 blocks, so a thread
// converts one of a row's 7 or 8 consecutive blocks, every byte is read once, and the taps are picked apart in LDS.
constexpr uint32_t CD_LAYOUTS = 32;  // matrices per launch
struct CdLayout {
    const uint8_t* w;
    uint16_t* out;
    uint32_t n, cin, taps;
    uint32_t ksteps, kstep0;  // the operand's channel steps, and this matrix's first
};
struct CdLayouts {
    CdLayout m[CD_LAYOUTS];
    uint32_t first[64];  // first block of each matrix, then 2^32 - 1: one entry a lane
};
__host__ __device__ constexpr uint32_t cd_layout_groups(uint32_t taps) { return taps == 1 ? 8 : 1; }  // of 32 channels
__global__ __launch_bounds__(256) void codec_layout_kernel(const CdLayouts a) {
    constexpr uint32_t PITCH = 2 * 129;  // bf16 per LDS row of 8 blocks: the 32 rows of a read lie in distinct banks
    __shared__ uint32_t ls[32 * PITCH / 2];
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const uint32_t i = __builtin_amdgcn_readfirstlane(__popcll(__ballot(a.first[lane] <= blockIdx.x)) - 1);
    const uint32_t n = a.m[i].n, cin = a.m[i].cin, taps = a.m[i].taps, b = blockIdx.x - a.first[i];
    const uint32_t ntiles = (n + 63) / 64 * 2, tile = b % ntiles, groups = cd_layout_groups(taps);
    const uint32_t group0 = b / ntiles * groups, blocks = (cin * taps + 31) / 32;
    {
        const uint32_t row = tid / 8, k = tid % 8, col = tile * 32 + row, blk = group0 * taps + k;
        GemmQ80::Raw r = {};
        r.inside = col < n && k < groups * taps && blk < blocks;  // others: zeros
        if (r.inside) {
            const uint8_t* p = a.m[i].w + ((size_t)col * blocks + blk) * 34;
            r.d = load_u16(p);
            r.q0 = load_u4_ua(p + 2);
            r.q1 = load_u4_ua(p + 18);
        }
        uint32_t o[16];
        GemmQ80::convert(r, 0, 0, o);
#pragma unroll
        for (int j = 0; j < 16; ++j) ls[row * (PITCH / 2) + 16 * k + j] = o[j];
    }
    __syncthreads();
    const uint16_t* row = reinterpret_cast<const uint16_t*>(ls) + (lane & 31) * PITCH;
    for (uint32_t u = wave; u < 2 * taps * groups; u += 4) {
        const uint32_t step = u & 1, tap = taps == 1 ? 0 : u >> 1, local = taps == 1 ? u >> 1 : 0;
        if (32 * (group0 + local) >= cin) break;  // past the last step
        const uint32_t c = 32 * local + 16 * step + 8 * (lane >> 5);  // cin % 8 == 0: 8 channels are all inside or none
        const uint32_t keep = 32 * group0 + c < cin ? 0xffffffffu : 0u;
        uint32_t f[4];
#pragma unroll
        for (int j = 0; j < 4; ++j)
            f[j] = ((uint32_t)row[(c + 2 * j) * taps + tap] | (uint32_t)row[(c + 2 * j + 1) * taps + tap] << 16) & keep;
        const size_t at = ((size_t)tap * a.m[i].ksteps + a.m[i].kstep0 + 2 * (group0 + local) + step) * ntiles + tile;
        *reinterpret_cast<uint4*>(a.m[i].out + (at * 64 + lane) * 8) = make_uint4(f[0], f[1], f[2], f[3]);
    }
}

// codes -> bf16 [T, codebooks * dim]: codebook c's Q8_0 row of code [c, t] at columns c dim .. (an id outside that
// table gives zeros), rounded to bf16 as the project_out product reads it.  One thread per 8 values; `latent` threads
// more sum the codebooks' biases.
struct CdTables {
    const uint8_t* rows[32];
    uint32_t count[32];  // rows of each table
    const float* bias[32];
};
__global__ __launch_bounds__(256) void codec_embed_kernel(const CdTables tables, const int64_t* __restrict__ codes,
                                                          uint32_t books, uint32_t dim, uint32_t len, uint32_t latent,
                                                          uint16_t* __restrict__ out, float* __restrict__ bias) {
    const uint32_t per = dim / 8;
    const uint64_t idx = (uint64_t)blockIdx.x * 256 + threadIdx.x, gathers = (uint64_t)len * books * per;
    if (idx >= gathers) {
        const uint64_t i = idx - gathers;
        if (i >= latent) return;
        float v = tables.bias[0][i];
        for (uint32_t c = 1; c < books; ++c) v += tables.bias[c][i];
        bias[i] = v;
        return;
    }
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
// most one per slab of channels; one column tile per block only where there is one, or too few blocks of two.  Measured
// over the codec's 34 convolutions (us, this rule / the fastest of the six forms for each layer): 1 frame 160 / 143,
// 12: 171 / 152, 75: 281 / 251, 200: 447 / 423, 500: 901 / 855, 1500: 2534 / 2496.  What it leaves are narrow layers of
// few blocks, where one column tile a block and a split past one wave per slab are faster (600 rows of 512, 7 taps: 10.5
// in 152 blocks of two tiles, 9.5 in 304 of one; 12000 of 128: 11.7 against 9.6; 960 of 32: 5.5 against 4.2 over 4 waves).
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
    if (o.dim % 32 || o.latent % 8 || o.hidden % 8 || (o.channels >> o.blocks) % 8 ||
        (o.channels >> o.blocks) == 0 || (o.channels & ((1u << o.blocks) - 1)))
        return T2H_ERR_UNSUPPORTED;
    for (uint32_t i = 0; i < o.blocks; ++i) {
        o.strides[i] = d[6 + i];
        if (o.strides[i] < 2) return T2H_ERR_UNSUPPORTED;  // an output padding of stride % 2 needs stride > 1
        if (o.strides[i] > 1024) return T2H_ERR_UNSUPPORTED;
    }
    return T2H_OK;
}

// bf16 values of one operand's fragments
static uint64_t cd_fragments(uint32_t cin, uint32_t n, uint32_t taps) {
    return (uint64_t)taps * ((cin + 31) / 32 * 2) * ((n + 63) / 64 * 2) * 512;
}

// workspace: bf16 gathered rows, bf16 sums, bf16 hidden, then per position and channel of the widest point two
// fp32 and two bf16 activations, then the summed bias and the weights' fragments
struct CdSpace {
    uint64_t gather, latent, hidden, act, bias, total;  // byte sizes; act: elements of the widest activation
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
    // every activation of the chain has 32-bit element offsets
    const uint64_t front = frames * (uint64_t)std::max({d.books * d.dim, d.latent, d.hidden});
    if (s.act > 0x7fffffffull || front > 0x7fffffffull) return T2H_ERR_SHAPE;
    s.act = up(s.act);
    s.bias = up(4ull * d.latent);
    uint64_t frags = cd_fragments(d.books * d.dim, d.latent, 1) + cd_fragments(d.latent, d.hidden, 1) +
                     cd_fragments(d.hidden, d.channels, CD_TAPS) + cd_fragments(d.channels >> d.blocks, 1, CD_TAPS);
    for (uint32_t b = 1; b <= d.blocks; ++b)
        frags += 3 * (cd_fragments(d.channels >> b, d.channels >> b, CD_TAPS) +
                      cd_fragments(d.channels >> b, d.channels >> b, 1));
    if (frags > 1ull << 40) return T2H_ERR_SHAPE;  // (a layout block converts 1024 or more: 2^30 blocks at most)
    s.total = s.gather + s.latent + s.hidden + s.act * (4 + 4 + 2 + 2) + s.bias + 2 * frags;
    return T2H_OK;
}

}  // namespace t2h

using namespace t2h;

extern "C" size_t t2h_codec_decode_workspace_bytes(const uint32_t* dims, uint32_t frames) {
    CdDims d;
    CdSpace s;
    if (!dims || frames == 0 || cd_dims(dims, d) != T2H_OK || cd_space(d, frames, s) != T2H_OK) return 0;
    return s.total;
}

extern "C" int t2h_codec_decode(const uint32_t* dims, uint32_t part, uint32_t parts, const void* const* ptrs,
                                uint32_t n_ptrs, const uint32_t* table_rows, const int64_t* codes, uint32_t frames,
                                float eps, float* out, float* const* stages, void* workspace, size_t workspace_bytes,
                                void* stream) {
    if (!dims || !ptrs || !table_rows || !codes || !out || !workspace) return T2H_ERR_NULL;
    CdDims d;
    int st = cd_dims(dims, d);
    if (st) return st;
    if (part >= d.blocks + 2 || parts == 0 || parts > d.blocks + 2 - part) return T2H_ERR_ARG;
    const uint32_t end = part + parts;
    // the operands of part q start at at(q); the first of a block and of the last part is the snake of the part before
    auto at = [&](uint32_t q) { return q == 0 ? 0 : 3 * d.books + 4 + 21 * (q - 1); };
    const uint32_t n_all = at(d.blocks + 1) + 3;
    if (n_ptrs != n_all) return T2H_ERR_ARG;
    for (uint32_t i = at(part); i < (end < d.blocks + 2 ? at(end) + 1 : n_all); ++i)
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
    float* bias0 = reinterpret_cast<float*>(take(sp.bias));

    auto f32 = [&](uint32_t i) { return reinterpret_cast<const float*>(ptrs[i]); };
    // the fragments of this call's parts, and the launches that lay them out
    CdLayouts lay;
    uint32_t lay_count = 0, lay_blocks = 0;
    uint16_t* front[3] = {};
    uint16_t* units[16][3][2] = {};
    uint16_t* last = nullptr;
    auto lay_flush = [&]() {
        if (lay_count == 0) return;
        for (uint32_t i = lay_count; i < 64; ++i) lay.first[i] = 0xffffffffu;
        hipLaunchKernelGGL(codec_layout_kernel, dim3(lay_blocks), dim3(256), 0, s, lay);
        lay_count = lay_blocks = 0;
    };
    auto lay_add = [&](uint32_t i, uint16_t* to, uint32_t cin, uint32_t n, uint32_t taps, uint32_t ksteps, uint32_t kstep0) {
        if (lay_count == CD_LAYOUTS) lay_flush();
        lay.m[lay_count] = {reinterpret_cast<const uint8_t*>(ptrs[i]), to, n, cin, taps, ksteps, kstep0};
        lay.first[lay_count++] = lay_blocks;
        lay_blocks += (n + 63) / 64 * 2 * ((cin + 32 * cd_layout_groups(taps) - 1) / (32 * cd_layout_groups(taps)));
    };
    auto lay_one = [&](uint32_t q, uint32_t i, uint32_t cin, uint32_t n, uint32_t taps) {
        uint16_t* to = reinterpret_cast<uint16_t*>(take(2 * cd_fragments(cin, n, taps)));
        if (q >= part && q < end) lay_add(i, to, cin, n, taps, (cin + 31) / 32 * 2, 0);
        return to;
    };
    const uint32_t dsteps = d.dim / 32 * 2;
    front[0] = reinterpret_cast<uint16_t*>(take(2 * cd_fragments(d.books * d.dim, d.latent, 1)));
    if (part == 0)
        for (uint32_t c = 0; c < d.books; ++c)
            lay_add(3 * c + 1, front[0], d.dim, d.latent, 1, d.books * dsteps, c * dsteps);
    front[1] = lay_one(0, 3 * d.books, d.latent, d.hidden, 1);
    front[2] = lay_one(0, 3 * d.books + 2, d.hidden, d.channels, CD_TAPS);
    for (uint32_t b = 0; b < d.blocks; ++b)
        for (uint32_t u = 0; u < 3; ++u) {
            const uint32_t i = at(b + 1) + 3 + 6 * u, co = d.channels >> (b + 1);
            units[b][u][0] = lay_one(b + 1, i + 2, co, co, CD_TAPS);
            units[b][u][1] = lay_one(b + 1, i + 4, co, co, 1);
        }
    last = lay_one(d.blocks + 1, at(d.blocks + 1) + 1, d.channels >> d.blocks, 1, CD_TAPS);
    lay_flush();
    T2H_LAUNCH_CHECK();

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

    if (part == 0) {
        CdTables tables = {};
        for (uint32_t c = 0; c < d.books; ++c) {
            tables.rows[c] = reinterpret_cast<const uint8_t*>(ptrs[3 * c]);
            tables.count[c] = table_rows[c];
            tables.bias[c] = f32(3 * c + 2);
        }
        const uint64_t work = (uint64_t)frames * d.books * (d.dim / 8) + d.latent;
        hipLaunchKernelGGL(codec_embed_kernel, dim3((uint32_t)((work + 255) / 256)), dim3(256), 0, s, tables, codes,
                           d.books, d.dim, frames, d.latent, gathered, bias0);
        T2H_LAUNCH_CHECK();
        const uint32_t i = 3 * d.books;
        conv(gathered, front[0], bias0, frames, d.books * d.dim, d.latent, 1, 0, nullptr, nullptr, latent, nullptr, nullptr);
        conv(latent, front[1], f32(i + 1), frames, d.latent, d.hidden, 1, 0, nullptr, nullptr, hidden, nullptr, nullptr);
        conv(hidden, front[2], f32(i + 3), frames, d.hidden, d.channels, CD_TAPS, 1, nullptr,
             stages ? stages[0] : nullptr, nullptr, xs, f32(i + 4));
        T2H_LAUNCH_CHECK();
    }
    static const uint32_t dils[3] = {1, 3, 9};
    for (uint32_t b = part == 0 ? 0 : part - 1; b < d.blocks && b + 1 < end; ++b) {
        const uint32_t ch = d.channels >> b, co = ch / 2, stride = d.strides[b], first = at(b + 1);
        const uint64_t li = d.len(frames, b), len = li * stride;
        float* x = stages ? stages[1 + 4 * b] : xr;
        const int64_t strides[3] = {(int64_t)(li * ch), 1, (int64_t)ch};
        st = conv_transpose1d_q8_0_launch(xs, strides, ptrs[first + 1], f32(first + 2), x, 1, ch, (uint32_t)li, co,
                                          2 * stride, stride, (stride + 1) / 2, (uint32_t)len, s1, f32(first + 3), eps,
                                          stream);
        if (st) return st;
        for (uint32_t u = 0; u < 3; ++u) {
            const uint32_t i = first + 3 + 6 * u;  // a1, a2, c1, its bias, c2, its bias; then the next snake's alpha
            conv(s1, units[b][u][0], f32(i + 3), len, co, co, CD_TAPS, dils[u], nullptr, nullptr, s2, nullptr, f32(i + 1));
            const bool third = u == 2, final = third && b + 1 == d.blocks;
            float* raw = stages ? stages[2 + 4 * b + u] : (third ? nullptr : xr);
            conv(s2, units[b][u][1], f32(i + 5), len, co, co, 1, 0, x, raw, third && !final ? nullptr : s1,
                 third && !final ? xs : nullptr, f32(i + 6));
            x = raw;
            T2H_LAUNCH_CHECK();
        }
    }
    if (end == d.blocks + 2) {
        const uint32_t i = at(d.blocks + 1);
        conv(s1, last, f32(i + 2), d.len(frames, d.blocks), d.channels >> d.blocks, 1, CD_TAPS, 1, nullptr, out, nullptr,
             nullptr, nullptr);
        T2H_LAUNCH_CHECK();
    }
    return T2H_OK;
}
