// The audio tower's conv2d front end (3 x 3, stride 2, pad 1, + bias + GELU; channels-last bf16 activations) as
// implicit GEMMs: no patch matrix is written (pytorch_modules.py:452-526 of the reference runs conv2d).
//
//   conv2d_kernel     C >= 64 input channels.  Weight rows are bf16 and tap-major (k = tap * C + channel, zero-padded to
//                     a whole 64-deep stage), so a 16-B chunk of a stage is 8 channels of one tap: the LDS-DMA that
//                     brings a stage reads it straight from the activation, or from zeros where the tap is outside.
//                     At 256 x 256 tiles one wave a SIMD issues both the DMA and the products, and the matrix cores
//                     are busy 43 % of the launch (250 tiles, waits 15 % of the waves' cycles); at 128 x 128 22 %,
//                     LDS 22 % (half of it bank conflicts), waits 43 %.  32000 pixels of C 480, N 480 in 142 us
//                     (930 TFLOP/s) against 421 us as a patch matrix (276 MB) and a GEMM, 8320 pixels in 62 against
//                     132, 208 pixels in 21 against 28.  Tried: 32-deep stages that walk the 9 taps of 32 channels at a
//                     time (fewer bytes from HBM, but 64-B requests run at two thirds of the L2's rate): 141 at 32000
//                     pixels, 67 at 8320, 30 at 208.
//   conv2d_1ch_kernel one fp32 input channel (the mel spectrogram): the at most 16 taps are one MFMA step; bound by
//                     the GELU's arithmetic (VALU busy three quarters of the launch) and the output's bytes (128000
//                     pixels, N 480: 58 us for 123 MB, against 92 as patch rows and a GEMM).
#include "gemm_formats.h"
#include "lds_dma.h"

namespace t2h {

// ------------------------------------------------------- many channels ----

struct Conv2dArgs {
    const uint16_t* x;    // [batch, h, w, c] bf16
    const uint16_t* wt;   // [n, kp] bf16, tap-major
    const float* bias;    // [n] or null
    uint16_t* out;        // [m, n] bf16, m = batch * oh * ow
    uint32_t h, w, c, kh, kw, stride, pad, oh, ow;
    uint32_t m, n, kp, act;
    uint32_t tiles_m, tiles_n;
};

constexpr int CV_THREADS = 256;
constexpr int CV_BK = 64;
constexpr int CV_ROWB = CV_BK * 2;  // bytes per LDS row of a stage

__device__ __align__(16) const uint8_t conv2d_zeros[16] = {};

// A DMA instruction writes 1 KB of LDS, lane after lane: 8 rows of 128 B.  Of an operand's R rows, instruction g of G =
// R / 8 brings rows g, g + G, .. and lies 1040 B after the one before: eight lanes read a row's 128 B in order, and a
// fragment read (one 16-B chunk of 32 consecutive rows) finds 16 consecutive rows in 16 distinct groups of 4 banks.  At
// 256 rows no conflicts are counted; at 128, where rows 16 to 31 lie 128 B after rows 0 to 15, half of the LDS cycles.
constexpr int CV_DMA_PITCH = 1024 + 16;
__device__ __forceinline__ constexpr uint32_t cv_lds_row(uint32_t r, uint32_t G) {
    return r % G * CV_DMA_PITCH + r / G * CV_ROWB;
}

// 4 waves (2 x 2), each (32 MI) x (32 NJ) of a (64 MI) x (64 NJ) tile; S stages of 64 K in LDS.  One barrier a stage,
// before its last 16-deep step, whose fragments are then in registers: after it every wave is done with the stage's
// buffer, and the DMA of the stage S ahead goes into it between that step's MFMAs.
template <int MI, int NJ, int S>
__global__ __launch_bounds__(CV_THREADS) void conv2d_kernel(const Conv2dArgs a) {
    constexpr int BM = 64 * MI, BN = 64 * NJ;
    constexpr int GA = BM / 8, GW = BN / 8;        // DMA instructions a stage
    constexpr int IA = GA / 4, IW = GW / 4;        // and a wave
    constexpr int DMA = IA + IW;
    constexpr int STAGE = (GA + GW) * CV_DMA_PITCH;
    constexpr int STEPS = CV_BK / 16;
    __shared__ __align__(16) uint8_t lds[S * STAGE];

    // columns first: the tiles that read the same pixels share an L2
    const uint32_t pid = xcd_run(a.tiles_m * a.tiles_n);
    const uint32_t m0 = pid / a.tiles_n * BM, n0 = pid % a.tiles_n * BN;

    const uint32_t t = threadIdx.x;
    const int lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int wm = wave >> 1, wn = wave & 1;
    const uint32_t KT = a.kp / CV_BK;
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane(
        (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)&lds[0]);

    const uint8_t* src_a[IA];   // the row's pixel (0, 0) of the patch, possibly outside the image
    uint32_t inside[IA];        // bit tap: the tap is inside the image
    const uint8_t* src_w[IW];
    const uint32_t chunk = (lane & 7) * 16;
#pragma unroll
    for (int i = 0; i < IA; ++i) {
        const uint32_t row = min(m0 + wave * IA + i + GA * (lane >> 3), a.m - 1);
        const uint32_t ox = row % a.ow, rest = row / a.ow, oy = rest % a.oh, b = rest / a.oh;
        const int iy = (int)(oy * a.stride) - (int)a.pad, ix = (int)(ox * a.stride) - (int)a.pad;
        src_a[i] = reinterpret_cast<const uint8_t*>(a.x) +
                   ((((int64_t)b * a.h + iy) * a.w + ix) * (int64_t)a.c) * 2 + chunk;
        uint32_t bits = 0, tap = 0;
        for (uint32_t ky = 0; ky < a.kh; ++ky)
            for (uint32_t kx = 0; kx < a.kw; ++kx, ++tap)
                if ((uint32_t)(iy + (int)ky) < a.h && (uint32_t)(ix + (int)kx) < a.w) bits |= 1u << tap;
        inside[i] = bits;
    }
#pragma unroll
    for (int i = 0; i < IW; ++i) {
        const uint32_t row = min(n0 + wave * IW + i + GW * (lane >> 3), a.n - 1);
        src_w[i] = reinterpret_cast<const uint8_t*>(a.wt + (size_t)row * a.kp) + chunk;
    }
    // where this lane's chunk of the next stage lies: its tap, the tap's column, the channel within the tap, and the byte
    // offset from the patch's first pixel (the taps of one patch row are contiguous in memory); and the stage's byte
    // offset in a weight row
    uint32_t tap = 0, kx = 0, ch = chunk / 2, off = 0, kb = 0;  // ch < 64 <= c
    const uint32_t next_row = (a.w - a.kw) * a.c * 2;
    const uint32_t dma_a = lds0 + wave * IA * CV_DMA_PITCH, dma_w = lds0 + (GA + wave * IW) * CV_DMA_PITCH;
    // past the last stage the taps are outside (zeros) and the last weights are re-read, so that the waits stay the same
    // for every stage
    auto advance = [&]() {
        kb = min(kb + CV_ROWB, (KT - 1) * CV_ROWB);
        ch += CV_BK;
        off += CV_ROWB;
        const bool wrap = ch >= a.c;
        ch -= wrap ? a.c : 0;
        tap += wrap ? 1 : 0;
        kx += wrap ? 1 : 0;
        const bool down = kx == a.kw;
        kx = down ? 0 : kx;
        off += down ? next_row : 0;
    };
    // DMA instruction q (0 .. DMA - 1, in order) of the next stage into buffer buf
    auto issue = [&](int q, uint32_t buf) {
        if (q < IA) {
            const uint8_t* g = (inside[q] >> tap) & 1 ? src_a[q] + off : conv2d_zeros;
            lds_dma16(g, dma_a + buf * STAGE + q * CV_DMA_PITCH);
        } else {
            lds_dma16(src_w[q - IA] + kb, dma_w + buf * STAGE + (q - IA) * CV_DMA_PITCH);
        }
        if (q == DMA - 1) advance();
    };

    f32x16_t acc[MI][NJ];
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;

    const uint32_t fr = lane & 31, fh = lane >> 5;
    uint32_t off_a[MI], off_w[NJ];
#pragma unroll
    for (int i = 0; i < MI; ++i) off_a[i] = cv_lds_row((wm * MI + i) * 32 + fr, GA);
#pragma unroll
    for (int j = 0; j < NJ; ++j) off_w[j] = GA * CV_DMA_PITCH + cv_lds_row((wn * NJ + j) * 32 + fr, GW);
    bf16x8_t fa[2][MI], fb[2][NJ];
    auto read_step = [&](uint32_t buf, int step, int b) {
        const uint8_t* st = lds + buf * STAGE;
        const uint32_t slot = (step * 2 + fh) * 16;
#pragma unroll
        for (int i = 0; i < MI; ++i) fa[b][i] = *reinterpret_cast<const bf16x8_t*>(st + off_a[i] + slot);
#pragma unroll
        for (int j = 0; j < NJ; ++j) fb[b][j] = *reinterpret_cast<const bf16x8_t*>(st + off_w[j] + slot);
    };
    auto mma_step = [&](int b) {
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int j = 0; j < NJ; ++j)
                acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[b][i], fb[b][j], acc[i][j], 0, 0, 0);
        if constexpr (MI * NJ >= MI + NJ) {
#pragma unroll
            for (int i = 0; i < MI + NJ; ++i) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // one MFMA
                __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // one LDS read
            }
            __builtin_amdgcn_sched_group_barrier(0x008, MI * NJ - MI - NJ, 0);
        }
    };

#pragma unroll
    for (int s = 0; s < S; ++s) {
#pragma unroll
        for (int q = 0; q < DMA; ++q) issue(q, s);
    }
    wait_vm<(S - 1) * DMA>();
    wave_barrier();
    read_step(0, 0, 0);
    uint32_t buf = 0;
    for (uint32_t kt = 0; kt + 1 < KT; ++kt) {
#pragma unroll
        for (int step = 0; step + 1 < STEPS; ++step) {
            read_step(buf, step + 1, (step + 1) & 1);
            mma_step(step & 1);
        }
        // stage kt + 1 landed (every wave's DMA), stage kt's reads done (every wave)
        wait_vm<(S - 2) * DMA>();
        wait_lgkm0();
        wave_barrier();
        const uint32_t next = buf + 1 == S ? 0 : buf + 1;
        read_step(next, 0, 0);
        constexpr int MM = MI * NJ;
#pragma unroll
        for (int q = 0; q < MM; ++q) {
            acc[q / NJ][q % NJ] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                fa[(STEPS - 1) & 1][q / NJ], fb[(STEPS - 1) & 1][q % NJ], acc[q / NJ][q % NJ], 0, 0, 0);
#pragma unroll
            for (int i = q * DMA / MM; i < (q + 1) * DMA / MM; ++i) issue(i, buf);
        }
        buf = next;
    }
#pragma unroll
    for (int step = 0; step < STEPS; ++step) {
        if (step + 1 < STEPS) read_step(buf, step + 1, (step + 1) & 1);
        mma_step(step & 1);
    }
    wait_vm<0>();  // the stages issued past the end still write LDS

    // lane holds column (lane % 32) of each 32 x 32 tile, rows 8(e/4) + 4(lane/32) + e%4
    const uint32_t row_base = m0 + wm * 32 * MI + (lane >> 5) * 4;
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
        const uint32_t col = n0 + (wn * NJ + j) * 32 + (lane & 31);
        const float bj = a.bias != nullptr && col < a.n ? a.bias[col] : 0.0f;
#pragma unroll
        for (int i = 0; i < MI; ++i) {
            float ov[16];
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                ov[e] = acc[i][j][e] + bj;
                if (a.act == GQACT_GELU) ov[e] = gelu_erf(ov[e]);
            }
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const uint32_t row = row_base + i * 32 + (e >> 2) * 8 + (e & 3);
                if (row < a.m && col < a.n) a.out[(size_t)row * a.n + col] = (uint16_t)f32_to_bf16_bits(ov[e]);
            }
        }
    }
}

// Q8_0 rows [n, c taps] (element c taps + tap) -> the weight rows above.  A block converts up to 512 channels of a row:
// 32 channels are `taps` whole Q8_0 blocks, one a thread, and the taps are picked apart in LDS.  Laid out before every
// convolution, so that it uses the weights as they are then: 480 rows of C 480, 9 taps, in 5 us.
constexpr uint32_t CR_CHANNELS = 512, CR_MAX_TAPS = 24;
__global__ __launch_bounds__(256) void conv2d_rows_kernel(const uint8_t* __restrict__ w, uint32_t c, uint32_t taps,
                                                          uint32_t kp, uint16_t* __restrict__ out) {
    __shared__ __align__(16) uint16_t ls[CR_CHANNELS * CR_MAX_TAPS];
    const uint32_t c0 = blockIdx.y * CR_CHANNELS, cn = min(CR_CHANNELS, c - c0);
    const uint32_t blocks = (c * taps + 31) / 32, b0 = c0 / 32 * taps, bn = min(CR_CHANNELS / 32 * taps, blocks - b0);
    const uint8_t* src = w + ((size_t)blockIdx.x * blocks + b0) * 34;
    for (uint32_t i = threadIdx.x; i < bn; i += 256) {
        GemmQ80::Raw r;
        r.d = load_u16(src + 34 * i);
        r.inside = true;
        r.q0 = load_u4_ua(src + 34 * i + 2);
        r.q1 = load_u4_ua(src + 34 * i + 18);
        uint32_t o[16];
        GemmQ80::convert(r, 0, 0, o);
#pragma unroll
        for (int j = 0; j < 4; ++j)
            *reinterpret_cast<uint4*>(ls + 32 * i + 8 * j) = make_uint4(o[4 * j], o[4 * j + 1], o[4 * j + 2], o[4 * j + 3]);
    }
    __syncthreads();
    uint16_t* row = out + (size_t)blockIdx.x * kp;
    const uint32_t chunks = (cn + 7) / 8;
    for (uint32_t i = threadIdx.x; i < chunks * taps; i += 256) {
        const uint32_t tap = i / chunks, ch = i % chunks * 8;
        uint16_t v[8];
#pragma unroll
        for (uint32_t j = 0; j < 8; ++j) v[j] = ls[min(ch + j, cn - 1) * taps + tap];
        uint16_t* dst = row + (size_t)tap * c + c0 + ch;
        if (c % 8 == 0) {
            *reinterpret_cast<uint4*>(dst) =
                make_uint4(v[0] | (uint32_t)v[1] << 16, v[2] | (uint32_t)v[3] << 16, v[4] | (uint32_t)v[5] << 16,
                           v[6] | (uint32_t)v[7] << 16);
        } else {
#pragma unroll
            for (uint32_t j = 0; j < 8; ++j)
                if (ch + j < cn) dst[j] = v[j];
        }
    }
    if (blockIdx.y == 0 && c * taps + threadIdx.x < kp) row[c * taps + threadIdx.x] = 0;  // fewer than 64
}

// --------------------------------------------------------- one channel ----

struct Conv2d1Args {
    const float* x;      // [batch, h, w]
    const uint8_t* wq;   // [n, 34] Q8_0 rows of 32 values: the taps, then zeros
    const float* bias;   // [n] or null
    uint16_t* out;       // [m, n] bf16
    uint32_t h, w, kh, kw, stride, pad, oh, ow, m, n, act;
};

constexpr int C1_TILES = 4;     // 32-pixel tiles per wave, over which the weights are read once
constexpr int C1_PITCH = 72;    // bf16 per LDS row of 64 channels (144 B: 8-B writes of 16 rows hit all the banks)

// Wave: C1_TILES tiles of 32 pixels, 64 channels (blockIdx.y).  The weights are the MFMA's row operand, so a lane holds
// 4 consecutive channels of a pixel; they pass through LDS and leave as 128-B runs of a pixel's row.
__global__ __launch_bounds__(256) void conv2d_1ch_kernel(const Conv2d1Args a) {
    __shared__ __align__(16) uint16_t lds[4][32 * C1_PITCH];
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const uint32_t n0 = blockIdx.y * 64, taps = a.kh * a.kw;
    const uint32_t half = lane >> 5;  // taps 8 half .. + 7
    uint16_t* tile = lds[wave];

    bf16x8_t fw[2];
    float bias[2][16];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const uint32_t n = n0 + 32 * j + (lane & 31);
        const uint8_t* row = a.wq + (size_t)min(n, a.n - 1) * 34;
        const float d = f16_bits_to_f32(load_u16(row));
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const uint32_t tap = 8 * half + i;
            fw[j][i] = (__bf16)(tap < taps ? d * (float)(int8_t)row[2 + tap] : 0.0f);
        }
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const uint32_t ch = n0 + 32 * j + (e >> 2) * 8 + 4 * half + (e & 3);
            bias[j][e] = a.bias != nullptr && ch < a.n ? a.bias[ch] : 0.0f;
        }
    }
    const uint32_t first = (blockIdx.x * 4 + wave) * C1_TILES;
    for (uint32_t i = 0; i < C1_TILES; ++i) {
        const uint32_t m0 = (first + i) * 32;
        if (m0 < a.m) {
            const uint32_t row = min(m0 + (lane & 31), a.m - 1);
            const uint32_t ox = row % a.ow, rest = row / a.ow, oy = rest % a.oh, b = rest / a.oh;
            const int iy = (int)(oy * a.stride) - (int)a.pad, ix = (int)(ox * a.stride) - (int)a.pad;
            const float* image = a.x + (size_t)b * a.h * a.w;
            bf16x8_t fx;
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                const uint32_t tap = 8 * half + k;
                const uint32_t y = (uint32_t)(iy + (int)(tap / a.kw)), xx = (uint32_t)(ix + (int)(tap % a.kw));
                fx[k] = (__bf16)(tap < taps && y < a.h && xx < a.w ? image[(size_t)y * a.w + xx] : 0.0f);
            }
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                f32x16_t acc;
#pragma unroll
                for (int e = 0; e < 16; ++e) acc[e] = 0.0f;
                acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fw[j], fx, acc, 0, 0, 0);
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    float v[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        v[e] = acc[4 * g + e] + bias[j][4 * g + e];
                        if (a.act == GQACT_GELU) v[e] = gelu_erf(v[e]);
                    }
                    *reinterpret_cast<uint2*>(tile + (lane & 31) * C1_PITCH + 32 * j + 8 * g + 4 * half) =
                        make_uint2(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]));
                }
            }
        }
        __syncthreads();
        if (m0 < a.m) {
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                const uint32_t pixel = 8 * s + (lane >> 3), ch = (lane & 7) * 8;
                const uint4 v = *reinterpret_cast<const uint4*>(tile + pixel * C1_PITCH + ch);
                if (m0 + pixel < a.m && n0 + ch < a.n)
                    *reinterpret_cast<uint4*>(a.out + (size_t)(m0 + pixel) * a.n + n0 + ch) = v;
            }
        }
        __syncthreads();
    }
}

// ------------------------------------------------------------- entries ----

// Output size of one axis, 0 where the kernel does not fit.
static uint32_t conv2d_out(uint32_t size, uint32_t k, uint32_t stride, uint32_t pad) {
    const uint64_t padded = (uint64_t)size + 2ull * pad;
    return padded < k ? 0 : (uint32_t)((padded - k) / stride + 1);
}

static int conv2d_geometry(uint32_t batch, uint32_t h, uint32_t w, uint32_t kh, uint32_t kw, uint32_t stride, uint32_t pad,
                           uint32_t max_taps, uint32_t* oh, uint32_t* ow, uint64_t* m) {
    if (batch == 0 || h == 0 || w == 0 || kh == 0 || kw == 0 || stride == 0) return T2H_ERR_SHAPE;
    if (kh > max_taps || kw > max_taps || kh * kw > max_taps || pad > 0xffff || stride > 0xffff || h > 0xffffff ||
        w > 0xffffff)
        return T2H_ERR_UNSUPPORTED;
    *oh = conv2d_out(h, kh, stride, pad);
    *ow = conv2d_out(w, kw, stride, pad);
    if (*oh == 0 || *ow == 0) return T2H_ERR_SHAPE;
    *m = (uint64_t)batch * *oh * *ow;
    return *m >= (1ull << 31) ? T2H_ERR_UNSUPPORTED : T2H_OK;
}

template <int MI, int NJ, int S>
static void conv2d_launch(Conv2dArgs& a, hipStream_t s) {
    a.tiles_m = (a.m + 64 * MI - 1) / (64 * MI);
    a.tiles_n = (a.n + 64 * NJ - 1) / (64 * NJ);
    hipLaunchKernelGGL((conv2d_kernel<MI, NJ, S>), dim3(a.tiles_m * a.tiles_n), dim3(CV_THREADS), 0, s, a);
}

}  // namespace t2h

using namespace t2h;

extern "C" int t2h_conv2d_bf16(const void* x, const void* w_rows, const void* bias, int act, void* out, uint32_t batch,
                               uint32_t h, uint32_t w, uint32_t channels, uint32_t n, uint32_t kh, uint32_t kw,
                               uint32_t stride, uint32_t pad, int tile, void* stream) {
    if (!x || !w_rows || !out) return T2H_ERR_NULL;
    if (act != 0 && act != GQACT_GELU) return T2H_ERR_UNSUPPORTED;
    if (n == 0 || channels == 0) return T2H_ERR_SHAPE;
    if (channels % 8 != 0 || channels < CV_BK || channels > 0xffff) return T2H_ERR_UNSUPPORTED;
    uint32_t oh, ow;
    uint64_t m;
    const int rc = conv2d_geometry(batch, h, w, kh, kw, stride, pad, 24, &oh, &ow, &m);
    if (rc != T2H_OK) return rc;
    if (kw > w || (uint64_t)kh * w * channels * 2 >= (1ull << 31)) return T2H_ERR_UNSUPPORTED;  // 32-bit patch offsets
    if (((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w_rows)) & 15) != 0) return T2H_ERR_ALIGN;
    if ((reinterpret_cast<uintptr_t>(bias) & 3) != 0 || (reinterpret_cast<uintptr_t>(out) & 1) != 0) return T2H_ERR_ALIGN;
    Conv2dArgs a = {};
    a.x = static_cast<const uint16_t*>(x);
    a.wt = static_cast<const uint16_t*>(w_rows);
    a.bias = static_cast<const float*>(bias);
    a.out = static_cast<uint16_t*>(out);
    a.h = h, a.w = w, a.c = channels, a.kh = kh, a.kw = kw, a.stride = stride, a.pad = pad, a.oh = oh, a.ow = ow;
    a.m = (uint32_t)m, a.n = n, a.act = (uint32_t)act;
    a.kp = (kh * kw * channels + CV_BK - 1) / CV_BK * CV_BK;
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    // The largest tile that still fills the chip: a 64 x 64 tile reads 2 LDS fragments a product, a 128 x 128 one 1, a
    // 256 x 256 one half, but 256 CUs run 768, 512 (256 of the three-stage form) and 256 of them at once.  C 480, N 480,
    // 3 x 3, us as 64 x 64 / 128 x 128 (3 stages) / 128 x 128 (2 stages) / 256 x 256:
    //   208 rows 21 / 39 / 39 / 106      3120 rows 29 / 40 / 49 / 110     4160 rows 40 / 42 / 50 / 110
    //   6240 rows 56 / 41 / 49 / 110     8000 rows 66 / 49 / 60 / 122    12000 rows 92 / 86 / 75 / 123
    //   24000 rows 178 / 134 / 131 / 128 32000 rows 237 / 177 / 156 / 142
    // C = N 64, 128, 256 and 768 at 56 to 48000 rows: within 6 % of the fastest of the four, but for two of the 40:
    // 8320 rows of 256 (26.7 against 22.9 as 64 x 64) and 48000 of 64, half of whose 128 columns are padding (18.8
    // against 11.9)
    if (tile < 0) {
        const uint64_t t64 = ((m + 63) / 64) * ((n + 63) / 64), t128 = ((m + 127) / 128) * ((n + 127) / 128);
        const uint64_t t256 = ((m + 255) / 256) * ((n + 255) / 256);
        if (t64 <= 512) tile = 0;
        else if (t128 <= 256) tile = 1;
        else tile = (t256 + 255) / 256 * 7 <= (t128 + 511) / 512 * 4 ? 3 : 2;  // a round of 256 x 256 costs 1.75 of 128 x 128
    }
    if (tile == 0) conv2d_launch<1, 1, 3>(a, s);
    else if (tile == 1) conv2d_launch<2, 2, 3>(a, s);
    else if (tile == 2) conv2d_launch<2, 2, 2>(a, s);
    else if (tile == 3) conv2d_launch<4, 4, 2>(a, s);
    else return T2H_ERR_UNSUPPORTED;
    T2H_LAUNCH_CHECK();
    return T2H_OK;
}

extern "C" int t2h_conv2d_rows_q8_0(const void* w, uint32_t n, uint32_t channels, uint32_t taps, void* out, void* stream) {
    if (!w || !out) return T2H_ERR_NULL;
    if (n == 0 || channels == 0 || taps == 0) return T2H_ERR_SHAPE;
    if (taps > CR_MAX_TAPS || channels > 0xffff || n > 0x7fffffffu) return T2H_ERR_UNSUPPORTED;
    if ((reinterpret_cast<uintptr_t>(w) & 1) != 0 || (reinterpret_cast<uintptr_t>(out) & 15) != 0) return T2H_ERR_ALIGN;
    hipLaunchKernelGGL(conv2d_rows_kernel, dim3(n, (channels + CR_CHANNELS - 1) / CR_CHANNELS), dim3(256), 0,
                       reinterpret_cast<hipStream_t>(stream), reinterpret_cast<const uint8_t*>(w), channels, taps,
                       (channels * taps + CV_BK - 1) / CV_BK * CV_BK, reinterpret_cast<uint16_t*>(out));
    T2H_LAUNCH_CHECK();
    return T2H_OK;
}

extern "C" int t2h_conv2d_1ch_q8_0(const void* x, const void* w, const void* bias, int act, void* out, uint32_t batch,
                                   uint32_t h, uint32_t w_in, uint32_t n, uint32_t kh, uint32_t kw, uint32_t stride,
                                   uint32_t pad, void* stream) {
    if (!x || !w || !out) return T2H_ERR_NULL;
    if (act != 0 && act != GQACT_GELU) return T2H_ERR_UNSUPPORTED;
    if (n == 0) return T2H_ERR_SHAPE;
    if (n % 8 != 0 || n > 64u * 65535u) return T2H_ERR_UNSUPPORTED;
    uint32_t oh, ow;
    uint64_t m;
    const int rc = conv2d_geometry(batch, h, w_in, kh, kw, stride, pad, 16, &oh, &ow, &m);
    if (rc != T2H_OK) return rc;
    if ((reinterpret_cast<uintptr_t>(x) & 3) != 0 || (reinterpret_cast<uintptr_t>(bias) & 3) != 0) return T2H_ERR_ALIGN;
    if ((reinterpret_cast<uintptr_t>(w) & 1) != 0 || (reinterpret_cast<uintptr_t>(out) & 15) != 0) return T2H_ERR_ALIGN;
    Conv2d1Args a = {};
    a.x = static_cast<const float*>(x);
    a.wq = static_cast<const uint8_t*>(w);
    a.bias = static_cast<const float*>(bias);
    a.out = static_cast<uint16_t*>(out);
    a.h = h, a.w = w_in, a.kh = kh, a.kw = kw, a.stride = stride, a.pad = pad, a.oh = oh, a.ow = ow;
    a.m = (uint32_t)m, a.n = n, a.act = (uint32_t)act;
    const uint32_t per_block = 4 * C1_TILES * 32;
    hipLaunchKernelGGL(conv2d_1ch_kernel, dim3((uint32_t)((m + per_block - 1) / per_block), (n + 63) / 64), dim3(256), 0,
                       reinterpret_cast<hipStream_t>(stream), a);
    T2H_LAUNCH_CHECK();
    return T2H_OK;
}
