// Transposed conv1d over Q8_0 weights, fp32 (the audio codec's upsampling):
//   CONV_TRANSPOSE1D_Q8_0W_F32B_F32
//   (src/models/quantized_omnivoice/shaders/conv_transpose1d_q8_0w_f32b_f32.py:
//    deconv_input_value, deconv_weight_value)
//
//   y[b, t, co] = bias[co] + sum_ci sum_k W[ci, co K + k] x[b, ci, i] over the taps k with
//   t + pad - k = i * stride, 0 <= i < L_in,
// reading the reference's Q8_0 rows [Ci, Co K] (34-byte blocks: fp16 scale + 32 int8) as they are.
//
// As a product it is G[i, e] = sum_ci x[i, ci] W[ci, e], e = co K + k, followed by a fold that adds, for an
// output position u = t + pad, the entries k = u % stride, k + stride, ... of rows i = u / stride, i - 1, ...
// Everything stays fp32: weights d * q, inputs, products and sums (v_mfma_f32_32x32x2_f32).
#include "codec.h"

namespace t2h {

typedef float ct_f32x16_t __attribute__((ext_vector_type(16)));

struct ConvTArgs {
    const float* x;
    int64_t sb, sc, sl;     // x strides (elements): batch, channel, position
    const uint8_t* w;
    const float* bias;
    float* out;             // [B, L_out, Co] contiguous
    uint32_t ci, li, co, kh, stride, pad, lo;
    uint32_t row_bytes;     // Q8_0 bytes per weight row (ceil(Co K / 32) * 34)
    uint64_t n;             // B * L_out * Co
    uint32_t nt;            // tiled kernel: 32-column tiles per block
    uint32_t halo;          // rows of G before an output's own that its taps reach: ceil(K / stride) - 1
    int32_t i_first;        // pad / stride, the row of the first output
    uint32_t vec;           // x rows can be read 4 channels at a time
    uint16_t* snaked;       // bf16 [B, L_out, Co] of snake(y, alpha), or null
    const float* alpha;
    float eps;
};

// One block: 32 rows i (the first `halo` of them only feed the others' outputs) x nt column tiles of 32
// entries e, one wave per column tile, so a tile's B operand is exactly one Q8_0 block per channel and nt K is
// a whole number of output channels: the fold needs nothing from other blocks and G never leaves LDS.
// Channels stream through LDS 32 at a time, CT_RING - 1 stages of loads in flight to registers.  What bounds a block is
// its chain of stages: a wave and stage is 16 MFMAs of 64 cycles, and staging B (dequantising 16 values a lane, writing
// and reading them once in LDS) comes before them for a tile of only 32 rows.  Measured over the codec's five upsampling
// layers at 75 frames (1024 to 64 channels, strides 8, 5, 4, 2, 3; 5.8 GFLOP): 2917 us for the per-output kernel below,
// 160 us here (36 + 41 + 33 + 24 + 26).  Counters of the first, second, fourth and last: matrix cores busy 24, 23, 18
// and 11 % of the launch, LDS 17, 14, 16 and 9 %, waves waiting 28, 37, 29 and 43 % of their cycles; the first fills 192 CUs.
constexpr int CT_ROWS = 32;     // rows of G per block
constexpr int CT_CB = 32;       // channels per LDS stage
constexpr int CT_MAX_NT = 8;
constexpr int CT_RING = 4;
constexpr int CT_AROW = CT_CB + 4;  // LDS row of A: 16-byte reads of 16 consecutive rows hit distinct banks

__global__ __launch_bounds__(CT_MAX_NT * 64) void conv_transpose1d_tile_kernel(const ConvTArgs a) {
    __shared__ __align__(16) float as[CT_ROWS * CT_AROW];
    __shared__ __align__(16) float bs[CT_CB * (32 * CT_MAX_NT + 8)];  // B stage, then the G tile
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const uint32_t nt = a.nt, nthreads = nt * 64;
    const uint32_t brow = 32 * nt + 8;  // = 8 (mod 16) words: the half-waves' rows, 4 apart, use distinct banks
    const uint32_t useful = CT_ROWS - a.halo;
    const int i0 = a.i_first + (int)(blockIdx.x * useful) - (int)a.halo;  // row of G of tile row 0
    const uint32_t eb0 = blockIdx.y * nt;                                  // first 32-entry block of the tile
    const uint32_t eb_count = a.row_bytes / 34;
    const float* xb = a.x + (int64_t)blockIdx.z * a.sb;

    // Register stages: CT_RING - 1 stages of loads are in flight while one is multiplied (a stage's 16 MFMAs are
    // 0.4 us, a load under load about 1 us; few blocks share a CU where channels are many and positions few)
    struct Stage {
        float4 a;
        uint4 q;
        uint32_t d;
    } st[CT_RING];
    // A: thread idx < 256 takes row idx / 8, channels 4 (idx % 8)
    const bool a_thread = tid < CT_ROWS * CT_CB / 4;
    const uint32_t ac = 4 * (tid & 7);
    const int ai = i0 + (int)(tid >> 3);
    const bool a_in = a_thread && ai >= 0 && ai < (int)a.li;
    const float* ax = xb + (int64_t)(a_in ? ai : 0) * a.sl;
    // B: thread pair 2 j, 2 j + 1 takes the halves of block (channel j / nt, column tile j % nt)
    const uint32_t half = tid & 1, bc = (tid >> 1) / nt, bt = (tid >> 1) % nt;
    const uint8_t* bw = a.w + (size_t)min(eb0 + bt, eb_count - 1) * 34;  // a tile past the row's end: never stored
    auto load_stage = [&](uint32_t c0, Stage& s) {
        s.a = make_float4(0.f, 0.f, 0.f, 0.f);
        const uint32_t c = c0 + ac;
        if (a_in && c < a.ci) {
            const float* p = ax + (int64_t)c * a.sc;
            if (a.vec) {
                s.a = *reinterpret_cast<const float4*>(p);
            } else {
                s.a.x = p[0];
                if (c + 1 < a.ci) s.a.y = p[a.sc];
                if (c + 2 < a.ci) s.a.z = p[2 * a.sc];
                if (c + 3 < a.ci) s.a.w = p[3 * a.sc];
            }
        }
        const uint8_t* p = bw + (size_t)min(c0 + bc, a.ci - 1) * a.row_bytes;
        s.d = load_u16(p);
        s.q = load_u4_ua(p + 2 + 16 * half);
    };
    auto store_stage = [&](uint32_t c0, const Stage& s) {
        if (a_thread) *reinterpret_cast<float4*>(&as[(tid >> 3) * CT_AROW + ac]) = s.a;
        const float d = c0 + bc < a.ci ? f16_bits_to_f32(s.d) : 0.0f;  // past the last channel: zero, as A is
        const uint32_t q[4] = {s.q.x, s.q.y, s.q.z, s.q.w};
        float* dst = &bs[bc * brow + 32 * bt + 16 * half];
#pragma unroll
        for (int j = 0; j < 4; ++j)
            *reinterpret_cast<float4*>(dst + 4 * j) =
                make_float4(d * (float)(int8_t)(q[j] & 0xffu), d * (float)(int8_t)((q[j] >> 8) & 0xffu),
                            d * (float)(int8_t)((q[j] >> 16) & 0xffu), d * (float)(int8_t)(q[j] >> 24));
    };

    ct_f32x16_t acc;
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[e] = 0.0f;
    const uint32_t r32 = lane & 31, h = lane >> 5;
#pragma unroll
    for (int i = 0; i + 1 < CT_RING; ++i)
        if (i * CT_CB < a.ci) load_stage(i * CT_CB, st[i]);
    for (uint32_t cr = 0; cr < a.ci; cr += CT_RING * CT_CB) {
#pragma unroll
        for (int i = 0; i < CT_RING; ++i) {
            const uint32_t c0 = cr + i * CT_CB;
            if (c0 >= a.ci) break;  // block-uniform
            store_stage(c0, st[i]);
            __syncthreads();
            const uint32_t cn = c0 + (CT_RING - 1) * CT_CB;
            if (cn < a.ci) load_stage(cn, st[(i + CT_RING - 1) % CT_RING]);
            // lane half h supplies channels 8 g + 4 h + j of step (g, j) to both operands
            const float* ap = &as[r32 * CT_AROW + 4 * h];
            const float* bp = &bs[4 * h * brow + 32 * wave + r32];
#pragma unroll
            for (int g = 0; g < CT_CB / 8; ++g) {
                const float4 av = *reinterpret_cast<const float4*>(ap + 8 * g);
                const float av4[4] = {av.x, av.y, av.z, av.w};
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    acc = __builtin_amdgcn_mfma_f32_32x32x2f32(av4[j], bp[(8 * g + j) * brow], acc, 0, 0, 0);
            }
            __syncthreads();
        }
    }
    // G tile: lane holds column r32 of its wave's tile, rows 8 (e / 4) + 4 h + e % 4
#pragma unroll
    for (int e = 0; e < 16; ++e) bs[(8 * (e >> 2) + 4 * h + (e & 3)) * brow + 32 * wave + r32] = acc[e];
    __syncthreads();
    // fold: outputs (row, phase, channel), consecutive threads along channels.  nthreads is 2 K times the tile's
    // channels, so a thread keeps its channel and steps 2 K (row, phase) pairs: no division in the loop.
    const uint32_t nco = 32 * nt / a.kh, cl = tid % nco, co = 32 * eb0 / a.kh + cl;
    if (co >= a.co) return;
    const float bias = a.bias ? a.bias[co] : 0.0f;
    const float alpha = a.snaked ? a.alpha[co] : 0.0f;
    const uint32_t drow = 2 * a.kh / a.stride, dphase = 2 * a.kh % a.stride;
    uint32_t row = a.halo + tid / nco / a.stride, phase = tid / nco % a.stride;
    for (; row < CT_ROWS; row += drow, phase += dphase) {
        if (phase >= a.stride) {
            phase -= a.stride;
            if (++row >= CT_ROWS) break;
        }
        const int64_t t = (int64_t)(i0 + (int)row) * a.stride + phase - a.pad;
        if (t < 0 || t >= (int64_t)a.lo) continue;
        float v = bias;
        uint32_t gr = row;
        for (uint32_t k = phase; k < a.kh; k += a.stride, --gr) {
            const int i = i0 + (int)gr;  // rows outside the input are no taps (not zeros: 0 * inf)
            if (i >= 0 && i < (int)a.li) v += bs[gr * brow + cl * a.kh + k];
        }
        const uint64_t at = ((uint64_t)blockIdx.z * a.lo + (uint64_t)t) * a.co + co;
        a.out[at] = v;
        if (a.snaked) a.snaked[at] = (uint16_t)f32_to_bf16_bits(snake_f32(v, alpha, a.eps));
    }
}

// Kernel sizes whose whole channels do not fill CT_MAX_NT column tiles, or that reach more than half a tile of
// rows back: one thread per output (b, t, co), consecutive threads along co, so a wave shares every x it reads.
__global__ __launch_bounds__(256) void conv_transpose1d_q8_0_kernel(const ConvTArgs a) {
    const uint64_t idx = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= a.n) return;
    const uint32_t co = (uint32_t)(idx % a.co);
    const uint64_t r = idx / a.co;
    const uint32_t t = (uint32_t)(r % a.lo);
    const uint64_t b = r / a.lo;
    // first tap whose input position is a whole step: (t + pad - k) % stride == 0
    const uint32_t k0 = (t + a.pad) % a.stride;
    float acc = a.bias ? a.bias[co] : 0.0f;
    for (uint32_t k = k0; k < a.kh; k += a.stride) {
        const int num = (int)t + (int)a.pad - (int)k;
        if (num < 0) break;  // k only grows
        const uint32_t i = (uint32_t)num / a.stride;
        if (i >= a.li) continue;
        const uint32_t e = co * a.kh + k;          // element of every weight row
        const uint32_t blk = e >> 5, q = e & 31u;
        const float* xi = a.x + (int64_t)b * a.sb + (int64_t)i * a.sl;
        const uint8_t* wb = a.w + (size_t)blk * 34;
        for (uint32_t c = 0; c < a.ci; ++c) {
            const uint8_t* row = wb + (size_t)c * a.row_bytes;
            const float d = f16_bits_to_f32((uint32_t)row[0] | ((uint32_t)row[1] << 8));
            const float wv = d * (float)(int8_t)row[2 + q];
            acc = fmaf(wv, xi[(int64_t)c * a.sc], acc);
        }
    }
    a.out[idx] = acc;
    if (a.snaked) a.snaked[idx] = (uint16_t)f32_to_bf16_bits(snake_f32(acc, a.alpha[co], a.eps));
}

static uint32_t ct_gcd(uint32_t a, uint32_t b) {
    while (b) {
        const uint32_t t = a % b;
        a = b;
        b = t;
    }
    return a;
}

// Column tiles per block of the tiled kernel: the fewest 32-entry blocks that hold whole channels, times what
// keeps at least 4 waves in a block (A is loaded by 256 threads); 0: the kernel size does not fit.
static uint32_t ct_tiles(uint32_t kh) {
    const uint32_t base = kh / ct_gcd(kh, 32);
    if (base > (uint32_t)CT_MAX_NT) return 0;
    return base * (base >= 4 ? 1 : (4 + base - 1) / base);
}

int conv_transpose1d_q8_0_launch(const float* x, const int64_t* x_strides, const void* w, const float* bias,
                                 float* out, uint32_t batch, uint32_t ci, uint32_t li, uint32_t co, uint32_t kh,
                                 uint32_t stride, uint32_t pad, uint32_t lo, uint16_t* snaked, const float* alpha,
                                 float eps, void* stream) {
    if (!x || !x_strides || !w || !out) return T2H_ERR_NULL;
    if (ci == 0 || co == 0 || kh == 0 || stride == 0 || li == 0) return T2H_ERR_SHAPE;
    // L_out of a transposed conv plus an output padding in [0, stride): the extra last positions take the taps
    // that reach them (the reference's blocks produce stride * L_in outputs, output padding stride % 2)
    const int64_t lo_min = ((int64_t)li - 1) * stride - 2 * (int64_t)pad + kh;
    if ((int64_t)lo < lo_min || (int64_t)lo >= lo_min + stride) return T2H_ERR_SHAPE;
    if ((uint64_t)co * kh > 0x7fffffffu || pad > 0xffffu || li > 0x7fffffffu) return T2H_ERR_SHAPE;
    if (reinterpret_cast<uintptr_t>(w) % 2 != 0) return T2H_ERR_ALIGN;
    for (int i = 0; i < 3; ++i)
        if (x_strides[i] < 0) return T2H_ERR_ARG;
    ConvTArgs a = {};
    a.x = x;
    a.sb = x_strides[0];
    a.sc = x_strides[1];
    a.sl = x_strides[2];
    a.w = reinterpret_cast<const uint8_t*>(w);
    a.bias = bias;
    a.out = out;
    a.ci = ci;
    a.li = li;
    a.co = co;
    a.kh = kh;
    a.stride = stride;
    a.pad = pad;
    a.lo = lo;
    a.snaked = snaked;
    a.alpha = alpha;
    a.eps = eps;
    a.row_bytes = (uint32_t)(((uint64_t)co * kh + 31) / 32 * 34);
    a.n = (uint64_t)batch * lo * co;
    if (a.n == 0) return T2H_OK;
    if (a.n / 256 >= 0x7fffffffu) return T2H_ERR_SHAPE;
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    a.nt = ct_tiles(kh);
    a.halo = (kh - 1) / stride;
    a.i_first = (int32_t)(pad / stride);
    // rows past 2^30 and grids past the launch limits stay on the per-output kernel
    const uint64_t last = (uint64_t)(lo - 1 + pad) / stride;
    if (a.nt != 0 && a.halo <= CT_ROWS / 2 && last < (1u << 30) && batch <= 65535u) {
        const uint32_t useful = CT_ROWS - a.halo;
        const uint32_t mblocks = (uint32_t)((last - a.i_first + useful) / useful);
        const uint32_t nblocks = (a.row_bytes / 34 + a.nt - 1) / a.nt;
        if (nblocks <= 65535u) {
            a.vec = a.sc == 1 && ci % 4 == 0 && a.sl % 4 == 0 && a.sb % 4 == 0 &&
                    (reinterpret_cast<uintptr_t>(x) & 15) == 0;
            hipLaunchKernelGGL(conv_transpose1d_tile_kernel, dim3(mblocks, nblocks, batch), dim3(a.nt * 64), 0, s, a);
            T2H_LAUNCH_CHECK();
            return T2H_OK;
        }
    }
    hipLaunchKernelGGL(conv_transpose1d_q8_0_kernel, dim3((uint32_t)((a.n + 255) / 256)), dim3(256), 0, s, a);
    T2H_LAUNCH_CHECK();
    return T2H_OK;
}

}  // namespace t2h

extern "C" int t2h_conv_transpose1d_q8_0(const float* x, const int64_t* x_strides, const void* w, const float* bias,
                                         float* out, uint32_t batch, uint32_t ci, uint32_t li, uint32_t co,
                                         uint32_t kh, uint32_t stride, uint32_t pad, uint32_t lo, void* stream) {
    return t2h::conv_transpose1d_q8_0_launch(x, x_strides, w, bias, out, batch, ci, li, co, kh, stride, pad, lo,
                                             nullptr, nullptr, 0.0f, stream);
}
