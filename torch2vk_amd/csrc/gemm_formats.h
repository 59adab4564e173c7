// Operands of the matrix-core GEMMs: arguments, weight rows and the formats that turn packed blocks into bf16.
#pragma once

#include "common.h"

namespace t2h {

// GQEPI_GATED_F32: the SwiGLU form's gate | up tile columns written as fp32 products (split-K partials).
enum GemmEpilogue { GQEPI_F32 = 0, GQEPI_BF16 = 1, GQEPI_RESID = 2, GQEPI_SWIGLU = 3, GQEPI_GATED_F32 = 4 };

enum GemmAct { GQACT_NONE = 0, GQACT_GELU = 1 };

struct GemmArgs {
    const uint16_t* a;     // bf16 [M, K]
    const uint8_t* w;      // packed rows [N, row_bytes]
    void* c;               // [M, N] fp32 or bf16
    const float* residual; // GQEPI_RESID: fp32 [M, N] (may alias c)
    const float* bias;     // fp32 [N] or null
    int act;               // GemmAct, applied after the bias and before the residual
    uint32_t m, n, k;
    uint32_t row_bytes;
    uint32_t w_blocks;     // quant blocks per weight row; K columns past them multiply zeros
    uint32_t tiles_m, tiles_n;
    const uint8_t* w_up;   // GQEPI_SWIGLU: up rows (w holds the gate rows)
    uint32_t n_ff;         // GQEPI_SWIGLU: features; n = 2 n_ff
    uint32_t split_stages; // split-K: 64-wide K stages per split (blockIdx.y), split s writing its fp32
                           // products to c + s m n; 0: the whole K range in one pass
    uint32_t vec;          // gemm_tile_kernel: rows of C and the residual can be accessed 4 values at a time
};

// The tile of `total` that this block computes: blocks are dealt round-robin to the 8 XCDs, and each XCD takes a
// contiguous run of tiles.
__device__ __forceinline__ uint32_t xcd_run(uint32_t total) {
    const uint32_t xcd = blockIdx.x % 8;
    return xcd * (total / 8) + min(xcd, total % 8) + blockIdx.x / 8;
}

// Packed row of B-tile row r (0..255) of the tile at n0.  Plain: weight row
// n0 + r.  Gated (SwiGLU): each wave's 64 columns are 32 gate rows then the 32
// up rows of the same features, so the epilogue finds g and u in one lane:
// feature n0/2 + 32 (r / 64) + r % 32, from gate when (r / 32) is even.
template <bool GATED>
__device__ __forceinline__ const uint8_t* gemm_w_row(const GemmArgs& a, uint32_t n0, uint32_t r) {
    if constexpr (GATED) {
        uint32_t f = n0 / 2 + (r >> 6) * 32 + (r & 31);
        f = f < a.n_ff ? f : a.n_ff - 1;
        return ((r >> 5) & 1 ? a.w_up : a.w) + (size_t)f * a.row_bytes;
    } else {
        uint32_t row = n0 + r;
        row = row < a.n ? row : a.n - 1;
        return a.w + (size_t)row * a.row_bytes;
    }
}

// GELU of the bias + GELU epilogues (gelu_as: erf by Abramowitz-Stegun 7.1.26, as the reference's GELU)
__device__ __forceinline__ float gelu_erf(float v) { return gelu_as(v); }

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));

// ------------------------------------------------------ weight formats ----

// A format converts 32 values of a weight row at a time: values k0 + 32 h .. + 31, k0 a multiple of 64 (a 64-wide K
// stage, or half of a wider one), h 0 or 1.  load() issues their loads into Raw and convert() makes the 32 bf16
// values, packed in pairs.

// Q8_0: block k0 / 32 + h.
struct GemmQ80 {
    static constexpr int BLOCK_VALUES = 32;
    static constexpr int BLOCK_BYTES = 34;
    static constexpr int ALIGN = 2;
    // MFMA step after which the next stage's A is stored, at 128- and at 256-row tiles (measured)
    static constexpr int STORE_STEP = 2, STORE_STEP_256 = 2;
    struct Raw {
        uint4 q0, q1;
        uint32_t d;
        bool inside;  // false: a block past the row's end, dequantised as zeros
    };
    __device__ static __forceinline__ void load(const uint8_t* row, uint32_t w_blocks, uint32_t k0, uint32_t h, Raw& r) {
        // a stage past the row's last block (K padded to the 64-wide stage) reads
        // the last block again with a zero scale
        const uint32_t blk = k0 / 32 + h;
        const bool inside = blk < w_blocks;
        const uint8_t* p = row + (size_t)(inside ? blk : w_blocks - 1) * 34;
        r.d = load_u16(p);  // unconditional (p is always inside the row) and not
        r.inside = inside;  // selected here, so nothing waits on the load before its use
        r.q0 = load_u4_ua(p + 2);
        r.q1 = load_u4_ua(p + 18);
    }
    // the block's 32 values as bf16 pairs: d * q, rounded once
    __device__ static __forceinline__ void convert(const Raw& r, uint32_t, uint32_t, uint32_t (&o)[16]) {
        const float d = r.inside ? f16_bits_to_f32(r.d) : 0.0f;
        const uint32_t q[8] = {r.q0.x, r.q0.y, r.q0.z, r.q0.w, r.q1.x, r.q1.y, r.q1.z, r.q1.w};
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            const uint32_t w = q[c];
            const float v0 = d * (float)(int8_t)(w & 0xffu);
            const float v1 = d * (float)(int8_t)((w >> 8) & 0xffu);
            const float v2 = d * (float)(int8_t)((w >> 16) & 0xffu);
            const float v3 = d * (float)(int8_t)(w >> 24);
            o[2 * c] = pack_bf16x2(v0, v1);
            o[2 * c + 1] = pack_bf16x2(v2, v3);
        }
    }
};

// Q4_K: sub-block 2 g + h of superblock k0 / 256, g = (k0 % 256) / 64 its nibble group.
struct GemmQ4K {
    static constexpr int BLOCK_VALUES = 256;
    static constexpr int BLOCK_BYTES = 144;
    static constexpr int ALIGN = 16;
    static constexpr int STORE_STEP = 0, STORE_STEP_256 = 0;
    struct Raw {
        uint4 hdr, q0, q1;
    };
    __device__ static __forceinline__ void load(const uint8_t* row, uint32_t, uint32_t k0, uint32_t, Raw& r) {
        const uint8_t* p = row + (size_t)(k0 / 256) * 144;
        const uint32_t g = (k0 % 256) / 64;
        r.hdr = load_u4(p);
        r.q0 = load_u4(p + 16 + g * 32);
        r.q1 = load_u4(p + 32 + g * 32);
    }
    __device__ static __forceinline__ void convert(const Raw& r, uint32_t k0, uint32_t h, uint32_t (&o)[16]) {
        const uint32_t g = (k0 % 256) / 64;
        const uint32_t j = 2 * g + h;  // sub-block
        const float d = f16_bits_to_f32(r.hdr.x & 0xffffu);
        const float dmin = f16_bits_to_f32(r.hdr.x >> 16);
        // 6-bit scale/min of sub-block j (12 bytes at 4..15: hdr.y, hdr.z, hdr.w)
        const uint8_t sb[12] = {
            (uint8_t)r.hdr.y, (uint8_t)(r.hdr.y >> 8), (uint8_t)(r.hdr.y >> 16), (uint8_t)(r.hdr.y >> 24),
            (uint8_t)r.hdr.z, (uint8_t)(r.hdr.z >> 8), (uint8_t)(r.hdr.z >> 16), (uint8_t)(r.hdr.z >> 24),
            (uint8_t)r.hdr.w, (uint8_t)(r.hdr.w >> 8), (uint8_t)(r.hdr.w >> 16), (uint8_t)(r.hdr.w >> 24)};
        uint32_t sc, mn;
        if (j < 4) {
            sc = sb[j] & 63u;
            mn = sb[j + 4] & 63u;
        } else {
            sc = (sb[j + 4] & 0xfu) | ((sb[j - 4] >> 6) << 4);
            mn = (sb[j + 4] >> 4) | ((sb[j] >> 6) << 4);
        }
        const float ds = d * (float)sc;
        const float dm = dmin * (float)mn;
        const uint32_t q[8] = {r.q0.x, r.q0.y, r.q0.z, r.q0.w, r.q1.x, r.q1.y, r.q1.z, r.q1.w};
        const int sh = (int)h * 4;  // low nibbles: sub-block 2g, high: 2g+1
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            const uint32_t w = q[c] >> sh;
            const float v0 = ds * (float)(w & 0xfu) - dm;
            const float v1 = ds * (float)((w >> 8) & 0xfu) - dm;
            const float v2 = ds * (float)((w >> 16) & 0xfu) - dm;
            const float v3 = ds * (float)((w >> 24) & 0xfu) - dm;
            o[2 * c] = pack_bf16x2(v0, v1);
            o[2 * c + 1] = pack_bf16x2(v2, v3);
        }
    }
};

// Q6_K: part p = (k0 % 128) / 32 + h of half H = (k0 % 256) / 128 of superblock k0 / 256 (values 128 H + 32 p + l,
// l < 32):  value = (d * sc[8h + 2p + l/16]) * (q - 32), with that half as h,
//   q = (ql[64h + 32(p&1) + l] >> 4(p>>1) & 15) | ((qh[32h + l] >> 2p) & 3) << 4.
// Blocks are 210 B, so only halfword aligned: the 16-B loads are unaligned.
struct GemmQ6K {
    static constexpr int BLOCK_VALUES = 256;
    static constexpr int BLOCK_BYTES = 210;
    static constexpr int ALIGN = 2;
    static constexpr int STORE_STEP = 0, STORE_STEP_256 = 1;  // at 256 rows, 0 spills registers
    struct Raw {
        uint4 ql0, ql1, qh0, qh1;
        uint32_t sc, d;
    };
    __device__ static __forceinline__ void load(const uint8_t* row, uint32_t, uint32_t k0, uint32_t h32, Raw& r) {
        const uint8_t* blk = row + (size_t)(k0 / 256) * 210;
        const uint32_t h = (k0 % 256) / 128;
        const uint32_t p = (k0 % 128) / 32 + h32;
        const uint8_t* ql = blk + 64 * h + 32 * (p & 1);
        r.ql0 = load_u4_ua(ql);
        r.ql1 = load_u4_ua(ql + 16);
        r.qh0 = load_u4_ua(blk + 128 + 32 * h);
        r.qh1 = load_u4_ua(blk + 128 + 32 * h + 16);
        r.sc = load_u16(blk + 192 + 8 * h + 2 * p);
        r.d = load_u16(blk + 208);
    }
    __device__ static __forceinline__ void convert(const Raw& r, uint32_t k0, uint32_t h32, uint32_t (&o)[16]) {
        const uint32_t p = (k0 % 128) / 32 + h32;
        const uint32_t shl = 4 * (p >> 1), shh = 2 * p;
        const float d = f16_bits_to_f32(r.d);
        const float a0 = d * (float)(int8_t)(r.sc & 0xffu);  // values l < 16
        const float a1 = d * (float)(int8_t)(r.sc >> 8);     // values l >= 16
        const uint32_t ql[8] = {r.ql0.x, r.ql0.y, r.ql0.z, r.ql0.w, r.ql1.x, r.ql1.y, r.ql1.z, r.ql1.w};
        const uint32_t qh[8] = {r.qh0.x, r.qh0.y, r.qh0.z, r.qh0.w, r.qh1.x, r.qh1.y, r.qh1.z, r.qh1.w};
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            const float a = c < 4 ? a0 : a1;
            float v[4];
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                const uint32_t q = ((ql[c] >> (8 * b + shl)) & 15u) | (((qh[c] >> (8 * b + shh)) & 3u) << 4);
                v[b] = a * (float)((int)q - 32);
            }
            o[2 * c] = pack_bf16x2(v[0], v[1]);
            o[2 * c + 1] = pack_bf16x2(v[2], v[3]);
        }
    }
};

// bf16 rows (GGUF BF16): no dequantisation, the values as they are.  Weights a prefill pass dequantised once
// (t2h_dequantize_bf16), or a model kept in bf16.
struct GemmBF16 {
    static constexpr int BLOCK_VALUES = 64;
    static constexpr int BLOCK_BYTES = 128;
    static constexpr int ALIGN = 16;
    // measured at M 16384: after step 0 fastest (1: 2-3 % slower, 2: 3 %); tile groups of 8 down M as the
    // other formats (4 and 16: 1-2 % slower)
    static constexpr int STORE_STEP = 0, STORE_STEP_256 = 0;
    struct Raw {
        uint4 v[4];
        bool inside;  // false: a stage past the row's end, stored as zeros
    };
    __device__ static __forceinline__ void load(const uint8_t* row, uint32_t w_blocks, uint32_t k0, uint32_t h, Raw& r) {
        const uint32_t blk = k0 / 64;
        r.inside = blk < w_blocks;
        const uint8_t* p = row + (size_t)(r.inside ? blk : w_blocks - 1) * 128 + h * 64;
#pragma unroll
        for (int i = 0; i < 4; ++i) r.v[i] = load_u4(p + 16 * i);
    }
    __device__ static __forceinline__ void convert(const Raw& r, uint32_t, uint32_t, uint32_t (&o)[16]) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            o[4 * i] = r.inside ? r.v[i].x : 0u;
            o[4 * i + 1] = r.inside ? r.v[i].y : 0u;
            o[4 * i + 2] = r.inside ? r.v[i].z : 0u;
            o[4 * i + 3] = r.inside ? r.v[i].w : 0u;
        }
    }
};

// 32 converted values to LDS.
template <class F>
__device__ __forceinline__ void store_w(const typename F::Raw& r, uint32_t k0, uint32_t h, uint16_t* dst) {
    uint32_t o[16];
    F::convert(r, k0, h, o);
#pragma unroll
    for (int i = 0; i < 4; ++i)
        *reinterpret_cast<uint4*>(dst + 8 * i) = make_uint4(o[4 * i], o[4 * i + 1], o[4 * i + 2], o[4 * i + 3]);
}

}  // namespace t2h
