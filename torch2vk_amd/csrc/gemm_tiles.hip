// Matrix-core GEMM for few rows: small tiles in one pass.
//
//   C[M, N] = A[M, K] . deq(W[N, K])^T, the operands, epilogues and rounding of gemm_q_kernel
//
// A prompt of some hundred tokens or an utterance's encoder frames make grids of 4 to 100 tiles of 128 x 256, so
// gemm_q_kernel splits K over blocks there, writes fp32 partials and sums them in a second launch.  Here the tiles are small
// enough to fill the chip in one launch: groups of waves split K inside a block and add their tiles in LDS, and 2
// or 4 register stages of 128 K are in flight per group, with one stage in LDS (two of any tile exceed its 160 KB).
// What bounds a block is the chain of its stages (loads, conversion, LDS, barrier, products) at two waves a SIMD, and
// idle CUs the launch: counters over the shapes below show the matrix cores busy 1 to 6 %, LDS 3 to 19 % and waves
// waiting 29 to 47 % of their cycles.  Measured against the split-K pair (us, weights not in cache): 128 rows, Q4_K:
// K 1024 N 4096 20.7 -> 7.4; K 2048 N 1024 with residual 15.1 -> 9.3; gate|up K 1024 N 2 x 3072 22.8 -> 9.4; Q6_K K 3072
// N 1024 20.5 -> 16.9; 520 rows, Q8_0: K 896 N 2688 26.4 -> 12.9; K 3584 N 896 21.8 -> 17.3.
#include "gemm_formats.h"

namespace t2h {

constexpr int GT_BK = 128;
constexpr int GT_ROW = GT_BK + 8;  // LDS row: 16-byte reads of 16 consecutive rows hit 16 distinct 4-bank groups

// The block's tile, M fastest, so the M tiles that share weight rows share an L2.
__device__ __forceinline__ void gt_tile_of(const GemmArgs& a, uint32_t& tile_m, uint32_t& tile_n) {
    const uint32_t i = xcd_run(a.tiles_m * a.tiles_n);
    tile_m = i % a.tiles_m;
    tile_n = i / a.tiles_m;
}

template <class F, int EPI, int WM, int MI, int WN, int KS>
__global__ __launch_bounds__(64 * WM * WN * KS) void gemm_tile_kernel(const GemmArgs a) {
    constexpr bool GATED = EPI == GQEPI_SWIGLU;
    constexpr int GT = 64 * WM * WN, NT = GT * KS;
    constexpr int BM = 32 * WM * MI, BN = 32 * WN;  // a wave: MI x 1 MFMA tiles
    constexpr int AT = BM * (GT_BK / 8) / GT;   // 16-B A chunks per thread and stage
    constexpr int WT = BN * (GT_BK / 32) / GT;  // 32-value weight conversions per thread and stage
    static_assert(AT >= 1 && WT >= 1, "tile too small for its threads");
    constexpr int BUF = (BM + BN) * GT_ROW;
    constexpr int TS = BN + 8;                  // row of the fp32 result tile
    constexpr int LDS_BYTES = KS * BUF * 2;
    static_assert(KS * BM * TS * 4 <= LDS_BYTES, "the result tiles reuse the stage buffers");
    __shared__ __align__(16) uint8_t lds_raw[LDS_BYTES];

    uint32_t tile_m, tile_n;
    gt_tile_of(a, tile_m, tile_n);
    const uint32_t m0 = tile_m * BM, n0 = tile_n * BN;
    const uint32_t tid = threadIdx.x;
    const uint32_t kg = __builtin_amdgcn_readfirstlane(tid / GT);  // K group of this wave
    const uint32_t t = tid % GT;
    const int lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int wm = wave / WN, wn = wave % WN;
    uint16_t* lds = reinterpret_cast<uint16_t*>(lds_raw) + kg * BUF;

    const uint32_t KT = (a.k + GT_BK - 1) / GT_BK;      // stages; group kg takes kg, kg + KS, ...
    const uint32_t NST = (KT + KS - 1) / KS;
    const uint16_t* arow[AT];
    const uint8_t* wrow[WT];
#pragma unroll
    for (int i = 0; i < AT; ++i) arow[i] = a.a + (size_t)min(m0 + (t + GT * i) / 16, a.m - 1) * a.k;
#pragma unroll
    for (int i = 0; i < WT; ++i) wrow[i] = gemm_w_row<GATED>(a, n0, (t + GT * i) / 4);
    const uint32_t ach = (t % 16) * 8;  // GT is a multiple of 16: the same chunk and quarter for every i
    const uint32_t wk0 = 64 * ((t & 3) >> 1), wh = t & 1;

    struct Stage {
        uint4 ra[AT];
        typename F::Raw rw[WT];
    };
    constexpr int RING = NT >= 1024 || sizeof(Stage) > 160 ? 2 : 4;
    Stage st[RING];
    // Stages past the end re-read the last one (never multiplied; no branch around loads).  The half of a last stage past K reads its
    // first half again and is stored as zeros.
    auto load_stage = [&](uint32_t s, Stage& r) {
        const uint32_t k0 = min(s * KS + kg, KT - 1) * GT_BK;
        const uint32_t ka = k0 + ach < a.k ? k0 + ach : k0;
#pragma unroll
        for (int i = 0; i < AT; ++i) r.ra[i] = load_u4(arow[i] + ka);
#pragma unroll
        for (int i = 0; i < WT; ++i) F::load(wrow[i], a.w_blocks, k0 + wk0, wh, r.rw[i]);
    };
    auto store_stage = [&](uint32_t s, const Stage& r, uint16_t* buf) {
        const uint32_t k0 = min(s * KS + kg, KT - 1) * GT_BK;
        const bool a_in = k0 + ach < a.k;
#pragma unroll
        for (int i = 0; i < AT; ++i)
            *reinterpret_cast<uint4*>(&buf[((t + GT * i) / 16) * GT_ROW + ach]) =
                a_in ? r.ra[i] : make_uint4(0u, 0u, 0u, 0u);
#pragma unroll
        for (int i = 0; i < WT; ++i)
            store_w<F>(r.rw[i], k0 + wk0, wh, &buf[(BM + (t + GT * i) / 4) * GT_ROW + 32 * (t & 3)]);
    };

    f32x16_t acc[MI];
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[i][e] = 0.0f;
    const int r32 = lane & 31, h = lane >> 5;
    const uint32_t off_a = (wm * 32 * MI + r32) * GT_ROW + 8 * h, off_w = (BM + wn * 32 + r32) * GT_ROW + 8 * h;
    auto mma_stage = [&](uint32_t s, const uint16_t* buf) {
        if (s * KS + kg >= KT) return;  // wave-uniform
#pragma unroll
        for (int kk = 0; kk < GT_BK; kk += 16) {
            const bf16x8_t fb = *reinterpret_cast<const bf16x8_t*>(buf + off_w + kk);
#pragma unroll
            for (int i = 0; i < MI; ++i) {
                const bf16x8_t fa = *reinterpret_cast<const bf16x8_t*>(buf + off_a + 32 * i * GT_ROW + kk);
                acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa, fb, acc[i], 0, 0, 0);
            }
        }
    };

#pragma unroll
    for (int i = 0; i < RING; ++i)
        load_stage(i, st[i]);
    for (uint32_t s0 = 0; s0 < NST; s0 += RING) {
#pragma unroll
        for (int i = 0; i < RING; ++i) {
            const uint32_t s = s0 + i;
            if (s >= NST) break;  // block-uniform
            store_stage(s, st[i], lds);
            load_stage(s + RING, st[i]);
            __syncthreads();
            mma_stage(s, lds);
            __syncthreads();
        }
    }

    // results through LDS: the K groups' tiles are added there and rows leave in 16-byte pieces
    float* tile = reinterpret_cast<float*>(lds_raw);
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int e = 0; e < 16; ++e)
            tile[(kg * BM + (wm * MI + i) * 32 + 8 * (e >> 2) + 4 * h + (e & 3)) * TS + wn * 32 + r32] = acc[i][e];
    __syncthreads();
    auto sum4 = [&](uint32_t row, uint32_t col) {
        float4 v = *reinterpret_cast<const float4*>(&tile[row * TS + col]);
#pragma unroll
        for (int p = 1; p < KS; ++p) {
            const float4 u = *reinterpret_cast<const float4*>(&tile[(p * BM + row) * TS + col]);
            v.x += u.x;
            v.y += u.y;
            v.z += u.z;
            v.w += u.w;
        }
        return v;
    };
    if constexpr (EPI == GQEPI_SWIGLU) {
        constexpr int G = BN / 8;  // groups of 4 features per row
#pragma unroll
        for (uint32_t i = 0; i < BM * G; i += NT) {
            const uint32_t idx = i + tid, row = idx / G, g = idx % G;
            if (BM * G % NT != 0 && idx >= BM * G) break;
            const uint32_t f = n0 / 2 + (g / 8) * 32 + (g % 8) * 4, c = (g / 8) * 64 + (g % 8) * 4;
            if (m0 + row >= a.m || f >= a.n_ff) continue;
            const float4 gv = sum4(row, c), uv = sum4(row, c + 32);
            const float gs[4] = {gv.x, gv.y, gv.z, gv.w}, us[4] = {uv.x, uv.y, uv.z, uv.w};
            float o[4];
#pragma unroll
            for (int j = 0; j < 4; ++j)
                o[j] = gs[j] * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-1.4426950408889634f * gs[j])) * us[j];
            uint16_t* dst = reinterpret_cast<uint16_t*>(a.c) + (size_t)(m0 + row) * a.n_ff + f;
            if (a.vec) {
                *reinterpret_cast<uint2*>(dst) = make_uint2(pack_bf16x2(o[0], o[1]), pack_bf16x2(o[2], o[3]));
            } else {
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    if (f + j < a.n_ff) dst[j] = (uint16_t)f32_to_bf16_bits(o[j]);
            }
        }
        return;
    }
    constexpr int G = BN / 4;
#pragma unroll
    for (uint32_t i = 0; i < BM * G; i += NT) {
        const uint32_t idx = i + tid, row = idx / G, c = idx % G * 4, col = n0 + c;
        if (BM * G % NT != 0 && idx >= BM * G) break;
        if (m0 + row >= a.m || col >= a.n) continue;
        const size_t at = (size_t)(m0 + row) * a.n + col;
        const uint32_t cols = min(4u, a.n - col);
        float4 rv = make_float4(0.f, 0.f, 0.f, 0.f);
        float rs[4] = {0.f, 0.f, 0.f, 0.f}, bs[4] = {0.f, 0.f, 0.f, 0.f};
        if (a.vec) {
            if constexpr (EPI == GQEPI_RESID) rv = *reinterpret_cast<const float4*>(a.residual + at);
            rs[0] = rv.x;
            rs[1] = rv.y;
            rs[2] = rv.z;
            rs[3] = rv.w;
        } else if constexpr (EPI == GQEPI_RESID) {
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if ((uint32_t)j < cols) rs[j] = a.residual[at + j];
        }
        if (a.bias) {
#pragma unroll
            for (int j = 0; j < 4; ++j) bs[j] = a.bias[min(col + j, a.n - 1)];
        }
        const float4 v = sum4(row, c);
        float o[4] = {v.x + bs[0], v.y + bs[1], v.z + bs[2], v.w + bs[3]};
        if (a.act == GQACT_GELU) {
#pragma unroll
            for (int j = 0; j < 4; ++j) o[j] = gelu_erf(o[j]);
        }
        if constexpr (EPI == GQEPI_RESID) {
#pragma unroll
            for (int j = 0; j < 4; ++j) o[j] = rs[j] + o[j];
        }
        if (a.vec) {
            if constexpr (EPI == GQEPI_BF16)
                *reinterpret_cast<uint2*>(reinterpret_cast<uint16_t*>(a.c) + at) =
                    make_uint2(pack_bf16x2(o[0], o[1]), pack_bf16x2(o[2], o[3]));
            else
                *reinterpret_cast<float4*>(reinterpret_cast<float*>(a.c) + at) = make_float4(o[0], o[1], o[2], o[3]);
        } else {
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if ((uint32_t)j < cols) {
                    if constexpr (EPI == GQEPI_BF16)
                        reinterpret_cast<uint16_t*>(a.c)[at + j] = (uint16_t)f32_to_bf16_bits(o[j]);
                    else
                        reinterpret_cast<float*>(a.c)[at + j] = o[j];
                }
        }
    }
}

template <class F, int EPI, int WM, int MI, int WN, int KS>
static int gt_launch(GemmArgs& a, hipStream_t s) {
    a.tiles_m = (a.m + 32 * WM * MI - 1) / (32 * WM * MI);
    a.tiles_n = (a.n + 32 * WN - 1) / (32 * WN);
    hipLaunchKernelGGL((gemm_tile_kernel<F, EPI, WM, MI, WN, KS>), dim3(a.tiles_m * a.tiles_n), dim3(64 * WM * WN * KS),
                       0, s, a);
    T2H_LAUNCH_CHECK();
    return T2H_OK;
}

// tile 0: 32 x 32 outputs, K over 8 groups of waves; 1: 64 x 32 over 4; 2: 64 x 64 over 4; 3: 128 x 64 over 2.  Each
// block fills a CU's LDS (104 to 139 KB).  The gated form needs whole 64-column groups.
template <class F, int EPI>
static int gt_dispatch(GemmArgs& a, uint32_t tile, hipStream_t s) {
    if constexpr (EPI != GQEPI_SWIGLU) {
        if (tile == 0) return gt_launch<F, EPI, 1, 1, 1, 8>(a, s);
        if (tile == 1) return gt_launch<F, EPI, 2, 1, 1, 4>(a, s);
    }
    if (tile == 2) return gt_launch<F, EPI, 2, 1, 2, 4>(a, s);
    if (tile == 3) return gt_launch<F, EPI, 2, 2, 2, 2>(a, s);
    return T2H_ERR_ARG;
}

template <class F>
static int gemm_tiles_launch(const void* x, const void* w, const void* w_up, const float* bias, int act, void* y,
                             int out_dtype, const float* residual, uint32_t m, uint32_t k, uint32_t n, uint32_t w_k,
                             uint32_t tile, void* stream) {
    if (!x || !w || !y) return T2H_ERR_NULL;
    const bool gated = w_up != nullptr;
    if (k == 0 || k % 64 != 0) return T2H_ERR_SHAPE;
    if (w_k == 0 || w_k > k || w_k % F::BLOCK_VALUES != 0) return T2H_ERR_SHAPE;
    if ((F::BLOCK_VALUES == 256 || gated) && w_k != k) return T2H_ERR_SHAPE;
    if (act != GQACT_NONE && act != GQACT_GELU) return T2H_ERR_ARG;
    if (gated && (bias || act != GQACT_NONE || residual || out_dtype != T2H_DTYPE_BF16)) return T2H_ERR_ARG;
    if (residual && out_dtype != T2H_DTYPE_F32) return T2H_ERR_DTYPE;
    if (out_dtype != T2H_DTYPE_F32 && out_dtype != T2H_DTYPE_BF16) return T2H_ERR_DTYPE;
    if ((reinterpret_cast<uintptr_t>(x) & 15) != 0) return T2H_ERR_ALIGN;
    if (((reinterpret_cast<uintptr_t>(w) | reinterpret_cast<uintptr_t>(w_up)) & (F::ALIGN - 1)) != 0)
        return T2H_ERR_ALIGN;
    if (n > 0x3fffffffu || (uint64_t)(m / 32 + 1) * (n / 32 + 1) > 0x7fffffffu) return T2H_ERR_SHAPE;
    if (m == 0 || n == 0) return T2H_OK;
    GemmArgs a = {};
    a.a = reinterpret_cast<const uint16_t*>(x);
    a.w = reinterpret_cast<const uint8_t*>(w);
    a.w_up = reinterpret_cast<const uint8_t*>(w_up);
    a.c = y;
    a.residual = residual;
    a.bias = bias;
    a.act = act;
    a.m = m;
    a.n = gated ? 2 * n : n;
    a.n_ff = gated ? n : 0;
    a.k = k;
    a.w_blocks = w_k / F::BLOCK_VALUES;
    a.row_bytes = a.w_blocks * F::BLOCK_BYTES;
    const uintptr_t out_align = out_dtype == T2H_DTYPE_BF16 ? 7 : 15;
    a.vec = n % 4 == 0 && (reinterpret_cast<uintptr_t>(y) & out_align) == 0 &&
            (reinterpret_cast<uintptr_t>(residual) & 15) == 0;
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    if (gated) return gt_dispatch<F, GQEPI_SWIGLU>(a, tile, s);
    if (residual) return gt_dispatch<F, GQEPI_RESID>(a, tile, s);
    if (out_dtype == T2H_DTYPE_F32) return gt_dispatch<F, GQEPI_F32>(a, tile, s);
    return gt_dispatch<F, GQEPI_BF16>(a, tile, s);
}

}  // namespace t2h

using namespace t2h;

extern "C" int t2h_gemm_tiles(int wtype, const void* x, const void* w, const void* w_up, const float* bias, int act,
                              void* y, int out_dtype, const float* residual, uint32_t m, uint32_t k, uint32_t n,
                              uint32_t w_k, uint32_t tile, void* stream) {
    switch (wtype) {
        case T2H_WTYPE_Q8_0:
            return gemm_tiles_launch<GemmQ80>(x, w, w_up, bias, act, y, out_dtype, residual, m, k, n, w_k, tile, stream);
        case T2H_WTYPE_Q4_K:
            return gemm_tiles_launch<GemmQ4K>(x, w, w_up, bias, act, y, out_dtype, residual, m, k, n, w_k, tile, stream);
        case T2H_WTYPE_Q6_K:
            return gemm_tiles_launch<GemmQ6K>(x, w, w_up, bias, act, y, out_dtype, residual, m, k, n, w_k, tile, stream);
        case T2H_WTYPE_BF16:
            return gemm_tiles_launch<GemmBF16>(x, w, w_up, bias, act, y, out_dtype, residual, m, k, n, w_k, tile, stream);
        default: return T2H_ERR_DTYPE;
    }
}
