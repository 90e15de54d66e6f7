// Instantiations of the f32 MFMA GEMM (multi-row passes, DiT linears, grouped convolutions) and the
// attention-partials merge.
#include <atomic>
#include <algorithm>

#include "vh_gemm_epi.hpp"
#include "vh_launch.hpp"

namespace vh {

// Merge of the kAttnMaxSplits attention partials of m rows into ao [m][heads * hd] (the PRO_ATTN prologue of the
// GEMV, as its own pass before a GEMM). grid (heads, m), block hd.
__global__ __launch_bounds__(128) void k_attn_merge(AttnPartials P, float *ao) {
    const int h = blockIdx.x, i = blockIdx.y, e = threadIdx.x;
    const int64_t base = (int64_t(i) * P.heads + h) * kAttnMaxSplits;
    float mx = -INFINITY;
#pragma unroll
    for (int q = 0; q < kAttnMaxSplits; ++q) mx = fmaxf(mx, P.pm[base + q]);
    float L = 0.f, O = 0.f;
#pragma unroll
    for (int q = 0; q < kAttnMaxSplits; ++q) {
        const float pmq = P.pm[base + q];
        const float wq = pmq == -INFINITY ? 0.f : expf(pmq - mx);
        L = fmaf(wq, P.pl[base + q], L);
        O = fmaf(wq, P.po[(base + q) * P.hd + e], O);
    }
    ao[int64_t(i) * P.heads * P.hd + h * P.hd + e] = O * (1.0f / L);
}

template <int WT, int EPI, int ASRC, int T>
static hipError_t gemm_run(const uint8_t *w, const float *scale, const float *A, const GemmArgs &g, int groups, hipStream_t s) {
    constexpr int B = 32 * T;
    const dim3 grid((g.n + B - 1) / B, (g.m + B - 1) / B, groups);
    return launch(k_gemm_f32<WT, EPI, ASRC, T, T>, grid, dim3(256), 0, s, w, scale, A, g);
}

// F32 weights: the three-product split-f16 kernel (z: groups of a grouped conv, or K slices when g.kchunk is set).
template <int EPI, int ASRC>
static hipError_t x3_run(const uint8_t *w, const float *A, const GemmArgs &g, int z, hipStream_t s) {
    const dim3 grid((g.n + 63) / 64, (g.m + 63) / 64, z);
    return launch(k_gemm_x3<EPI, ASRC>, grid, dim3(256), 0, s, w, A, g);
}

// F32 weights: the split kernel, or k_gemm_f32 (f32 matrix cores, one product) when the weights are too large for
// its scaled f16 halves (g.f32_wide).
template <int EPI, int ASRC>
static hipError_t f32w_run(const uint8_t *w, const float *A, const GemmArgs &g, int z, hipStream_t s) {
    if (g.f32_wide) return gemm_run<WT_F32, EPI, ASRC, 2>(w, nullptr, A, g, z, s);
    return x3_run<EPI, ASRC>(w, A, g, z, s);
}

template <int WT, int EPI, int TM, int TN>
static hipError_t gemm_run_h16(const uint8_t *w, const float *scale, const float *A, const GemmArgs &g, hipStream_t s) {
    constexpr int BM = 32 * TM, BN = 32 * TN;
    const dim3 grid((g.n + BN - 1) / BN, (g.m + BM - 1) / BM, g.kchunk ? (g.K + g.kchunk - 1) / g.kchunk : 1);
    // K steps of 64 throughout, A rows 16-byte aligned, and a tile's byte offsets within 32 bits: the buffered pipeline
    if (TM == 2 && TN == 2 && g.K % 64 == 0 && g.kchunk % 64 == 0 && g.lda % 4 == 0 && int64_t(64) * g.lda * 4 <= INT32_MAX &&
        int64_t(64) * g.K * 2 <= INT32_MAX)
        return launch(k_gemm_h16b<WT, EPI>, grid, dim3(256), 0, s, w, scale, A, g);
    return launch(k_gemm_h16<WT, EPI, TM, TN, 64>, grid, dim3(256), 0, s, w, scale, A, g);
}

// Split K for a grid of 64 x 64 tiles too small to fill the CUs with a long K (prefill down projections, small
// matrices): up to 8 slices of K (32 for grids under 64 tiles), each a multiple of 64 columns, summed in order by the
// reduce pass. Slices are
// added until the launch has about kSplitTargetBlocks blocks (two per CU: measured faster than one per CU on the
// 512-row prefill shapes even with the larger reduce).
constexpr int64_t kSplitTargetBlocks = 512;
constexpr int64_t kSplitMaxSmall = 32;
constexpr int64_t kSplitTargetOneRow = 1024;
// The K slices for a split of g (64 x 64 tiles): 0 when the tiles already fill the CUs, K is short or the workspace
// is too small; else the slice count, with *kchunk the slice width (a multiple of 64). A grid of fewer than 192
// tiles gets enough slices for about kSplitTargetBlocks blocks, at most 8, or at most kSplitMaxSmall for grids of
// under 64 tiles (few-row passes over large weights, such as a streaming codec frame's convolutions, whose tiles
// would otherwise each stream megabytes of weights) when their partials fit the workspace.
static int split_plan(const GemmArgs &g, int *kchunk) {
    const int64_t blocks = int64_t((g.n + 63) / 64) * ((g.m + 63) / 64);
    // one row tile: every tile streams its own columns of the weights, so such grids take slices up to about
    // kSplitTargetOneRow blocks (a streaming codec frame's transposed convolutions and pointwise products)
    const bool one_row = g.m <= 64 && blocks < kSplitTargetOneRow / 2;
    if (!g.ws || (blocks >= 192 && !one_row) || g.K < 512) return 0;
    const int64_t target = one_row ? kSplitTargetOneRow : kSplitTargetBlocks;
    const int64_t want = (target + blocks - 1) / blocks;
    auto plan = [&](int64_t cap) {
        int splits = int(std::min<int64_t>(cap, want));
        *kchunk = ((g.K + splits - 1) / splits + 63) / 64 * 64;
        splits = (g.K + *kchunk - 1) / *kchunk;
        return splits < 2 || int64_t(splits) * g.m * g.n > g.ws_cap ? 0 : splits;
    };
    if (want > 8)
        if (const int splits = plan(kSplitMaxSmall)) return splits;
    return plan(8);
}
template <int WT, int EPI>
static hipError_t gemm_splitk(const uint8_t *w, const float *scale, const float *A, const GemmArgs &g, hipStream_t s, bool *done) {
    *done = false;
    if constexpr (EPI != EPI_STORE && EPI != EPI_ACC && EPI != EPI_GATED_ACC && EPI != EPI_SWIGLU && EPI != EPI_ACC_SNAKE &&
                  EPI != EPI_GELU_ERF) {
        return hipSuccess;
    } else {
        GemmArgs gs = g;
        const int splits = split_plan(g, &gs.kchunk);
        if (!splits) return hipSuccess;
        hipError_t e = gemm_run_h16<WT, EPI_STORE, 2, 2>(w, scale, A, gs, s);
        if (e != hipSuccess) return e;
        *done = true;
        return launch_splitk_reduce<EPI>(g, splits, s);
    }
}

// 64 x 64 block tiles: measured faster than 128 x 128 and 128 x 64 on the DiT and prefill shapes, because more
// blocks per CU hide the global latency of each K step (split K when even these leave the CUs idle). F16 and Q8
// weights take the split-f16 matrix cores.
template <int WT, int EPI>
static hipError_t gemm_tile(const uint8_t *w, const float *scale, const float *A, const GemmArgs &g, hipStream_t s) {
    if constexpr (WT == WT_F16 || WT == WT_Q8) {
        bool split = false;
        hipError_t e = gemm_splitk<WT, EPI>(w, scale, A, g, s, &split);
        if (e != hipSuccess || split) return e;
        return gemm_run_h16<WT, EPI, 2, 2>(w, scale, A, g, s);
    } else {
        if constexpr (EPI == EPI_STORE || EPI == EPI_ACC || EPI == EPI_GATED_ACC || EPI == EPI_SWIGLU || EPI == EPI_ACC_SNAKE ||
                      EPI == EPI_GELU_ERF) {
            GemmArgs gs = g;  // the same K slices (few-row passes over f32 / bf16 weights)
            const int splits = split_plan(g, &gs.kchunk);
            if (splits) {
                hipError_t e = WT == WT_F32 ? f32w_run<EPI_STORE, ASRC_ROWS>(w, A, gs, splits, s)
                                            : gemm_run<WT, EPI_STORE, ASRC_ROWS, 2>(w, scale, A, gs, splits, s);
                return e != hipSuccess ? e : launch_splitk_reduce<EPI>(g, splits, s);
            }
        }
        if constexpr (WT == WT_F32) return f32w_run<EPI, ASRC_ROWS>(w, A, g, 1, s);
        return gemm_run<WT, EPI, ASRC_ROWS, 2>(w, scale, A, g, 1, s);
    }
}


bool rope_h16_ok(const GemmArgs &g) {
    return g.h16 && g.hd == kQkvHead && g.seq > 0 && g.rope_cols % (2 * g.hd) == 0 && g.m % g.seq == 0 &&
           g.n == g.rope_cols + g.rope_cols / 2 && g.seq_pad >= g.seq && g.seq_pad % 64 == 0;
}

// The operands an epilogue needs beyond y.
static bool gemm_args_ok(int epi, const GemmArgs &g) {
    switch (epi) {
        case EPI_GATED_ACC: return g.gate != nullptr;
        case EPI_ACC_SNAKE: return g.snake_a && g.snake_ib && g.snake_y;
        case EPI_ROPE_H16: return rope_h16_ok(g);
        default: return true;
    }
}
template <int WT>
static hipError_t gemm_epi(int epi, const uint8_t *w, const float *scale, const float *A, const GemmArgs &g, hipStream_t s) {
    switch (epi) {
        case EPI_STORE: return gemm_tile<WT, EPI_STORE>(w, scale, A, g, s);
        case EPI_ACC: return gemm_tile<WT, EPI_ACC>(w, scale, A, g, s);
        case EPI_SWIGLU: return gemm_tile<WT, EPI_SWIGLU>(w, scale, A, g, s);
        case EPI_GATED_ACC: return g.gate ? gemm_tile<WT, EPI_GATED_ACC>(w, scale, A, g, s) : hipErrorInvalidValue;
        case EPI_GELU: return gemm_tile<WT, EPI_GELU>(w, scale, A, g, s);
        case EPI_GELU_ERF: return gemm_tile<WT, EPI_GELU_ERF>(w, scale, A, g, s);
        case EPI_ACC_SNAKE:
            return g.snake_a && g.snake_ib && g.snake_y ? gemm_tile<WT, EPI_ACC_SNAKE>(w, scale, A, g, s) : hipErrorInvalidValue;
        case EPI_ROPE_H16:
            return rope_h16_ok(g) ? gemm_tile<WT, EPI_ROPE_H16>(w, scale, A, g, s) : hipErrorInvalidValue;
        default: return hipErrorInvalidValue;
    }
}

hipError_t launch_gemm(int wt, int epi, const uint8_t *w, const float *scale, const float *A, const GemmArgs &g0, hipStream_t s) {
    GemmArgs g = g0;
    g.status = status_word();
    if (g.m <= 0) return hipSuccess;
    if (g.K % 8 || g.n <= 0 || g.lda % 4) return hipErrorInvalidValue;
    if (epi == EPI_SWIGLU && g.n % 2) return hipErrorInvalidValue;
    if (wt == WT_F32 && g.wx && gemm_args_ok(epi, g)) {
        bool done = false;
        const hipError_t e = launch_gemm_x3p(ASRC_ROWS, epi, A, g, 1, s, &done);
        if (e != hipSuccess || done) return e;
    }
    switch (wt) {
        case WT_F32: return gemm_epi<WT_F32>(epi, w, scale, A, g, s);
        case WT_F16: return gemm_epi<WT_F16>(epi, w, scale, A, g, s);
        case WT_BF16: return gemm_epi<WT_BF16>(epi, w, scale, A, g, s);
        case WT_Q8: return g.K % 32 ? hipErrorInvalidValue : gemm_epi<WT_Q8>(epi, w, scale, A, g, s);
        default: return hipErrorInvalidValue;
    }
}

hipError_t launch_conv_gemm(int epi, const float *w, const float *A, const GemmArgs &g0, int groups, hipStream_t s) {
    GemmArgs g = g0;
    g.status = status_word();
    if (g.m <= 0) return hipSuccess;
    // K: ksize * cig, rounded up to a multiple of 8 with zero weights (the A loader reads zeros there)
    if (g.cig <= 0 || g.cig % 4 || g.ksize <= 0 || g.ksize % 2 == 0 || g.K < g.ksize * g.cig || g.K >= g.ksize * g.cig + 8 ||
        g.K % 8 || g.seq <= 0 || g.lda % 4 || groups <= 0 || g.n <= 0)
        return hipErrorInvalidValue;
    const uint8_t *wb = reinterpret_cast<const uint8_t *>(w);
    if (g.wx) {
        bool done = false;
        const hipError_t e = launch_gemm_x3p(ASRC_CONV, epi, A, g, groups, s, &done);
        if (e != hipSuccess || done) return e;
    }
    if (groups == 1 && (epi == EPI_STORE || epi == EPI_ACC)) {  // one group: K slices in place of groups when idle
        GemmArgs gs = g;
        const int splits = split_plan(g, &gs.kchunk);
        if (splits) {
            hipError_t e = f32w_run<EPI_STORE, ASRC_CONV>(wb, A, gs, splits, s);
            if (e != hipSuccess) return e;
            return epi == EPI_STORE ? launch_splitk_reduce<EPI_STORE>(g, splits, s) : launch_splitk_reduce<EPI_ACC>(g, splits, s);
        }
    }
    if (epi == EPI_MISH) return f32w_run<EPI_MISH, ASRC_CONV>(wb, A, g, groups, s);
    if (epi == EPI_MISH_ACC) return f32w_run<EPI_MISH_ACC, ASRC_CONV>(wb, A, g, groups, s);
    if (epi == EPI_STORE) return f32w_run<EPI_STORE, ASRC_CONV>(wb, A, g, groups, s);
    if (epi == EPI_ACC) return f32w_run<EPI_ACC, ASRC_CONV>(wb, A, g, groups, s);
    return hipErrorInvalidValue;
}

// The codec's streaming convolution: y = W im2col([hist; x]) + bias (qwen3.cpp:102-121), or Snake of it (EPI_SNAKE),
// F32 / F16 / BF16 weights [cout][K cin] on the MFMA GEMMs (f32 weights: three f16 products), split K when the
// 64 x 64 tiles leave the CUs idle.
template <int WT, int EPI>
static hipError_t stream_conv(const uint8_t *w, const float *scale, const float *x, const GemmArgs &g, hipStream_t s) {
    GemmArgs gs = g;
    const int splits = split_plan(g, &gs.kchunk);
    if (splits) {
        hipError_t e = WT == WT_F32 ? f32w_run<EPI_STORE, ASRC_STREAM>(w, x, gs, splits, s)
                                    : gemm_run<WT, EPI_STORE, ASRC_STREAM, 2>(w, scale, x, gs, splits, s);
        return e != hipSuccess ? e : launch_splitk_reduce<EPI>(g, splits, s);
    }
    if constexpr (WT == WT_F32) return f32w_run<EPI, ASRC_STREAM>(w, x, g, 1, s);
    return gemm_run<WT, EPI, ASRC_STREAM, 2>(w, scale, x, g, 1, s);
}
template <int EPI>
static hipError_t stream_conv_wt(int wt, const uint8_t *w, const float *scale, const float *x, const GemmArgs &g, hipStream_t s) {
    switch (wt) {
        case WT_F32: return stream_conv<WT_F32, EPI>(w, scale, x, g, s);
        case WT_F16: return stream_conv<WT_F16, EPI>(w, scale, x, g, s);
        case WT_BF16: return stream_conv<WT_BF16, EPI>(w, scale, x, g, s);
        default: return hipErrorInvalidValue;
    }
}
hipError_t launch_stream_conv(int wt, int epi, const uint8_t *w, const float *scale, const float *x, const GemmArgs &g0,
                              hipStream_t s) {
    GemmArgs g = g0;
    g.status = status_word();
    if (g.m <= 0) return hipSuccess;
    if (g.cig <= 0 || g.cig % 4 || g.ksize <= 0 || g.dil <= 0 || g.K != g.ksize * g.cig || g.K % 8 || g.lda % 4 || g.n <= 0 ||
        g.ctx != (g.ksize - 1) * g.dil || (g.ctx && !g.hist) || !g.y ||
        (g.hist_next && (!g.ctx || g.hist_next == g.hist)) || (epi == EPI_SNAKE && (!g.snake_a || !g.snake_ib)))
        return hipErrorInvalidValue;
    if (wt == WT_F32 && g.wx) {
        bool done = false;
        const hipError_t e = launch_gemm_x3p(ASRC_STREAM, epi, x, g, 1, s, &done);
        if (e != hipSuccess || done) return e;
    }
    if (epi == EPI_STORE) return stream_conv_wt<EPI_STORE>(wt, w, scale, x, g, s);
    if (epi == EPI_SNAKE) return stream_conv_wt<EPI_SNAKE>(wt, w, scale, x, g, s);
    return hipErrorInvalidValue;
}

hipError_t launch_attn_merge(const AttnPartials &P, float *ao, int m, hipStream_t s) {
    if (m <= 0) return hipSuccess;
    if (P.hd > 128) return hipErrorInvalidValue;
    return launch(k_attn_merge, dim3(P.heads, m), dim3(P.hd), 0, s, P, ao);
}

}  // namespace vh
