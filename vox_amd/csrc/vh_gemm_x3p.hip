// Launchers of k_gemm_x3p: F32 weights split and laid out once, on the f16 matrix cores.
#include <algorithm>

#include "vh_gemm_x3p.hpp"
#include "vh_launch.hpp"

namespace vh {

int64_t pack_x3_bytes(int64_t n, int64_t K) { return (n + 15) / 16 * ((K + 31) / 32) * 2048; }

hipError_t launch_pack_x3(const float *w, int64_t n, int64_t K, void *out, hipStream_t s) {
    if (!w || !out || n <= 0 || K <= 0 || K > INT32_MAX / 64) return hipErrorInvalidValue;
    const int64_t threads = pack_x3_bytes(n, K) / 32;  // 64 per 2 KiB tile
    if (threads > (int64_t(INT32_MAX) * 256)) return hipErrorInvalidValue;
    return launch(k_pack_x3, dim3(unsigned((threads + 255) / 256)), dim3(256), 0, s, w, n, int32_t(K), static_cast<_Float16 *>(out));
}

// Whether k_gemm_x3p can take the product: packed weights, and every byte offset of A, the history and W within 31 bits.
static bool x3p_ok(int asrc, const GemmArgs &g) {
    constexpr int64_t kMax = 0x7FFFFF00;
    const int64_t width = asrc == ASRC_ROWS ? g.K : asrc == ASRC_STREAM ? g.cig : g.lda;
    if (!g.wx || g.f32_wide || width > g.lda || int64_t(g.m) * g.lda * 4 > kMax || pack_x3_bytes(g.n, g.K) > kMax) return false;
    if (asrc == ASRC_ROWS) return true;
    return g.cig > 1 && (int64_t(g.K) + 128) * g.cig < (int64_t(1) << 32) && int64_t(g.ctx) * g.cig * 4 <= kMax &&
           (asrc != ASRC_CONV || g.m % g.seq == 0);
}

// The block tile and the K slices of a product, from its count of tiles:
// - 200 tiles of 64 x 64 or more fill the 256 CUs: 64 x 64 of 8 waves (2560 x 384, K 2688: 31.8 us against 52 with 4
//   waves and 46 with 64 x 96 of 4 waves; also where 64 x 96 would pad a third less: 30720 x 96 in the codec, K 672 34.5 against
//   38.4 us, K 96 17.0 against 21.1; 3840 x 80 x 8 groups, K 560 42.1 against 49.4).
// - below that 32 x 64 tiles of 8 waves: 333 x 64 x 16 groups, K 1984: 16.9 against 23.4 us; 1024 x 256, K 768: 8.4
//   against 10.2 us. From 100 of them on a K below 2048 is not split (1920 x 96, K 672, 120 tiles: 7.5 us against 8.9 with 2
//   slices and their reduce).
// - fewer: K slices up to about 200 blocks, of at least 128 columns (32 x 768, K 5376: 11.3 us with 14 slices, 11.7 with
//   21, 12.2 with 7; 160 x 384, K 2688: 10.1 with 7, 11.2 with 14), and at most 256 blocks, a round of the CUs (64 x 2112,
//   K 5376, 66 tiles: 23.4 us with 3 slices, 29.9 with 4). Up to K 768, or where the epilogue cannot follow a reduce,
//   32 x 32 tiles of 4 waves instead, since the reduce is a launch of 4.5 us (160 x 384, K 384: 5.0 us against 5.7 with 32 x 64,
//   6.6 with 2 slices; the flow estimator's 202 x 256, K 768: 8.2 against 5.0 + 4.6 with 6 slices; 16 x 1026, K 512 as a matmul
//   call 52 us against 56). At K 1024 it was faster still in the codec, but one chain of that length rounds more than the
//   slices did (1.7e-6 against 1.4e-6 of the samples).
// - a long K from 86 tiles on, where a round of them holds two slices or none: 64 x 64 tiles in slices up to 256 blocks where
//   they pad no rows, up to 64 of them from K 2048 (33 x 3072, K 5376: 22.8 us against 28.8 with 32 x 64 in 2 slices and 24.7-26.7
//   by k_gemm_x3; 128 x 1472, K 3072 18.4 against 21.8 and 22.0; 64 x 1024 x K 2048, 32 tiles, no gain), up to 96 from K 4096
//   (64 x 6144, K 5376: 40.4 against 45.2 unsplit; at K 2048 23.2 against 21.8). Odd counts of row tiles: two slices of 32 x 64
//   up to 128 tiles from K 2048 (400 x 512, K 5376: 29.5 us, unsplit 45.3, k_gemm_x3 31.2; K 2048: 16.6, 19.5, 19.1), three up to
//   170 from K 3072 (400 x 768, K 5376: 39.6 us, unsplit 46.2, k_gemm_x3 44.1; at K 2048 20.7 against 19.7).
enum { kT64x64, kT32x64, kT32x32 };
struct X3Plan {
    int tile, splits, kchunk;
};
static X3Plan x3p_plan(const GemmArgs &g, int groups, bool reducible) {
    auto tiles = [&](int bm, int bn) { return int64_t((g.m + bm - 1) / bm) * ((g.n + bn - 1) / bn) * groups; };
    if (tiles(64, 64) >= 200) return {kT64x64, 1, 0};
    const int64_t t = tiles(32, 64), t64 = tiles(64, 64);
    const bool split = reducible && groups == 1 && g.ws;
    X3Plan whole{t >= 100 ? kT32x64 : kT32x32, 1, 0}, p{kT32x64, 1, 0};
    int64_t want = 1;
    if (split && t > 85 && t == 2 * t64 && ((t64 <= 64 && g.K >= 2048) || (t64 <= 96 && g.K >= 4096))) {
        p.tile = kT64x64;
        want = 256 / t64;
    } else if (split && t >= 100) {
        if (t <= 128 && g.K >= 2048) want = 2;
        else if (t > 128 && t <= 170 && g.K >= 3072) want = 3;
    } else if (split && g.K > 768) {
        want = std::min<int64_t>({(200 + t - 1) / t, 256 / t, g.K / 128});
    }
    if (want < 2) return whole;
    p.kchunk = int(((g.K + want - 1) / want + 63) / 64 * 64);
    p.splits = (g.K + p.kchunk - 1) / p.kchunk;
    return p.splits < 2 || int64_t(p.splits) * g.m * g.n > g.ws_cap ? whole : p;
}

template <int EPI, int ASRC, int WM, int WN, int TM, int TN>
static hipError_t x3p_tile(const float *A, const GemmArgs &g, int z, hipStream_t s) {
    constexpr int BM = 16 * TM * WM, BN = 16 * TN * WN;
    const dim3 grid(unsigned((g.n + BN - 1) / BN), unsigned((g.m + BM - 1) / BM), unsigned(z));
    return launch(k_gemm_x3p<EPI, ASRC, WM, WN, TM, TN>, grid, dim3(64 * WM * WN), 0, s, static_cast<const uint8_t *>(g.wx), A, g);
}
template <int EPI, int ASRC>
static hipError_t x3p_tiles(int tile, const float *A, const GemmArgs &g, int z, hipStream_t s) {
    switch (tile) {
        case kT64x64: return x3p_tile<EPI, ASRC, 2, 4, 2, 1>(A, g, z, s);
        case kT32x64: return x3p_tile<EPI, ASRC, 2, 4, 1, 1>(A, g, z, s);
        default: return x3p_tile<EPI, ASRC, 2, 2, 1, 1>(A, g, z, s);
    }
}
template <int EPI, int ASRC>
static hipError_t x3p_run(const float *A, const GemmArgs &g, int groups, hipStream_t s) {
    const X3Plan p = x3p_plan(g, groups, kReduceEpi<EPI>);
    if (p.splits == 1) return x3p_tiles<EPI, ASRC>(p.tile, A, g, groups, s);
    if constexpr (kReduceEpi<EPI>) {
        GemmArgs gs = g;
        gs.kchunk = p.kchunk;
        const hipError_t e = x3p_tiles<EPI_STORE, ASRC>(p.tile, A, gs, p.splits, s);
        return e != hipSuccess ? e : launch_splitk_reduce<EPI>(g, p.splits, s);
    }
    return hipErrorInvalidValue;  // no plan splits such a product
}

hipError_t launch_gemm_x3p(int asrc, int epi, const float *A, const GemmArgs &g0, int groups, hipStream_t s, bool *done) {
    *done = x3p_ok(asrc, g0);
    if (!*done) return hipSuccess;
    GemmArgs g = g0;
    g.kchunk = 0;
    if (g.cig > 1) g.cig_magic = uint32_t(((int64_t(1) << 32) + g.cig - 1) / g.cig);
    if (asrc == ASRC_ROWS) {
        switch (epi) {
            case EPI_STORE: return x3p_run<EPI_STORE, ASRC_ROWS>(A, g, 1, s);
            case EPI_ACC: return x3p_run<EPI_ACC, ASRC_ROWS>(A, g, 1, s);
            case EPI_SWIGLU: return x3p_run<EPI_SWIGLU, ASRC_ROWS>(A, g, 1, s);
            case EPI_GATED_ACC: return x3p_run<EPI_GATED_ACC, ASRC_ROWS>(A, g, 1, s);
            case EPI_GELU: return x3p_run<EPI_GELU, ASRC_ROWS>(A, g, 1, s);
            case EPI_GELU_ERF: return x3p_run<EPI_GELU_ERF, ASRC_ROWS>(A, g, 1, s);
            case EPI_ACC_SNAKE: return x3p_run<EPI_ACC_SNAKE, ASRC_ROWS>(A, g, 1, s);
            case EPI_ROPE_H16: return x3p_run<EPI_ROPE_H16, ASRC_ROWS>(A, g, 1, s);
            default: break;
        }
    } else if (asrc == ASRC_CONV) {
        switch (epi) {
            case EPI_STORE: return x3p_run<EPI_STORE, ASRC_CONV>(A, g, groups, s);
            case EPI_ACC: return x3p_run<EPI_ACC, ASRC_CONV>(A, g, groups, s);
            case EPI_MISH: return x3p_run<EPI_MISH, ASRC_CONV>(A, g, groups, s);
            case EPI_MISH_ACC: return x3p_run<EPI_MISH_ACC, ASRC_CONV>(A, g, groups, s);
            default: break;
        }
    } else if (asrc == ASRC_STREAM) {
        switch (epi) {
            case EPI_STORE: return x3p_run<EPI_STORE, ASRC_STREAM>(A, g, 1, s);
            case EPI_SNAKE: return x3p_run<EPI_SNAKE, ASRC_STREAM>(A, g, 1, s);
            default: break;
        }
    }
    *done = false;  // an epilogue without an instance here: the caller's kernel
    return hipSuccess;
}

}  // namespace vh
