// Launchers of k_gemm_hh: split-f16 products of activations already in f16 planes.
#include <algorithm>
#include <atomic>

#include "vh_gemm_hh.hpp"
#include "vh_launch.hpp"

namespace vh {

int64_t pack_f16_halves(int64_t n, int64_t K) { return (n + 15) / 16 * 16 * K; }

hipError_t launch_pack_f16(const uint8_t *w, bool q8, int64_t n, int64_t K, _Float16 *out, hipStream_t s) {
    if (!w || !out || n <= 0 || K <= 0 || K % 32 || K > INT32_MAX / 64) return hipErrorInvalidValue;
    const int64_t threads = pack_f16_halves(n, K) / 8;
    const dim3 grid(unsigned((threads + 255) / 256));
    return q8 ? launch(k_pack_f16<true>, grid, dim3(256), 0, s, w, n, int32_t(K), out)
              : launch(k_pack_f16<false>, grid, dim3(256), 0, s, w, n, int32_t(K), out);
}
int64_t scale_t_floats(int64_t n, int64_t K) { return (n + 63) / 64 * 64 * (K / 32); }
hipError_t launch_scale_t(const float *sc, int64_t n, int64_t K, float *out, hipStream_t s) {
    if (!sc || !out || n <= 0 || K <= 0 || K % 32) return hipErrorInvalidValue;
    const int64_t t = scale_t_floats(n, K);
    return launch(k_scale_t, dim3(unsigned((t + 255) / 256)), dim3(256), 0, s, sc, n, int32_t(K / 32), (n + 63) / 64 * 64, out);
}
hipError_t launch_pack_planes(const _Float16 *hi, const _Float16 *lo, int64_t m, int64_t K, _Float16 *out, hipStream_t s) {
    if (!hi || !lo || !out || m <= 0 || K <= 0 || K % 32) return hipErrorInvalidValue;
    return launch(k_pack_planes, dim3(unsigned((m * K + 255) / 256)), dim3(256), 0, s, hi, lo, m, int32_t(K), out);
}

// The block tile of a product; every tile gives the same bits. Measured as launches of their own with an f32 store (us):
// - from 160 tiles of 64 x 128 (8 waves) up the widest wins: 2000 x 3072, K 1024 30.7 against 38.7 with 64 x 64; 512 x 9728,
//   K 896 (Q8) 27.7 against 28.6; 1000 x 3072, K 1024 19.2 against 23.2 with 32 x 64. 128 x 128 of 8 waves was no faster
//   there (2000 x 2048, K 1024 20.2) and slower on Q8 (512 x 9728 34.1).
// - F16 grids of at most one such tile per CU take 64 x 64: 2000 x 1024, K 1024 12.9 against 13.5, 1000 x 2048, K 1024
//   13.2 against 13.3; Q8 does not (512 x 4096, K 1024: 15.2 against 14.9).
// - below 160, 32 x 64: 333 x 3072, K 1024 11.0 against 11.4; 1000 x 1024, K 2048 14.9 against 18.6 with 64 x 128 and 16.5
//   with 64 x 64.
// - below 160 tiles of 32 x 64, 32 x 32 of 2 waves: 1024 x 256, K 512 4.7 against 5.1, 202 x 256, K 1024 6.4 against 6.6.
enum { kH32x32 = 1, kH32x64, kH64x64, kH64x128 };
static std::atomic<int> g_hh_tile{0};
void set_gemm_hh_tile(int tile) { g_hh_tile.store(tile); }
static int hh_tile(const GemmArgs &g, bool q8) {
    if (const int t = g_hh_tile.load()) return t;
    auto tiles = [&](int bm, int bn) { return int64_t((g.m + bm - 1) / bm) * ((g.n + bn - 1) / bn); };
    const int64_t wide = tiles(64, 128);
    if (wide >= 160) return !q8 && wide <= 256 ? kH64x64 : kH64x128;
    return tiles(32, 64) >= 160 ? kH32x64 : kH32x32;
}

template <int EPI, bool Q8, int TM, int TN, int WM, int WN, int S>
static hipError_t hh_launch(const _Float16 *w, const float *scale_t, const GemmArgs &g, hipStream_t s) {
    constexpr int BM = 16 * TM * WM, BN = 16 * TN * WN;
    const dim3 grid(unsigned((g.n + BN - 1) / BN), unsigned((g.m + BM - 1) / BM), unsigned(g.kchunk ? (g.K + g.kchunk - 1) / g.kchunk : 1));
    return launch(k_gemm_hh<EPI, TM, TN, WM, WN, S, Q8>, grid, dim3(64 * WM * WN), 0, s, w, scale_t, g);
}
template <int EPI, bool Q8>
static hipError_t hh_run(int tile, const _Float16 *w, const float *scale_t, const GemmArgs &g, hipStream_t s) {
    switch (tile) {
        case kH32x32: return hh_launch<EPI, Q8, 2, 1, 1, 2, 6>(w, scale_t, g, s);
        case kH32x64: return hh_launch<EPI, Q8, 1, 2, 2, 2, 4>(w, scale_t, g, s);
        case kH64x64: return hh_launch<EPI, Q8, 2, 2, 2, 2, 3>(w, scale_t, g, s);
        case kH64x128: return hh_launch<EPI, Q8, 2, 2, 2, 4, 3>(w, scale_t, g, s);
        default: return hipErrorInvalidValue;
    }
}
template <int EPI>
static hipError_t hh_wt(int tile, const _Float16 *w, const float *scale_t, const GemmArgs &g, hipStream_t s) {
    return scale_t ? hh_run<EPI, true>(tile, w, scale_t, g, s) : hh_run<EPI, false>(tile, w, nullptr, g, s);
}

// Operands the kernel can read: a tile's rows and the scales within 31-bit byte offsets.
static bool hh_args_ok(const _Float16 *w, const float *scale_t, const GemmArgs &g) {
    return w && g.a16 && g.n > 0 && g.K > 0 && g.K % 64 == 0 && int64_t(128) * g.K * 4 <= INT32_MAX &&
           (!scale_t || scale_t_floats(g.n, g.K) * 4 <= INT32_MAX);
}

// A long K on a grid too small to fill the CUs (the 512-row prefill's down projection, 512 x 896, K 4864: 224 tiles) splits
// K: slices of a multiple of 64 columns, at most 8, up to about kSplitBlocks blocks. 0: no split.
constexpr int64_t kSplitBlocks = 640;
static int hh_split(const GemmArgs &g, int *kchunk) {
    const int64_t t = int64_t((g.m + 31) / 32) * ((g.n + 63) / 64);
    if (!g.ws || t >= 256 || g.K < 2048) return 0;
    const int64_t want = std::min<int64_t>({8, (kSplitBlocks + t - 1) / t, g.K / 512});
    if (want < 2) return 0;
    *kchunk = int(((g.K + want - 1) / want + 63) / 64 * 64);
    const int splits = (g.K + *kchunk - 1) / *kchunk;
    return splits < 2 || int64_t(splits) * g.m * g.n > g.ws_cap ? 0 : splits;
}

template <int EPI>
static hipError_t hh_split_or_run(const _Float16 *w, const float *scale_t, const GemmArgs &g, hipStream_t s) {
    GemmArgs gs = g;
    const int splits = hh_split(g, &gs.kchunk);
    if (!splits) return hh_wt<EPI>(hh_tile(g, scale_t != nullptr), w, scale_t, g, s);
    const hipError_t e = hh_wt<EPI_STORE>(kH32x64, w, scale_t, gs, s);
    return e != hipSuccess ? e : launch_splitk_reduce<EPI>(g, splits, s);
}

hipError_t launch_gemm_hh_acc_rms(const _Float16 *w, const float *scale_t, const GemmArgs &g0, const float *gamma, float eps,
                                  _Float16 *out16, hipStream_t s, bool *normed) {
    GemmArgs g = g0;
    g.status = status_word();
    *normed = false;
    if (g.m <= 0) return hipSuccess;
    if (!hh_args_ok(w, scale_t, g) || !g.y) return hipErrorInvalidValue;
    GemmArgs gs = g;
    const int splits = hh_split(g, &gs.kchunk);
    // the row pass holds 8 columns per thread; without a split the ACC epilogue already wrote y
    if (!splits || g.n > 8 * 256 || g.n % 32 || !gamma || !out16) return launch_gemm_hh(EPI_ACC, w, scale_t, g, s);
    hipError_t e = hh_wt<EPI_STORE>(kH32x64, w, scale_t, gs, s);
    if (e != hipSuccess) return e;
    const dim3 grid(unsigned(g.m));
    if (g.n <= 4 * 256) e = launch(k_splitk_acc_rms_h16<4>, grid, dim3(256), 0, s, g, int32_t(splits), gamma, eps, out16);
    else e = launch(k_splitk_acc_rms_h16<8>, grid, dim3(256), 0, s, g, int32_t(splits), gamma, eps, out16);
    if (e == hipSuccess) *normed = true;
    return e;
}

hipError_t launch_gemm_hh(int epi, const _Float16 *w, const float *scale_t, const GemmArgs &g0, hipStream_t s) {
    GemmArgs g = g0;
    g.status = status_word();
    if (g.m <= 0) return hipSuccess;
    if (!hh_args_ok(w, scale_t, g)) return hipErrorInvalidValue;
    const bool y_ok = g.y != nullptr;
    switch (epi) {
        case EPI_STORE: return y_ok ? hh_split_or_run<EPI_STORE>(w, scale_t, g, s) : hipErrorInvalidValue;
        case EPI_ACC: return y_ok ? hh_split_or_run<EPI_ACC>(w, scale_t, g, s) : hipErrorInvalidValue;
        case EPI_SWIGLU_H16:  // gate|up rows in pairs; the outputs are planes of ldy = n / 2 columns
            return g.h16 && g.n % 64 == 0 && g.ldy == g.n / 2 ? hh_wt<EPI_SWIGLU_H16>(hh_tile(g, scale_t != nullptr), w, scale_t, g, s) : hipErrorInvalidValue;
        default: break;
    }
    if (scale_t) return hipErrorInvalidValue;  // the epilogues below serve the f16 models only
    switch (epi) {
        case EPI_GATED_ACC: return y_ok && g.gate ? hh_split_or_run<EPI_GATED_ACC>(w, nullptr, g, s) : hipErrorInvalidValue;
        case EPI_GELU_H16:  // planes of ldy = n columns
            return g.h16 && g.n % 32 == 0 && g.ldy == g.n ? hh_run<EPI_GELU_H16, false>(hh_tile(g, false), w, nullptr, g, s) : hipErrorInvalidValue;
        case EPI_ROPE_H16: return rope_h16_ok(g) ? hh_run<EPI_ROPE_H16, false>(hh_tile(g, false), w, nullptr, g, s) : hipErrorInvalidValue;
        default: return hipErrorInvalidValue;
    }
}

}  // namespace vh
