// Launchers of the F5-TTS DiT step kernels (AdaLN modulation, attention, input columns).
#include "vh_f5.hpp"
#include "vh_launch.hpp"

namespace vh {

hipError_t launch_norm_rows(const NormArgs &a0, hipStream_t s) {
    NormArgs a = a0;
    a.status = status_word();
    if (a.R <= 0) return hipSuccess;
    if (a.D <= 0 || a.D % 4 || !a.x || (!a.y && !a.y16) || (a.y16 && a.D % 32) || !a.sc || (!a.affine && !a.sh) || !(a.eps > 0.0))
        return hipErrorInvalidValue;
    // Rows of 256, 512, 768 and 1024 take k_norm_rows, a row per wave where its width allows (1000 x 1024 planes 3.7 us, two
    // rows per wave 4.2), except many planes rows, where half-waves' runs of 32 bytes per plane matter more (2000 x 1024:
    // 4.9 against 5.5).
    auto rows = [&](auto kernel, int lanes) { return launch(kernel, dim3(unsigned((a.R + 256 / lanes - 1) / (256 / lanes))), dim3(256), 0, s, a); };
    switch (a.D) {
        case 256: return rows(k_norm_rows<32, 1>, 32);
        case 512: return rows(k_norm_rows<64, 1>, 64);
        case 768: return rows(k_norm_rows<32, 3>, 32);
        case 1024: return a.y16 && a.R >= 1536 ? rows(k_norm_rows<32, 4>, 32) : rows(k_norm_rows<64, 2>, 64);
        default: break;
    }
    if (a.D <= 4 * 256) return launch(k_f5_modulate<4, true>, dim3(unsigned((a.R + 3) / 4)), dim3(256), 0, s, a);
    return launch(k_f5_modulate<kNormRegChunks, false>, dim3(unsigned((a.R + 3) / 4)), dim3(256), 0, s, a);
}

hipError_t launch_f5_modulate(const float *x, int64_t R, int D, const float *sc, const float *sh, float *y, _Float16 *y16,
                              hipStream_t s) {
    if (R > INT32_MAX) return hipErrorInvalidValue;
    NormArgs a{};
    a.x = x; a.y = y; a.y16 = y16; a.sc = sc; a.sh = sh;
    a.eps = 1e-6;  // the modulation adds the double 1e-6 (f5.cpp:608-625)
    a.R = int32_t(R); a.D = D;
    return launch_norm_rows(a, s);
}

hipError_t launch_layernorm_rows(const float *x, int64_t R, int D, const float *w, const float *b, float *y, hipStream_t s) {
    if (R > INT32_MAX || !y) return hipErrorInvalidValue;
    NormArgs a{};
    a.x = x; a.y = y; a.sc = w; a.sh = b;
    a.eps = double(1e-6f);  // LayerNorm's float eps 1e-6f, widened (kernels.cpp:721)
    a.R = int32_t(R); a.D = D; a.affine = 1;
    return launch_norm_rows(a, s);
}

hipError_t launch_dwconv(const float *x, const float *w, const float *b, float *y, int64_t R, int C, int K, int seq, hipStream_t s) {
    if (R <= 0) return hipSuccess;
    if (C <= 0 || K <= 0 || K % 2 == 0 || seq <= 0 || R % seq || !w) return hipErrorInvalidValue;
    const int64_t n = R * C;
    return launch(k_dwconv, dim3(unsigned((n + 255) / 256)), dim3(256), 0, s, x, w, b, y, R, int32_t(C), int32_t(K), int32_t(seq));
}

hipError_t launch_f5_fill_x(const float *x, int N, int mel, float *cat, int W, int B, hipStream_t s) {
    const int64_t n = int64_t(B) * N * mel;
    if (n <= 0) return hipSuccess;
    return launch(k_f5_fill_x, dim3(unsigned((n + 255) / 256)), dim3(256), 0, s, x, int32_t(N), int32_t(mel), cat, int32_t(W),
                  int32_t(B));
}

template <int W, int QT, int KS>
static hipError_t f5_attn(const F5AttnArgs &a, int heads, int B, hipStream_t s) {
    const hipError_t e = ensure_smem(reinterpret_cast<const void *>(&k_f5_attn<W, QT, KS>), f5_attn_smem(KS));
    if (e != hipSuccess) return e;
    return launch(k_f5_attn<W, QT, KS>, dim3(unsigned((a.N + 16 * QT * W - 1) / (16 * QT * W)), unsigned(heads), unsigned(B)),
                  dim3(64 * W * KS), f5_attn_smem(KS), s, a);
}
hipError_t launch_f5_attn(const _Float16 *qkv16, float *out, _Float16 *out16, int B, int N, int heads, int hd, int np, int ldo,
                          float scale, hipStream_t s) {
    if (B <= 0 || N <= 0) return hipSuccess;
    if (hd != kF5Hd || heads <= 0 || np < N || np % 64 || ldo % 4 || (out16 && ldo % 32) || (!out && !out16)) return hipErrorInvalidValue;
    if ((int64_t(N) + 64) * 2 * heads * hd * 2 > INT32_MAX) return hipErrorInvalidValue;
    const F5AttnArgs a{qkv16, out, out16, int32_t(N), int32_t(np), int32_t(ldo), scale};
    // One block per CU (128 KiB of LDS): the fewest query rows per block that still fit the CUs at once. flow estimator,
    // 2 x 8 heads of 512: 32-row blocks 9.6 us, 64-row 10.2, 128-row 14.8; DiT, 16 heads of 333: 7.8, 8.5, 12.6; 2 x 16 heads of
    // 1000, more than fit with any: 60, 38 and 32, where a key tile read for 32 rows per wave costs half the LDS reads.
    auto blocks = [&](int rows) { return int64_t((N + rows - 1) / rows) * heads * B; };
    if (blocks(64) > 256) return f5_attn<4, 2, 2>(a, heads, B, s);
    if (blocks(32) > 256) return f5_attn<4, 1, 2>(a, heads, B, s);
    return f5_attn<2, 1, 2>(a, heads, B, s);
}

}  // namespace vh
