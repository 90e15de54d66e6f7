// vh_f5.hpp — F5-TTS DiT step kernels besides the GEMMs: AdaLN modulation, non-causal softmax attention on the
// matrix cores, and the x columns of the step input.
#pragma once
#include "vh_common.hpp"
#include "vh_types.hpp"

namespace vh {

typedef float f32x4a __attribute__((ext_vector_type(4)));
typedef _Float16 f16x4a __attribute__((ext_vector_type(4)));

// mish as nn.hpp:103-107 (the CosyVoice2 / Chatterbox estimator's): x tanh(softplus(x)) with tanh(log(1 + e)) =
// n / (n + 2), n = e (e + 2), and x itself above 20.
VH_DEV float mish_nn_f(float x) {
    if (x > 20.f) return x;
    const float e = expf(x), n = e * (e + 2.0f);
    return x * (n / (n + 2.0f));
}

// Row LayerNorm (NormArgs) of any D, one wave per row (4 rows per 256-thread block): mean and variance in double (two passes
// over the row, which stays in L1), inv = float(1 / sqrt(var + eps)). The forms: AdaLN modulation without
// parameters (f5.cpp:608-625, eps 1e-6), y = (x - float(mean)) * inv * (1 + scale) + shift; LayerNorm with weight
// and bias (kernels.cpp:714-723 and nn.cpp:248-265, which compute alike), y = (x - float(mean)) * inv * w + b; then
// mish and a per-channel bias when asked (the estimator's CausalBlock1D and its time bias, cosyvoice.cpp:155-178).
// D % 4 == 0.
// NC chunks of 4 columns per lane stay in registers between the passes (NC = 8: rows up to 2048 values, longer rows
// are read again); PRE (rows of at most 4 x 256 = 1024 values): the row's parameters (scale, shift, time bias) are
// loaded with the row, before the statistics, instead of one more round trip after them; the arithmetic is the same.
constexpr int kNormRegChunks = 8;
template <int NC, bool PRE>
__global__ __launch_bounds__(256) void k_f5_modulate(NormArgs a) {
    static_assert(!PRE || NC <= 4, "parameters in registers only for short rows");
    const int lane = threadIdx.x & 63, row = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (row >= a.R) return;
    const int D = a.D;
    const float *xr = a.x + int64_t(row) * D;
    auto wsum = [&](double v) {
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, kWave);
        return v;
    };
    // the row is read once: chunk c of this lane is columns 4 lane + 256 c .. + 3; the first NC chunks stay in
    // registers (fully unrolled loops), columns beyond 256 NC are read again from memory
    f32x4a reg[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) {
        const int i = 4 * lane + 256 * c;
        reg[c] = i < D ? *reinterpret_cast<const f32x4a *>(xr + i) : f32x4a{0.f, 0.f, 0.f, 0.f};
    }
    // PRE: the parameters of this lane's chunks (shift / time bias read from the scale row when absent, never used)
    f32x4a pcs[PRE ? NC : 1], psh[PRE ? NC : 1], ptb[PRE ? NC : 1];
    if constexpr (PRE) {
        const float *shp = a.sh ? a.sh : a.sc, *tbp = a.tb ? a.tb : a.sc;
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            const int i = 4 * lane + 256 * c < D ? 4 * lane + 256 * c : 0;
            pcs[c] = *reinterpret_cast<const f32x4a *>(a.sc + i);
            psh[c] = *reinterpret_cast<const f32x4a *>(shp + i);
            ptb[c] = *reinterpret_cast<const f32x4a *>(tbp + i);
        }
    }
    const int tail0 = 256 * NC;
    double s = 0.0;
#pragma unroll
    for (int c = 0; c < NC; ++c)
        s += double(reg[c][0]) + double(reg[c][1]) + double(reg[c][2]) + double(reg[c][3]);  // zeros past D
    for (int i = tail0 + 4 * lane; i < D; i += 256) {
        const f32x4a v = *reinterpret_cast<const f32x4a *>(xr + i);
        s += double(v[0]) + double(v[1]) + double(v[2]) + double(v[3]);
    }
    const double mean = wsum(s) / D;
    double q = 0.0;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
        if (4 * lane + 256 * c >= D) continue;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const double dd = double(reg[c][e]) - mean;
            q += dd * dd;
        }
    }
    for (int i = tail0 + 4 * lane; i < D; i += 256) {
        const f32x4a v = *reinterpret_cast<const f32x4a *>(xr + i);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const double dd = double(v[e]) - mean;
            q += dd * dd;
        }
    }
    const double var = wsum(q) / D;
    const float inv = float(1.0 / sqrt(var + a.eps)), fm = float(mean);
    auto emit = [&](int i, const f32x4a &v, const f32x4a &cs, const f32x4a &t, const f32x4a &b) {
        f32x4a r;
#pragma unroll
        for (int e = 0; e < 4; ++e) r[e] = (v[e] - fm) * inv * (a.affine ? cs[e] : 1.0f + cs[e]) + (a.sh ? t[e] : 0.f);
        if (a.mish) {
#pragma unroll
            for (int e = 0; e < 4; ++e) r[e] = mish_nn_f(r[e]);
        }
        if (a.tb) {
#pragma unroll
            for (int e = 0; e < 4; ++e) r[e] += b[e];
        }
        if (a.y16) {
            f16x4a hi, lo;
            bool bad = false;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                _Float16 h, l;
                bad |= split_f16(r[e], h, l);
                hi[e] = h;
                lo[e] = l;
            }
            raise_status(a.status, bad, kStatusF16Range);
            _Float16 *hr = a.y16 + plane_off(row, i, D);
            *reinterpret_cast<f16x4a *>(hr) = hi;
            *reinterpret_cast<f16x4a *>(hr + kPlaneLo) = lo;
        } else {
            *reinterpret_cast<f32x4a *>(a.y + int64_t(row) * D + i) = r;
        }
    };
    auto emit_load = [&](int i, const f32x4a &v) {  // the parameters read here, after the statistics
        const f32x4a cs = *reinterpret_cast<const f32x4a *>(a.sc + i);
        const f32x4a t = a.sh ? *reinterpret_cast<const f32x4a *>(a.sh + i) : f32x4a{0.f, 0.f, 0.f, 0.f};
        const f32x4a b = a.tb ? *reinterpret_cast<const f32x4a *>(a.tb + i) : f32x4a{0.f, 0.f, 0.f, 0.f};
        emit(i, v, cs, t, b);
    };
#pragma unroll
    for (int c = 0; c < NC; ++c) {
        if (4 * lane + 256 * c >= D) continue;
        if constexpr (PRE) emit(4 * lane + 256 * c, reg[c], pcs[c], psh[c], ptb[c]);
        else emit_load(4 * lane + 256 * c, reg[c]);
    }
    for (int i = tail0 + 4 * lane; i < D; i += 256) emit_load(i, *reinterpret_cast<const f32x4a *>(xr + i));
}

// k_f5_modulate for rows of 8 L C values: L lanes per row (64 / L rows per wave), 8 neighbouring columns of a lane at a
// time (a lane's 8 halves of a plane are one store), the parameters loaded with the row. Both moments are summed in one
// pass over x minus the row's first value (a difference of floats: rounded at 2^-53, and a row far from zero or constant
// cancels nothing), their sums by DPP and row swaps. Bound by the round trip to rows another XCD wrote, and the launch; the
// two reductions of k_f5_modulate through LDS were a second round trip. Launches back to back, k_f5_modulate -> here (us):
// f32 rows 1024 x 256 2.9 -> 2.1, 938 x 512 3.0 -> 2.4, 2000 x 1024 4.8 -> 4.3; planes 1024 x 256 3.0 -> 2.4, 333 x 1024
// 3.7 -> 2.9, 2000 x 1024 6.1 -> 4.9. The outputs are the same bits there.
template <int CTRL>
VH_DEV double dpp_add(double v) {
    const uint64_t u = __builtin_bit_cast(uint64_t, v);
    const uint32_t lo = uint32_t(dpp<CTRL>(int(uint32_t(u)))), hi = uint32_t(dpp<CTRL>(int(uint32_t(u >> 32))));
    return v + __builtin_bit_cast(double, uint64_t(hi) << 32 | lo);
}
// v summed over groups of L lanes (16, 32, 64), the same bits in every lane of a group.
template <int L>
VH_DEV double lanes_sum(double v) {
    v = dpp_add<kDppXor1>(v);
    v = dpp_add<kDppXor2>(v);
    v = dpp_add<kDppRowHalfMirror>(v);
    v = dpp_add<kDppRowMirror>(v);
    auto swap_add = [&](auto sw) {
        const uint64_t u = __builtin_bit_cast(uint64_t, v);
        const auto l = sw(uint32_t(u)), h = sw(uint32_t(u >> 32));
        v = __builtin_bit_cast(double, uint64_t(h[0]) << 32 | l[0]) + __builtin_bit_cast(double, uint64_t(h[1]) << 32 | l[1]);
    };
    if (L >= 32) swap_add([](uint32_t x) { return __builtin_amdgcn_permlane16_swap(x, x, false, false); });
    if (L >= 64) swap_add([](uint32_t x) { return __builtin_amdgcn_permlane32_swap(x, x, false, false); });
    return v;
}
template <int L, int C>
__global__ __launch_bounds__(256) void k_norm_rows(NormArgs a) {
    constexpr int D = 8 * L * C, RB = 256 / L;
    const int l = threadIdx.x % L, row = blockIdx.x * RB + threadIdx.x / L;
    const float *xr = a.x + int64_t(min(row, a.R - 1)) * D;
    f32x4a v[C][2], cs[C][2], sh[C][2], tb[C][2];
#pragma unroll
    for (int c = 0; c < C; ++c)
#pragma unroll
        for (int h = 0; h < 2; ++h) v[c][h] = *reinterpret_cast<const f32x4a *>(xr + 8 * L * c + 8 * l + 4 * h);
    const float x0 = xr[0];
    const float *shp = a.sh ? a.sh : a.sc, *tbp = a.tb ? a.tb : a.sc;  // never used when absent
#pragma unroll
    for (int c = 0; c < C; ++c)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int i = 8 * L * c + 8 * l + 4 * h;
            cs[c][h] = *reinterpret_cast<const f32x4a *>(a.sc + i);
            sh[c][h] = *reinterpret_cast<const f32x4a *>(shp + i);
            tb[c][h] = *reinterpret_cast<const f32x4a *>(tbp + i);
        }
    double s = 0.0, q = 0.0;
#pragma unroll
    for (int c = 0; c < C; ++c)
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const double d = double(v[c][h][e]) - double(x0);
                s += d;
                q = __builtin_fma(d, d, q);
            }
    s = lanes_sum<L>(s) / D;
    q = lanes_sum<L>(q) / D;
    double var = q - s * s;
    var = var < 0.0 ? 0.0 : var;  // rounding only; a NaN stays
    const float inv = float(1.0 / sqrt(var + a.eps)), fm = float(double(x0) + s);
    if (row >= a.R) return;
#pragma unroll
    for (int c = 0; c < C; ++c) {
        float r[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const float p = cs[c][e / 4][e % 4];
            r[e] = (v[c][e / 4][e % 4] - fm) * inv * (a.affine ? p : 1.0f + p) + (a.sh ? sh[c][e / 4][e % 4] : 0.f);
        }
        if (a.mish) {
#pragma unroll
            for (int e = 0; e < 8; ++e) r[e] = mish_nn_f(r[e]);
        }
        if (a.tb) {
#pragma unroll
            for (int e = 0; e < 8; ++e) r[e] += tb[c][e / 4][e % 4];
        }
        const int i = 8 * L * c + 8 * l;
        if (a.y16) {
            f16x4a hi[2], lo[2];
            bool bad = false;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                _Float16 h, w;
                bad |= split_f16(r[e], h, w);
                hi[e / 4][e % 4] = h;
                lo[e / 4][e % 4] = w;
            }
            raise_status(a.status, bad, kStatusF16Range);
            _Float16 *o = a.y16 + plane_off(row, i, D);
            *reinterpret_cast<u32x4 *>(o) = __builtin_bit_cast(u32x4, hi);
            *reinterpret_cast<u32x4 *>(o + kPlaneLo) = __builtin_bit_cast(u32x4, lo);
        } else {
            float *o = a.y + int64_t(row) * D + i;
            *reinterpret_cast<f32x4a *>(o) = f32x4a{r[0], r[1], r[2], r[3]};
            *reinterpret_cast<f32x4a *>(o + 4) = f32x4a{r[4], r[5], r[6], r[7]};
        }
    }
}

// Depthwise "same" Conv1d (f5_ops.cpp:106-147 with groups = channels: the Vocos blocks' dwconv, f5.cpp:341) over
// batches of seq rows: y[t][c] = b[c] + sum_k w[c][k] x[t + k - K/2][c], zeros outside the batch, k in order. One
// thread per output, consecutive threads on consecutive channels.
__global__ __launch_bounds__(256) void k_dwconv(const float *__restrict__ x, const float *__restrict__ w, const float *__restrict__ b,
                                                float *__restrict__ y, int64_t R, int32_t C, int32_t K, int32_t seq) {
    const int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x;
    if (i >= R * C) return;
    const int64_t r = i / C;
    const int c = int(i % C), t = int(r % seq);
    const int64_t r0 = r - t;
    float acc = b ? b[c] : 0.f;
    for (int k = 0; k < K; ++k) {
        const int tt = t + k - K / 2;
        if (tt >= 0 && tt < seq) acc += w[int64_t(c) * K + k] * x[(r0 + tt) * C + c];
    }
    y[i] = acc;
}

// cat[b][t][0..mel) = x[t][0..mel) for every batch b (the x columns of the DiT input, gpu.hpp:85-88).
__global__ __launch_bounds__(256) void k_f5_fill_x(const float *__restrict__ x, int32_t N, int32_t mel, float *__restrict__ cat,
                                                   int32_t W, int32_t B) {
    const int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x;
    if (i >= int64_t(B) * N * mel) return;
    const int64_t r = i / mel, c = i % mel;
    cat[r * W + c] = x[(r % N) * mel + c];
}

// Non-causal softmax attention of one head over N keys (f5.cpp:626-650): S = (q . k) * scale, softmax per row,
// O = P V, for head_dim 64. grid (ceil(N / (16 QT W)), heads, B), block 64 W KS: each of the W query waves takes 16 QT query
// rows; the KS key groups take alternate tiles of 64 keys and are merged at the end. An online softmax (running max and sum
// per row, O rescaled) replaces the reference's whole-row max, which changes only the rounding; exp(x) is taken as
// 2^(x log2 e) on v_exp_f32.
// Both products run on the f16 matrix cores (v_mfma_f32_16x16x32_f16) with every f32 operand as two f16 halves,
// x = hi + lo, and three products per pair (hi.hi + hi.lo + lo.hi; the dropped lo.lo term is below 2^-22 relative):
// each product is exact in the f32 accumulator, so S and P V keep f32-level accuracy. q, k and v arrive split and in the
// order the MFMAs read them (qkv_off; the q|k|v GEMM's EPI_ROPE_H16 epilogue), the rows past N zero, so a key tile is 32
// fragments of 1 KiB, copied to LDS by DMA one tile ahead of the one in use.
// The products are taken transposed, S^T = K Q^T and O^T = V^T P^T, so that a lane holds one query row (lane % 16)
// throughout: its S^T values (keys 16 j + 4 (lane / 16) + i) are already the B operand of P^T once the 32 keys
// of a chunk are numbered in the order the lanes hold them (V^T's A operand stored in that same order), P never
// leaves registers, and the row's max needs only two row swaps (its sum is kept per lane until the end).
// What bounds it (2 x 16 heads of 1000 keys): the MFMAs, 24.6 GFLOP in three products or 20 us at a large product's rate, and
// the softmax on the vector units, about as long, which overlap only in part. Against row-major halves staged through
// registers (16 rows per wave): 40 -> 32 us there, 16 heads of 333 12 -> 7.8, the flow estimator's 2 x 8 heads of 512 11.8 -> 9.6.
struct F5AttnArgs {
    const _Float16 *h16;  // q, k, v (qkv_off)
    float *out;           // [B N][ldo], head h at column h * 64
    _Float16 *out16;      // when set: the output as f16 planes of ldo columns (plane_off's layout)
    int32_t N, np, ldo;   // np: N padded to 64
    float scale;
};
constexpr int kF5Hd = kF5HeadDim;
static_assert(kF5Hd == kQkvHead, "the head layout of qkv_off");
typedef _Float16 h16x8 __attribute__((ext_vector_type(8)));
// Four tiles c[j] += a[j] b, a and b as halves; the tiles in turn, so that no MFMA waits for the one before it.
VH_DEV void mfma3(const h16x8 (&ah)[4], const h16x8 (&al)[4], h16x8 bh, h16x8 bl, f32x4a (&c)[4]) {
#pragma unroll
    for (int j = 0; j < 4; ++j) c[j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah[j], bh, c[j], 0, 0, 0);
#pragma unroll
    for (int j = 0; j < 4; ++j) c[j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah[j], bl, c[j], 0, 0, 0);
#pragma unroll
    for (int j = 0; j < 4; ++j) c[j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(al[j], bh, c[j], 0, 0, 0);
}
// The other three lanes' values of a row of S^T: lanes lr, lr + 16, lr + 32, lr + 48.
template <class F>
VH_DEV float row4(float v, F f) {
    const uint32_t u = __builtin_bit_cast(uint32_t, v);
    const auto p = __builtin_amdgcn_permlane16_swap(u, u, false, false);
    const uint32_t p0 = p[0], p1 = p[1];
    v = f(__builtin_bit_cast(float, p0), __builtin_bit_cast(float, p1));
    const uint32_t t = __builtin_bit_cast(uint32_t, v);
    const auto q = __builtin_amdgcn_permlane32_swap(t, t, false, false);
    const uint32_t q0 = q[0], q1 = q[1];
    return f(__builtin_bit_cast(float, q0), __builtin_bit_cast(float, q1));
}
constexpr int kF5Tile = 32 * 1024;  // bytes of 64 keys: k, then v
inline size_t f5_attn_smem(int KS) { return size_t(KS) * 2 * kF5Tile; }

template <int W, int QT, int KS>
__global__ __launch_bounds__(64 * W * KS, W * KS >= 4 ? W * KS / 4 : 1) void k_f5_attn(F5AttnArgs a) {
    extern __shared__ __align__(1024) uint8_t lds[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6), lr = lane & 15, lg = lane >> 4;
    const int qw = wave % W, kh = wave / W, vo = lane * 16;
    // a contiguous run of (batch, head) pairs per XCD, so each head's keys and values stay in one L2
    const int qt = gridDim.x, heads = gridDim.y, B = gridDim.z;
    const int t = xcd_tile(int(blockIdx.x) + qt * (int(blockIdx.y) + heads * int(blockIdx.z)), qt * heads * B);
    const int q0 = (t % qt) * (16 * QT * W) + qw * 16 * QT, h = (t / qt) % heads, b = t / (qt * heads);
    const _Float16 *Q = a.h16 + qkv_off(0, b, h, 0, 0, B, heads, a.np);
    const u32x4s rk = dma_rsrc(a.h16 + qkv_off(1, b, h, 0, 0, B, heads, a.np)), rv = dma_rsrc(a.h16 + qkv_off(2, b, h, 0, 0, B, heads, a.np));
    // B operand of S^T: lane holds q[q0 + 16 i + lr][32 c + 8 lg + e] (row blocks past the last read it; not stored)
    h16x8 qh[QT][2], ql[QT][2];
#pragma unroll
    for (int i = 0; i < QT; ++i)
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            const _Float16 *p = Q + int64_t(min(q0 / 16 + i, a.np / 16 - 1) * 2 + c) * 1024 + lane * 8;
            qh[i][c] = *reinterpret_cast<const h16x8 *>(p);
            ql[i][c] = *reinterpret_cast<const h16x8 *>(p + kPlaneLo);
        }
    const uint8_t *st = lds + kh * 2 * kF5Tile;  // this key group's two stages
    const uint32_t base = uint32_t(reinterpret_cast<uintptr_t>((lds_void *)lds)) + kh * 2 * kF5Tile;
    auto issue = [&](int tile, int buf) {  // this wave's share of the tile's fragments
#pragma unroll
        for (int p = 0; p < 16 / W; ++p) {
            const int o = (qw + W * p) * 1024;
            dma_b128(rk, base + buf * kF5Tile + o, vo, tile * 16384 + o);
            dma_b128(rv, base + buf * kF5Tile + 16384 + o, vo, tile * 16384 + o);
        }
    };
    const float sl = a.scale * 1.4426950408889634f;  // scores in log2 units
    float mrow[QT], lrow[QT];                         // of query row lr: the max of S, and this lane's part of the sum
    f32x4a o[QT][4];                                  // O^T: lane holds O[row lr][16 dt + 4 lg + i]
#pragma unroll
    for (int i = 0; i < QT; ++i) {
        mrow[i] = -INFINITY;
        lrow[i] = 0.f;
#pragma unroll
        for (int d = 0; d < 4; ++d) o[i][d] = f32x4a{0.f, 0.f, 0.f, 0.f};
    }
    auto compute = [&](const uint8_t *kv, int kt) {
        auto frag = [&](int f) { return *reinterpret_cast<const h16x8 *>(kv + f * 1024 + vo); };
        // S^T tiles: A operand lane holds K[16 j + lr][32 c + 8 lg + e]; lane gets S^T[16 j + 4 lg + e][lr]
        f32x4a s[QT][4];
#pragma unroll
        for (int i = 0; i < QT; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) s[i][j] = f32x4a{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            h16x8 fh[4], fl[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                fh[j] = frag((j * 2 + c) * 2);
                fl[j] = frag((j * 2 + c) * 2 + 1);
            }
#pragma unroll
            for (int i = 0; i < QT; ++i) mfma3(fh, fl, qh[i][c], ql[i][c], s[i]);
        }
        h16x8 ph[QT][2], pl[QT][2];
#pragma unroll
        for (int i = 0; i < QT; ++i) {
            if (kt + 64 > a.N) {  // the last, partial tile: keys past N drop out
#pragma unroll
                for (int j = 0; j < 4; ++j)
#pragma unroll
                    for (int e = 0; e < 4; ++e) s[i][j][e] = kt + 16 * j + 4 * lg + e < a.N ? s[i][j][e] : -INFINITY;
            }
            float mx = s[i][0][0];
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int e = 0; e < 4; ++e) mx = fmaxf(mx, s[i][j][e]);
            const float mnew = fmaxf(mrow[i], row4(mx, [](float x, float y) { return fmaxf(x, y); }));
            const float alpha = __builtin_amdgcn_exp2f((mrow[i] - mnew) * sl), ms = mnew * sl;  // alpha 0 on the first tile
            float sum = 0.f;
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    s[i][j][e] = __builtin_amdgcn_exp2f(fmaf(s[i][j][e], sl, -ms));
                    sum += s[i][j][e];
                }
            lrow[i] = lrow[i] * alpha + sum;
            mrow[i] = mnew;
#pragma unroll
            for (int d = 0; d < 4; ++d) o[i][d] *= alpha;
            // P^T's operand over the 32 keys of chunk c, numbered as the lanes hold them: index 8 lg + e is key
            // 32 c + 4 lg + e (e < 4) or 32 c + 16 + 4 lg + (e - 4)
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                uint32_t hw[4], lw[4];  // elements 2u, 2u + 1 of P's hi and lo halves
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    split_f16x2(s[i][2 * c + (u >> 1)][2 * (u & 1)], s[i][2 * c + (u >> 1)][2 * (u & 1) + 1], hw[u], lw[u]);
                ph[i][c] = __builtin_bit_cast(h16x8, u32x4{hw[0], hw[1], hw[2], hw[3]});
                pl[i][c] = __builtin_bit_cast(h16x8, u32x4{lw[0], lw[1], lw[2], lw[3]});
            }
        }
        // O^T += V^T P^T: A operand lane holds V^T[16 d + lr][the keys above]
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            h16x8 fh[4], fl[4];
#pragma unroll
            for (int d = 0; d < 4; ++d) {
                fh[d] = frag(16 + (c * 4 + d) * 2);
                fl[d] = frag(16 + (c * 4 + d) * 2 + 1);
            }
#pragma unroll
            for (int i = 0; i < QT; ++i) mfma3(fh, fl, ph[i][c], pl[i][c], o[i]);
        }
    };
    const int ntile = (a.N + 63) / 64, niter = (ntile + KS - 1) / KS;  // the same count in every group: barriers stay uniform
    // the two waves of a SIMD out of step: one's softmax runs beside the other's MFMAs (2 x 16 heads of 1000: 33.4 -> 32.5 us)
    if (wave >= W * KS / 2) __builtin_amdgcn_s_setprio(1);
    issue(min(kh, ntile - 1), 0);
    for (int it = 0; it < niter; ++it) {
        const int tile = it * KS + kh;
        wait_step<0>();  // this wave's DMAs of the tile landed, and its reads of the stage the next DMAs fill returned
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if (it + 1 < niter) issue(min(tile + KS, ntile - 1), (it + 1) & 1);
        if (KS == 1 || tile < ntile) compute(st + (it & 1) * kF5Tile, tile * 64);  // a group past the keys only keeps the barriers
    }
    if constexpr (KS > 1) {  // merge the other groups' (max, sum, O) into the first's through LDS
        constexpr int LD = 64 * QT;
        __syncthreads();
        float *mg = reinterpret_cast<float *>(lds) + (qw * 18) * LD + lane;
        float *own = mg + (kh - 1) * W * 18 * LD;
        if (kh > 0) {
#pragma unroll
            for (int i = 0; i < QT; ++i) {
                own[64 * i] = mrow[i];
                own[64 * i + LD] = lrow[i];
#pragma unroll
                for (int d = 0; d < 4; ++d)
#pragma unroll
                    for (int e = 0; e < 4; ++e) own[64 * i + (2 + 4 * d + e) * LD] = o[i][d][e];
            }
        }
        __syncthreads();
        if (kh > 0) return;
        for (int k = 1; k < KS; ++k, mg += W * 18 * LD)
#pragma unroll
            for (int i = 0; i < QT; ++i) {
                const float m1 = mg[64 * i], l1 = mg[64 * i + LD], mn = fmaxf(mrow[i], m1);
                const float a0 = __builtin_amdgcn_exp2f((mrow[i] - mn) * sl), a1 = __builtin_amdgcn_exp2f((m1 - mn) * sl);
                mrow[i] = mn;
                lrow[i] = lrow[i] * a0 + l1 * a1;
#pragma unroll
                for (int d = 0; d < 4; ++d)
#pragma unroll
                    for (int e = 0; e < 4; ++e) o[i][d][e] = o[i][d][e] * a0 + mg[64 * i + (2 + 4 * d + e) * LD] * a1;
            }
    }
#pragma unroll
    for (int i = 0; i < QT; ++i) {
        const int qr = q0 + 16 * i + lr;
        const float inv = 1.0f / row4(lrow[i], [](float x, float y) { return x + y; });
        if (qr >= a.N) continue;
        const int64_t orow = int64_t(b) * a.N + qr;
        const int ocol = h * kF5Hd + 4 * lg;
#pragma unroll
        for (int d = 0; d < 4; ++d) {
            const f32x4a y = o[i][d] * inv;
            if (a.out16) {
                uint32_t hi[2], lo[2];
                split_f16x2(y[0], y[1], hi[0], lo[0]);
                split_f16x2(y[2], y[3], hi[1], lo[1]);
                _Float16 *o16 = a.out16 + plane_off(orow, ocol + 16 * d, a.ldo);
                *reinterpret_cast<uint2 *>(o16) = uint2{hi[0], hi[1]};
                *reinterpret_cast<uint2 *>(o16 + kPlaneLo) = uint2{lo[0], lo[1]};
            } else {
                *reinterpret_cast<f32x4a *>(a.out + orow * a.ldo + ocol + 16 * d) = y;
            }
        }
    }
}

}  // namespace vh
