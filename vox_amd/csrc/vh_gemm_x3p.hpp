// vh_gemm_x3p.hpp — F32 weights on the f16 matrix cores with the weights already split and in fragment order.
#pragma once
#include "vh_gemm_epi.hpp"

namespace vh {

// F32 weights and f32 activations on the f16 matrix cores, as k_gemm_x3 takes them (both as f16 halves, three products
// per pair, the weights scaled by 2^10), for weights laid
// out once by k_pack_x3 in the order the MFMA reads them: [n / 16][k / 32][hi, lo][lane][8]. A wave then loads its W
// fragments straight into registers, 1 KiB of consecutive bytes per load and plane, and only A goes through LDS: f32
// loads two K steps of 64 ahead (two register sets), split on the way into one of two LDS stages of the same fragment
// order (reads without bank conflicts), one barrier per step.
//
// What bounds it: k_gemm_x3 split W again in every block (a quarter of its VALU work), had one K step of 32 in flight and
// two barriers a step, about 1.2 us each whatever the block count. Here a K step of 64 takes 0.45 us with 120 blocks; large
// grids are bound by the split's VALU work and the LDS and L1 reads together. Eight waves per 64 x 64 tile
// (32 x 16 outputs each) halve each wave's share of the split. Measured, k_gemm_x3 against this kernel (us):
// 2560 x 384, K 2688 (streaming conv) 95.6 -> 31.8; 10240 x 192, K 1344 62.4 -> 29.7; 30720 x 96, K 672 with Snake 55.9 -> 35.3;
// 333 x 64 x 16 groups, K 1984 78.3 -> 16.9; 1024 x 256, K 768 14.9 -> 8.3; 160 x 384, K 384 14.1 -> 5.0.
//
// Block: WM x WN waves of 16 TM x 16 TN outputs; W is the MFMA's A operand, the activations its B (epi_tile's layout).
// A sources as k_gemm_f32 (rows, grouped "same" / causal conv, streaming conv); HIST: this block's rows reach into the
// history of a streaming conv. All offsets fit 31 bits and K cig < 2^32 (the launcher checks), so a column's tap is one
// multiply by g.cig_magic.
template <int EPI, int ASRC, int WM, int WN, int TM, int TN, bool HIST>
VH_DEV void x3p_body(const uint8_t *__restrict__ w, const float *__restrict__ A, const GemmArgs &g, int m0, int n0, int grp, int kbeg,
                     int kend, _Float16 *lds) {
    constexpr int BK = 64, NW = WM * WN, RB = TM * WM;  // 16-row blocks
    constexpr int QW = 4 * RB / NW;                     // 16-column pieces of its row block that a wave stages
    constexpr int STG = RB * 2 * 2 * 512;               // halves of one LDS stage: [row block][k32][hi, lo][512]
    static_assert(NW % RB == 0 && QW >= 1, "row blocks shared out over the waves");
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, wm = wave / WN, wn = wave % WN, lr = lane & 15, lg = lane >> 4;
    const int rb = wave % RB, q0 = wave / RB * QW;
    const int K32 = (g.K + 31) / 32;
    // A: this thread's rows (16 (wave + 4 p) + lane / 4), columns 16 q + 4 (lane % 4)
    const int ar = lane >> 2, ac = (lane & 3) * 4;
    const int32_t xrows = g.m;
    const __amdgpu_buffer_rsrc_t rx = buf_rsrc(A, int32_t(((xrows - 1) * g.lda + (ASRC == ASRC_CONV ? g.lda : ASRC == ASRC_STREAM ? g.cig : g.K)) * 4));
    const __amdgpu_buffer_rsrc_t rhist = buf_rsrc(HIST ? g.hist : A, HIST ? g.ctx * g.cig * 4 : 0);
    const int row = m0 + 16 * rb + ar, srow = ASRC == ASRC_CONV ? row % g.seq : 0;
    const bool rin = row < g.m;
    f32x4v ra[2][QW];
    auto fetch_a = [&](f32x4v(&a)[QW], int k0) {
        constexpr int32_t kOut = 0x7FFFFFF0;  // past every buffer: reads zeros
#pragma unroll
        for (int u = 0; u < QW; ++u) {
            const int k = k0 + 16 * (q0 + u) + ac;
            const bool in = rin && k < kend;
            if (ASRC == ASRC_ROWS) {
                a[u] = __builtin_bit_cast(f32x4v, buf_ld16(rx, in ? int32_t((row * g.lda + k) * 4) : kOut, 0));
                continue;
            }
            const int kt = int(__umulhi(uint32_t(k), g.cig_magic)), i = k - kt * g.cig;
            if (ASRC == ASRC_STREAM) {
                const int r = row + kt * g.dil - g.ctx;
                a[u] = __builtin_bit_cast(f32x4v, buf_ld16(rx, in && (!HIST || r >= 0) ? int32_t((r * g.lda + i) * 4) : kOut, 0));
                if (HIST) {
                    const u32x4 h = buf_ld16(rhist, in && r < 0 ? ((r + g.ctx) * g.cig + i) * 4 : kOut, 0);
                    a[u] = __builtin_bit_cast(f32x4v, __builtin_bit_cast(u32x4, a[u]) | h);
                }
            } else {
                const int d = kt - (g.causal ? g.ksize - 1 : g.ksize / 2), tt = srow + d;
                const bool inc = in && kt < g.ksize && tt >= 0 && tt < g.seq;
                a[u] = __builtin_bit_cast(f32x4v, buf_ld16(rx, inc ? int32_t(((row + d) * g.lda + grp * g.cig + i) * 4) : kOut, 0));
            }
        }
    };
    uint32_t mn = 0xFFFFFFFFu;
    auto stage_a = [&](const f32x4v(&a)[QW], int buf) {
#pragma unroll
        for (int u = 0; u < QW; ++u) {
            const int q = q0 + u;
            uint2 hi, lo;
            mn = ovf4(a[u], mn);
            split4(a[u], hi, lo);
            // row block, k32 = q / 2, lane group 2 (q % 2) + ac / 8, its lane's row, half ac % 8
            _Float16 *d = lds + buf * STG + (rb * 2 + (q >> 1)) * 1024 + ((2 * (q & 1) + (ac >> 3)) * 16 + ar) * 8 + (ac & 7);
            *reinterpret_cast<uint2 *>(d) = hi;
            *reinterpret_cast<uint2 *>(d + 512) = lo;
        }
    };
    // W: fragment order, [n / 16][k / 32][hi, lo][lane][8]
    const int ntile = (g.n + 15) / 16;
    const __amdgpu_buffer_rsrc_t rw = buf_rsrc(w, int32_t(int64_t(ntile) * K32 * 2048));
    int vw[TN];
#pragma unroll
    for (int j = 0; j < TN; ++j) {
        const int t = n0 / 16 + wn * TN + j;
        vw[j] = t < ntile ? t * K32 * 2048 + 16 * lane : 0x7FFFFFF0;
    }
    u32x4 bh[2][2][TN], bl[2][2][TN];
    auto fetch_w = [&](int d, int k0) {
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const int so = min(k0 / 32 + q, K32 - 1) * 2048;
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                bh[d][q][j] = buf_ld16(rw, vw[j], so);
                bl[d][q][j] = buf_ld16(rw, vw[j], so + 1024);
            }
        }
    };
    // hi.hi and the two cross products in accumulators of their own: the cross terms, 2^-11 of the sum, then add no
    // rounding of the sum's size (one rounding a step instead of three)
    f32x4v acc[TM][TN], acx[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = acx[i][j] = f32x4v{0.f, 0.f, 0.f, 0.f};
    auto mma = [&](int d) {
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            f16x8v ah[TM], al[TM];
#pragma unroll
            for (int i = 0; i < TM; ++i) {
                const _Float16 *p = lds + d * STG + ((wm * TM + i) * 2 + q) * 1024 + lane * 8;
                ah[i] = *reinterpret_cast<const f16x8v *>(p);
                al[i] = *reinterpret_cast<const f16x8v *>(p + 512);
            }
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j) {
                    const f16x8v BH = __builtin_bit_cast(f16x8v, bh[d][q][j]), BL = __builtin_bit_cast(f16x8v, bl[d][q][j]);
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(BH, ah[i], acc[i][j], 0, 0, 0);
                    acx[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(BL, ah[i], acx[i][j], 0, 0, 0);
                    acx[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(BH, al[i], acx[i][j], 0, 0, 0);
                }
        }
    };
    const int ns = (kend - kbeg + BK - 1) / BK;
    const int rbase = m0 + 16 * wm * TM + lr, cbase = n0 + 16 * wn * TN + 4 * lg;
    fetch_a(ra[0], kbeg);
    fetch_w(0, kbeg);
    __builtin_amdgcn_sched_barrier(0);
    fetch_a(ra[1], kbeg + BK);
    fetch_w(1, kbeg + BK);
    __builtin_amdgcn_sched_barrier(0);
    for (int s = 0; s < ns; s += 2) {
#pragma unroll
        for (int d = 0; d < 2; ++d) {
            if (d == 1 && s + 1 >= ns) break;
            stage_a(ra[d], d);
            fetch_a(ra[d], kbeg + (s + d + 2) * BK);
            __syncthreads();
            mma(d);
            fetch_w(d, kbeg + (s + d + 2) * BK);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    raise_status(g.status, mn < kOvfSpan, kStatusF16Range);
    constexpr float kWsInv = 1.0f / 1024.0f;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = (acc[i][j] + acx[i][j]) * kWsInv;
    if (g.kchunk) {
        float *ws = g.ws + int64_t(blockIdx.z) * g.m * g.n;
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
                store_partial(acc[i][j], ws, g, rbase + 16 * i, cbase + 16 * j);
        return;
    }
    bool bad = false;
    EpiOps<EPI, TM, TN> ops;  // here, not before the loop: its registers are the loop's own
    ops.load(g, rbase, cbase);
    ops.finish(acc, g, rbase, cbase, lane, bad);
    raise_status(g.status, bad, kStatusF16Range);
}

template <int EPI, int ASRC, int WM, int WN, int TM, int TN>
__global__ __launch_bounds__(64 * WM * WN) void k_gemm_x3p(const uint8_t *__restrict__ w, const float *__restrict__ A, GemmArgs g) {
    __shared__ __align__(16) _Float16 lds[2 * (WM * TM) * 2 * 2 * 512];
    const int grp = g.kchunk ? 0 : int(blockIdx.z);
    const int kbeg = g.kchunk ? int(blockIdx.z) * g.kchunk : 0, kend = g.kchunk ? min(g.K, kbeg + g.kchunk) : g.K;
    int tm, tn;
    gemm_tile(gridDim.x, gridDim.y, g.n > g.m, tm, tn);
    const int m0 = tm * 16 * TM * WM, n0 = tn * 16 * TN * WN;
    if (ASRC == ASRC_CONV) {
        w += int64_t(grp) * ((g.n + 15) / 16) * ((g.K + 31) / 32) * 2048;
        g.y += int64_t(grp) * g.n;
        if (g.bias) g.bias += int64_t(grp) * g.n;
    }
    if (ASRC == ASRC_STREAM && g.hist_next) stream_hist_next(A, g);  // the history moves on in the same launch
    if (ASRC == ASRC_STREAM && m0 < g.ctx) x3p_body<EPI, ASRC, WM, WN, TM, TN, true>(w, A, g, m0, n0, grp, kbeg, kend, lds);
    else x3p_body<EPI, ASRC, WM, WN, TM, TN, false>(w, A, g, m0, n0, grp, kbeg, kend, lds);
}

// F32 weights [n][K] (2^10 w split into f16 halves, as k_gemm_x3 splits them) in fragment order: [n / 16][k / 32][hi,
// lo][lane][8], zeros past n and K. One thread per 8 columns of a row.
__global__ __launch_bounds__(256) void k_pack_x3(const float *__restrict__ w, int64_t n, int32_t K, _Float16 *__restrict__ out) {
    const int K32 = (K + 31) / 32;
    const int64_t t = int64_t(blockIdx.x) * 256 + threadIdx.x, tile = t / 64;
    if (tile >= (n + 15) / 16 * K32) return;
    const int lane = int(t % 64);
    const int64_t r = tile / K32 * 16 + (lane & 15);
    const int k = int(tile % K32) * 32 + 8 * (lane >> 4);
    f16x8v hi, lo;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        _Float16 h = 0, l = 0;
        if (r < n && k + e < K) (void)split_f16(w[r * K + k + e] * 1024.0f, h, l);
        hi[e] = h;
        lo[e] = l;
    }
    *reinterpret_cast<f16x8v *>(out + tile * 1024 + lane * 8) = hi;
    *reinterpret_cast<f16x8v *>(out + tile * 1024 + 512 + lane * 8) = lo;
}

}  // namespace vh
