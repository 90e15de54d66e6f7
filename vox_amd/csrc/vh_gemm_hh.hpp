// vh_gemm_hh.hpp — the split-f16 MFMA GEMM of passes whose producers already split the activations (F5 and estimator
// blocks, prefill planes): both operands in MFMA fragment order, fed by LDS DMA.
#pragma once
#include "vh_gemm_epi.hpp"

namespace vh {

// y = A W^T with A = hi + lo (g.a16, plane_off's layout of m rows of K halves and planes) and W f16 in fragment order
// (launch_pack_f16: [n / 16][k / 32][lane][8]), or (Q8) the int8 values of Q8 weights as f16 in that order with their
// block scales transposed, [K / 32][ceil64(n)]; K a multiple of 64. Each f16 x f16 product is exact in the f32
// accumulator. F16: the hi and lo products accumulate apart (the lo ones, 2^-11 of the sum, then add no rounding of the
// sum's size). Q8: a 32-deep step is one scale block, so its two MFMAs start from zero and the block sum is scaled into the
// accumulator: s (q . a) for the reference's (float(q) s) . a, equal up to rounding.
//
// Per step of 32 columns a block copies 16-row fragments of A (hi, lo) and W, 1 KiB of consecutive bytes each, to one of S
// LDS stages by DMA, up to S - 1 steps ahead; a wave reads its fragments of step s (1 KiB per read, no bank conflicts)
// while the MFMAs of step s - 1 run; one barrier a step. A stage is refilled only after the barrier that follows the last
// reads of it (wait_step has them returned before the barrier).
//
// What bounds it: the row-major planes it replaces cost 16 rows of 64 bytes per load, a third of the rate of 1 KiB runs;
// with them gone, per step of a 64 x 128 tile about 0.26 us with one block per CU: its DMAs alone (no reads, no MFMAs) take
// 0.19, its reads and MFMAs alone 0.23, the MFMAs 0.11 at the nominal rate; S = 5 or 8 is no faster than 3, so neither is
// the load latency it. Against the register-staged kernel on row-major planes (us, f32 store): 2000 x 3072, K 1024 41.3 ->
// 30.7; 2000 x 2048, K 1024 27.0 -> 20.9; 2000 x 1024, K 2048 27.6 -> 22.5; 2000 x 1024, K 1024 16.8 -> 12.9; 333 x 3072,
// K 1024 14.6 -> 10.9; 333 x 1024, K 2048 12.4 -> 10.4; 1024 x 1024, K 256 6.8 -> 5.3. In the DiT step (2 x 1000 frames)
// the epilogues' operands were a third of the time of the products that add into y; EpiOps loads them before the loop
// (whole step 3.82 -> 3.72 ms).
//
// Block: WM x WN waves of 16 TM x 16 TN outputs; W is the MFMA's A operand (epi_tile's layout). g.kchunk: slice blockIdx.z
// of K (a multiple of 64) as partial sums into g.ws.
template <int EPI, int TM, int TN, int WM, int WN, int S, bool Q8>
__global__ __launch_bounds__(64 * WM * WN, 2) void k_gemm_hh(const _Float16 *__restrict__ w, const float *__restrict__ scale_t, GemmArgs g) {
    constexpr int NW = WM * WN, RA = TM * WM, RW = TN * WN;  // waves; 16-row blocks of A and of W
    constexpr int PA = 2 * RA / NW, PB = RW / NW, PW = PA + PB + (Q8 ? 1 : 0);  // DMAs per wave and step
    constexpr int STAGE = (2 * RA + RW) * 1024 + (Q8 ? (RW + 3) / 4 * 256 : 0);
    static_assert(2 * RA % NW == 0 && RW % NW == 0 && (RW % 4 == 0 || RW < 4), "every wave issues the same DMAs");
    __shared__ __align__(1024) uint8_t lds[S * STAGE];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), wm = wave / WN, wn = wave % WN;
    const int lr = lane & 15, lg = lane >> 4;
    int tm, tn;  // A as two f16 planes (4 bytes an element) against W f16 (2)
    gemm_tile(gridDim.x, gridDim.y, g.n > 2 * g.m, tm, tn);
    const int m0 = tm * RA * 16, n0 = tn * RW * 16, K32 = g.K / 32;
    const int mb = (g.m + 15) / 16 - m0 / 16, nb = (g.n + 15) / 16 - n0 / 16, ns64 = (g.n + 63) / 64 * 64;
    const u32x4s ra = dma_rsrc(g.a16 + int64_t(m0) * g.K * 2), rw = dma_rsrc(w + int64_t(n0) * g.K), rs = dma_rsrc(Q8 ? static_cast<const void *>(scale_t) : w);
    // this wave's fragments of a stage (block rows past the last read the last: their outputs are not stored)
    int ca[PA], cw[PB];
    uint32_t da[PA], dw[PB];
    const uint32_t base = uint32_t(reinterpret_cast<uintptr_t>((lds_void *)lds));
#pragma unroll
    for (int p = 0; p < PA; ++p) {
        const int r = wave + NW * p;
        ca[p] = min(r / 2, mb - 1) * K32 * 2048 + (r & 1) * 1024;
        da[p] = base + r * 1024;
    }
#pragma unroll
    for (int p = 0; p < PB; ++p) {
        const int r = wave + NW * p;
        cw[p] = min(r, nb - 1) * K32 * 1024;
        dw[p] = base + (2 * RA + r) * 1024;
    }
    // Q8: the scales of the 64 columns that hold this wave's (waves that share them write the same values)
    const int s64 = wn * TN / 4;
    const uint32_t ds = base + (2 * RA + RW) * 1024 + s64 * 256;
    const int vo = lane * 16, vs = min(n0 + s64 * 64 + lane, ns64 - 1) * 4;
    auto issue = [&](int buf, int step) {
#pragma unroll
        for (int p = 0; p < PA; ++p) dma_b128(ra, da[p] + buf * STAGE, vo, ca[p] + step * 2048);
#pragma unroll
        for (int p = 0; p < PB; ++p) dma_b128(rw, dw[p] + buf * STAGE, vo, cw[p] + step * 1024);
        if (Q8) dma_b32(rs, ds + buf * STAGE, vs, step * ns64 * 4);
    };
    constexpr int XM = Q8 ? 1 : TM, XN = Q8 ? 1 : TN;
    f32x4v acc[TM][TN], acx[XM][XN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            acc[i][j] = f32x4v{0.f, 0.f, 0.f, 0.f};
            if (!Q8) acx[i % XM][j % XN] = f32x4v{0.f, 0.f, 0.f, 0.f};
        }
    f16x8v fh[2][TM], fl[2][TM], fb[2][TN];
    f32x4v fs[2][TN];
    auto read = [&](int f, int buf) {
        const uint8_t *st = lds + buf * STAGE;
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            fh[f][i] = *reinterpret_cast<const f16x8v *>(st + (wm * TM + i) * 2048 + vo);
            fl[f][i] = *reinterpret_cast<const f16x8v *>(st + (wm * TM + i) * 2048 + 1024 + vo);
        }
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            fb[f][j] = *reinterpret_cast<const f16x8v *>(st + (2 * RA + wn * TN + j) * 1024 + vo);
            if (Q8) fs[f][j] = *reinterpret_cast<const f32x4v *>(st + (2 * RA + RW) * 1024 + (wn * TN + j) * 64 + lg * 16);
        }
    };
    auto mma = [&](int f) {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                if constexpr (Q8) {
                    f32x4v t = {0.f, 0.f, 0.f, 0.f};
                    t = __builtin_amdgcn_mfma_f32_16x16x32_f16(fb[f][j], fh[f][i], t, 0, 0, 0);
                    t = __builtin_amdgcn_mfma_f32_16x16x32_f16(fb[f][j], fl[f][i], t, 0, 0, 0);
#pragma unroll
                    for (int v = 0; v < 4; ++v) acc[i][j][v] = fmaf(t[v], fs[f][j][v], acc[i][j][v]);
                } else {
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fb[f][j], fh[f][i], acc[i][j], 0, 0, 0);
                    acx[i % XM][j % XN] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fb[f][j], fl[f][i], acx[i % XM][j % XN], 0, 0, 0);
                }
            }
    };
    const int s0 = g.kchunk ? int(blockIdx.z) * (g.kchunk / 32) : 0, s1 = g.kchunk ? min(K32, s0 + g.kchunk / 32) : K32;  // s1 - s0 even
    const int rbase = m0 + 16 * wm * TM + lr, cbase = n0 + 16 * wn * TN + 4 * lg;
    EpiOps<EPI, TM, TN> ops;
    if (!g.kchunk) ops.load(g, rbase, cbase);
#pragma unroll
    for (int s = 0; s < S - 1; ++s) issue(s, min(s0 + s, s1 - 1));
    int buf = 0;
    auto step = [&](int s, int f) {  // stage of step s landed: the next one's DMA starts, its fragments go to set f
        wait_step<(S - 2) * PW>();
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        issue(buf == 0 ? S - 1 : buf - 1, min(s + S - 1, s1 - 1));  // past the end: the last step again (exact wait counts)
        read(f, buf);
        buf = buf == S - 1 ? 0 : buf + 1;
    };
    step(s0, 0);
    for (int s = s0 + 1; s + 1 < s1; s += 2) {
        step(s, 1);
        mma(0);
        step(s + 1, 0);
        mma(1);
    }
    step(s1 - 1, 1);
    mma(0);
    mma(1);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no DMA is in flight when the block's LDS is given back
    if (!Q8) {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) acc[i][j] += acx[i % XM][j % XN];
    }
    if (g.kchunk) {
        float *ws = g.ws + int64_t(blockIdx.z) * g.m * g.n;
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) store_partial(acc[i][j], ws, g, rbase + 16 * i, cbase + 16 * j);
        return;
    }
    bool bad = false;
    ops.finish(acc, g, rbase, cbase, lane, bad);
    raise_status(g.status, bad, kStatusF16Range);
}

// f16 weights [n][K] (or the int8 values of Q8 weights, as f16) in fragment order, zeros past n: one thread per 8 columns of
// a row. K % 32 == 0.
template <bool Q8>
__global__ __launch_bounds__(256) void k_pack_f16(const uint8_t *__restrict__ w, int64_t n, int32_t K, _Float16 *__restrict__ out) {
    const int64_t t = int64_t(blockIdx.x) * 256 + threadIdx.x, tile = t / 64;
    if (tile >= (n + 15) / 16 * (K / 32)) return;
    const int lane = int(t % 64);
    const int64_t r = tile / (K / 32) * 16 + (lane & 15);
    const int64_t src = r * K + tile % (K / 32) * 32 + 8 * (lane >> 4);
    f16x8v v = {0, 0, 0, 0, 0, 0, 0, 0};
    if (r < n) {
        if (Q8) {
            const uint2 u = *reinterpret_cast<const uint2 *>(w + src);
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = _Float16(int8_t((e < 4 ? u.x : u.y) >> (8 * (e & 3))));
        } else {
            v = *reinterpret_cast<const f16x8v *>(w + src * 2);
        }
    }
    *reinterpret_cast<f16x8v *>(out + tile * 512 + lane * 8) = v;
}

// Block scales [n][nb] as [nb][ns] (ns >= n, zeros past n).
__global__ __launch_bounds__(256) void k_scale_t(const float *__restrict__ s, int64_t n, int32_t nb, int64_t ns, float *__restrict__ out) {
    const int64_t t = int64_t(blockIdx.x) * 256 + threadIdx.x;
    if (t >= ns * nb) return;
    const int64_t r = t % ns, b = t / ns;
    out[t] = r < n ? s[r * nb + b] : 0.f;
}

// f16 planes hi, lo ([m][K] each) in plane_off's layout (the benchmark's operand).
__global__ __launch_bounds__(256) void k_pack_planes(const _Float16 *__restrict__ hi, const _Float16 *__restrict__ lo, int64_t m, int32_t K,
                                                     _Float16 *__restrict__ out) {
    const int64_t t = int64_t(blockIdx.x) * 256 + threadIdx.x;
    if (t >= m * K) return;
    const int64_t r = t / K, o = plane_off(r, int(t % K), K);
    out[o] = hi[t];
    out[o + kPlaneLo] = lo[t];
}

// The split-K slices of an EPI_ACC product added into its rows, y[row][c] += (sum_z ws[z][row][c]) + bias[c], as
// k_gemm_splitk_reduce<EPI_ACC> does, then the RMSNorm (gamma, eps) of each updated row into f16 planes of n
// columns with k_rmsnorm_rows_h16's arithmetic: the residual add and the next norm in one pass over the row. grid m,
// block 256, n <= 256 NV, n % 32 == 0, splits <= 8.
template <int NV>
__global__ __launch_bounds__(256) void k_splitk_acc_rms_h16(GemmArgs g, int32_t splits, const float *gamma, float eps,
                                                           _Float16 *out16) {
    __shared__ float red[4];
    const int row = int(blockIdx.x);
    const int64_t slice = int64_t(g.m) * g.n;
    float *yr = g.y + int64_t(row) * g.ldy;
    // every slice's value and the row's own first, so the loads are in flight together (slices past `splits`, at
    // most kMaxSplits, read slice 0 and are left out), then the sums in split order as the reduce kernel adds them
    constexpr int kMaxSplits = 8;
    float t[NV][kMaxSplits], hv[NV];
#pragma unroll
    for (int k = 0; k < NV; ++k) {
        const int c = min(int(threadIdx.x) + 256 * k, g.n - 1);
        hv[k] = yr[c];
#pragma unroll
        for (int z = 0; z < kMaxSplits; ++z) t[k][z] = g.ws[(z < splits ? z : 0) * slice + int64_t(row) * g.n + c];
    }
    float ss = 0.f;
#pragma unroll
    for (int k = 0; k < NV; ++k) {
        const int c = int(threadIdx.x) + 256 * k;
        if (c < g.n) {
            float v = 0.f;
#pragma unroll
            for (int z = 0; z < kMaxSplits; ++z)
                if (z < splits) v += t[k][z];
            v = v + (g.bias ? g.bias[c] : 0.f);
            hv[k] = hv[k] + v;
            yr[c] = hv[k];
            ss = fmaf(hv[k], hv[k], ss);
        } else {
            hv[k] = 0.f;
        }
    }
    ss = block_sum<256>(ss, red);
    const float inv = 1.0f / sqrtf(ss / float(g.n) + eps);
    bool bad = false;
#pragma unroll
    for (int k = 0; k < NV; ++k) {
        const int c = int(threadIdx.x) + 256 * k;
        if (c < g.n) {
            _Float16 hi, lo;
            bad |= split_f16(gamma[c] * (hv[k] * inv), hi, lo);
            _Float16 *o = out16 + plane_off(row, c, g.n);
            o[0] = hi;
            o[kPlaneLo] = lo;
        }
    }
    raise_status(g.status, bad, kStatusF16Range);
}

}  // namespace vh
