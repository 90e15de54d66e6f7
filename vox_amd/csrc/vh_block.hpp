// vh_block.hpp — the row-local part of a transformer block of 256 channels (the flow estimator's) in one kernel.
#pragma once
#include <type_traits>

#include "vh_gemm_epi.hpp"

namespace vh {

// x += A Wo^T + bo; h = gelu_erf(LN(x) W1^T + b1); x += h W2^T + b2; out16 = the next LN of x (when asked), for 16 rows per
// block: A, LN(x), h and out16 are f16 planes (plane_off's layout), the three products split-f16 as k_gemm_hh's (W in its
// fragment order, the hi and lo products apart), the norms those of k_norm_rows. A, LN(x) and h stay in LDS in fragment
// order; x stays in registers.
//
// Each of the 8 waves owns 32 channels of x and, per 256 columns of h, 32 of them, so no wave reads another's weights: they
// go from L2 straight to registers, 8 steps ahead across all three products (2 KiB per step and wave, 128 KiB in flight per
// CU), and the waves meet only at the norms and around h.
//
// NS > 1 blocks share 16 rows: each takes A Wo^T and LN(x) whole and 1 / NS of the columns of h, and the last of them to
// finish adds the NS partial products h W2^T, in their order, and does the rest.
//
// What bounds it: the weights through one CU, at about 50 bytes a clock (16 KiB a step in 0.13 us; without the GELU, or with
// half the MFMAs, it is 0.3 us faster): 1.25 MB at inner 512, ff 1024 with one block per 16 rows, 0.5 MB with four. The five
// launches it replaces (o, norm, ff1, ff2, norm) took about 29 us in the estimator's step at 202 and at 1024 rows, one block per
// 16 rows 18.8 and 18.2, four 13.7 and 15.6.
constexpr int kTailC = 256, kTailRed = 8 * 16 * 2;  // doubles of one norm's partial moments
inline size_t block_tail_smem(int inner, int ff) {  // ff: a block's part
    return size_t(inner > ff ? inner : ff) * 64 + kTailC * 64 + 2 * kTailRed * sizeof(double);
}

template <int NS>
__global__ __launch_bounds__(512, 2) void k_block_tail(BlockTailArgs a) {
    constexpr int PF = 8, FS = 1024;  // weight steps in flight; bytes of a fragment
    extern __shared__ __align__(16) uint8_t lds[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6), lr = lane & 15, lg = lane >> 4;
    // blocks of one tile are 8 apart, on one XCD where blocks go round-robin
    const int tile = NS == 1 ? int(blockIdx.x) : int(blockIdx.x) / (8 * NS) * 8 + int(blockIdx.x) % 8, part = NS == 1 ? 0 : int(blockIdx.x) / 8 % NS;
    if (NS > 1 && tile * 16 >= a.R) return;
    const int row = tile * 16 + lr, rc = min(row, a.R - 1), vo = lane * 16;
    const bool rin = row < a.R;
    const int KI = a.inner / 32, KF = a.ff / 32, FF = a.ff / NS, c0 = wave * 32 + 4 * lg;  // this lane's channels: c0 .. + 3, c0 + 16 .. + 19
    uint8_t *act = lds, *xn = lds + max(a.inner, FF) * 64;                 // A, then this block's part of h; LN(x)
    double *red = reinterpret_cast<double *>(xn + kTailC * 64);
    auto frag = [&](const _Float16 *w, int f, int K32) { return reinterpret_cast<const uint8_t *>(w) + int64_t(f) * K32 * FS + vo; };
    auto sync = [&] { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); __builtin_amdgcn_s_barrier(); asm volatile("" ::: "memory"); };

    // everything the first product needs is on its way before the first wait: A's 16 rows (2 KiB per 32 columns,
    // consecutive; 16 KiB per 256 columns), x, the parameters, the first weights
    const uint8_t *src = reinterpret_cast<const uint8_t *>(a.a16) + int64_t(tile) * a.inner * 64 + threadIdx.x * 16;
    constexpr int AP = 4;
    u32x4 ar[AP];
#pragma unroll
    for (int i = 0; i < AP; ++i) ar[i] = *reinterpret_cast<const u32x4 *>(src + min(i * 8192, a.inner * 64 - 8192));
    f32x4v x[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) x[j] = *reinterpret_cast<const f32x4v *>(a.x + int64_t(rc) * kTailC + c0 + 16 * j);
    // four values of v; of any vector when v is null: the uses select (a select here would wait for the load here)
    auto vec = [&](const float *v, int c) { return *reinterpret_cast<const f32x4v *>(v ? v + c : a.lw); };
    const f32x4v zero = {0.f, 0.f, 0.f, 0.f};
    f32x4v bias[2], lw[2], lb[2], n[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        bias[j] = vec(a.bo, c0 + 16 * j);
        lw[j] = vec(a.lw, c0 + 16 * j);
        lb[j] = vec(a.lb, c0 + 16 * j);
    }
    asm volatile("" ::: "memory");  // the weights are the newest loads in flight
    f16x8v w[PF][2];
    const uint8_t *p = frag(a.wo, 2 * wave, KI);
#pragma unroll
    for (int u = 0; u < PF; ++u)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            w[u][j] = *reinterpret_cast<const f16x8v *>(p + (j * KI + u) * FS);
            __builtin_amdgcn_sched_barrier(0);
        }
    asm volatile("" ::: "memory");  // the loads above stay above the stores to LDS
#pragma unroll
    for (int i = 0; i < AP; ++i)
        if (i * 8192 < a.inner * 64) *reinterpret_cast<u32x4 *>(act + i * 8192 + threadIdx.x * 16) = ar[i];
    for (int i = AP * 8192; i < a.inner * 64; i += 8192)
        *reinterpret_cast<u32x4 *>(act + i + threadIdx.x * 16) = *reinterpret_cast<const u32x4 *>(src + i);

    f32x4v acc[2], acx[2];
    // acc = the product of the rows at `rows` (LDS, `steps` 32-column tiles) with this wave's two fragment rows (K32 tiles
    // each) at cur; the last PF steps fetch the first ones of the next product (next). The order within a step is pinned: the next
    // tile's LDS reads, this one's MFMAs, the weights PF steps on, so a wait for weights leaves the newer ones in flight.
    auto product = [&](auto has_next, const uint8_t *rows, int steps, const uint8_t *cur, int K32, const uint8_t *next, int next_K32) {
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[j] = acx[j] = f32x4v{0.f, 0.f, 0.f, 0.f};
        const uint8_t *r = rows + vo, *last = r + (steps - 1) * 2048;
        f16x8v h = *reinterpret_cast<const f16x8v *>(r), l = *reinterpret_cast<const f16x8v *>(r + 1024);
        auto step = [&](int u) {
            r = r < last ? r + 2048 : last;
            const f16x8v hn = *reinterpret_cast<const f16x8v *>(r), ln = *reinterpret_cast<const f16x8v *>(r + 1024);
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(w[u][j], h, acc[j], 0, 0, 0);
                acx[j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(w[u][j], l, acx[j], 0, 0, 0);
            }
            h = hn;
            l = ln;
            __builtin_amdgcn_sched_barrier(0);
        };
        const uint8_t *q = cur + PF * FS;
        for (int s = PF; s < steps; s += PF, q += PF * FS)
#pragma unroll
            for (int u = 0; u < PF; ++u) {
                step(u);
#pragma unroll
                for (int j = 0; j < 2; ++j) w[u][j] = *reinterpret_cast<const f16x8v *>(q + (j * K32 + u) * FS);
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
        for (int u = 0; u < PF; ++u) {
            step(u);
            if constexpr (decltype(has_next)::value) {
#pragma unroll
                for (int j = 0; j < 2; ++j) w[u][j] = *reinterpret_cast<const f16x8v *>(next + (j * next_K32 + u) * FS);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[j] += acx[j];
    };
    bool bad = false;
    // LN of x (rows lr): each wave's 32 columns give (sum, squares about their own mean), merged by every wave. One barrier.
    auto norm = [&](double *rd, const f32x4v (&g)[2], const f32x4v (&b)[2], f32x4v (&n)[2]) {
        auto quad = [](double v) {  // over the four lanes of a row
            const uint64_t u = __builtin_bit_cast(uint64_t, v);
            const auto l = __builtin_amdgcn_permlane16_swap(uint32_t(u), uint32_t(u), false, false);
            const auto h = __builtin_amdgcn_permlane16_swap(uint32_t(u >> 32), uint32_t(u >> 32), false, false);
            v = __builtin_bit_cast(double, uint64_t(h[0]) << 32 | l[0]) + __builtin_bit_cast(double, uint64_t(h[1]) << 32 | l[1]);
            const uint64_t t = __builtin_bit_cast(uint64_t, v);
            const auto l2 = __builtin_amdgcn_permlane32_swap(uint32_t(t), uint32_t(t), false, false);
            const auto h2 = __builtin_amdgcn_permlane32_swap(uint32_t(t >> 32), uint32_t(t >> 32), false, false);
            return __builtin_bit_cast(double, uint64_t(h2[0]) << 32 | l2[0]) + __builtin_bit_cast(double, uint64_t(h2[1]) << 32 | l2[1]);
        };
        double s = 0.0, q = 0.0;
#pragma unroll
        for (int j = 0; j < 2; ++j) s += (double(x[j][0]) + double(x[j][1])) + (double(x[j][2]) + double(x[j][3]));
        s = quad(s);
        const double m = s / 32;
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const double d = double(x[j][e]) - m;
                q = __builtin_fma(d, d, q);
            }
        q = quad(q);
        if (lg == 0) {
            rd[(wave * 16 + lr) * 2] = s;
            rd[(wave * 16 + lr) * 2 + 1] = q;
        }
        sync();
        double S = 0.0, Q = 0.0;
#pragma unroll
        for (int v = 0; v < 8; ++v) S += rd[(v * 16 + lr) * 2];
        const double mean = S / kTailC;
#pragma unroll
        for (int v = 0; v < 8; ++v) {
            const double d = rd[(v * 16 + lr) * 2] / 32 - mean;
            Q += rd[(v * 16 + lr) * 2 + 1] + 32.0 * d * d;
        }
        const float inv = float(1.0 / sqrt(Q / kTailC + a.eps)), fm = float(mean);
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e) n[j][e] = (x[j][e] - fm) * inv * g[j][e] + b[j][e];
    };
    // four values of columns c .. c + 3 (in 32-column tiles of 2 KiB) as halves
    auto put = [&](uint8_t *dst, int c, f32x4v v) {
        uint2 hi, lo;
        const bool o = split_f16x4(v, hi, lo);
        bad |= o && rin;
        uint8_t *t = dst + (c >> 5) * 2048 + (((c >> 3) & 3) * 16 + lr) * 16 + (c & 7) * 2;
        *reinterpret_cast<uint2 *>(t) = hi;
        *reinterpret_cast<uint2 *>(t + 1024) = lo;
    };

    sync();
    const uint8_t *w1 = frag(a.w1, part * (FF / 16) + 2 * wave, 8), *w2 = frag(a.w2, 2 * wave, KF) + part * (FF / 32) * FS;
    product(std::true_type{}, act, KI, p, KI, w1, 8);
#pragma unroll
    for (int j = 0; j < 2; ++j) x[j] += acc[j] + (a.bo ? bias[j] : zero);
    norm(red, lw, lb, n);  // its barrier: every wave has read A, whose LDS h takes
#pragma unroll
    for (int j = 0; j < 2; ++j) put(xn, c0 + 16 * j, n[j]);
    sync();
    for (int f = 0; f < FF; f += 256) {
#pragma unroll
        for (int j = 0; j < 2; ++j) bias[j] = vec(a.b1, part * FF + f + c0 + 16 * j);
        const bool more = f + 256 < FF;
        const uint8_t *nw1 = w1 + 16 * 8 * FS;
        product(std::true_type{}, xn, 8, w1, 8, more ? nw1 : w2, more ? 8 : KF);
        w1 = nw1;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            f32x4v v = acc[j] + (a.b1 ? bias[j] : zero);
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = gelu_erf_f(v[e]);
            put(act, f + c0 + 16 * j, v);
        }
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        bias[j] = vec(a.b2, c0 + 16 * j);
        lw[j] = vec(a.nw, c0 + 16 * j);
        lb[j] = vec(a.nb, c0 + 16 * j);
    }
    sync();
    product(std::false_type{}, act, FF / 32, w2, KF, nullptr, 0);
    if constexpr (NS > 1) {
        // the last of the tile's blocks to get here adds the parts, in their order whoever it is. The parts go past the
        // caches that other XCDs do not see (agent-scope stores and loads), written before the count (the wait).
        float *ws = a.ws + int64_t(tile) * NS * kTailC * 16 + threadIdx.x;
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e)
                __hip_atomic_store(ws + part * kTailC * 16 + (4 * j + e) * 512, acc[j][e], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        int *last = reinterpret_cast<int *>(red);  // the first norm's moments are read
        if (threadIdx.x == 0) *last = __hip_atomic_fetch_add(a.count + tile, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == NS - 1;
        __syncthreads();
        if (!*last) {
            raise_status(a.status, bad, kStatusF16Range);
            return;
        }
        if (threadIdx.x == 0) __hip_atomic_store(a.count + tile, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // for the next launch
        float pv[NS][8];
#pragma unroll
        for (int k = 0; k < NS; ++k)
#pragma unroll
            for (int e = 0; e < 8; ++e)
                pv[k][e] = __hip_atomic_load(ws + k * kTailC * 16 + e * 512, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                acc[j][e] = pv[0][4 * j + e];
#pragma unroll
                for (int k = 1; k < NS; ++k) acc[j][e] += pv[k][4 * j + e];
            }
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        x[j] += acc[j] + (a.b2 ? bias[j] : zero);
        if (rin) *reinterpret_cast<f32x4v *>(a.x + int64_t(row) * kTailC + c0 + 16 * j) = x[j];
    }
    if (a.nw) {
        norm(red + kTailRed, lw, lb, n);
        if (rin) {
            uint8_t *o = reinterpret_cast<uint8_t *>(a.out16) + int64_t(tile) * kTailC * 64;
#pragma unroll
            for (int j = 0; j < 2; ++j) put(o, c0 + 16 * j, n[j]);
        }
    }
    raise_status(a.status, bad, kStatusF16Range);
}

}  // namespace vh
