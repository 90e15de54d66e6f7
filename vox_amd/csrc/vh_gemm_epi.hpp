// vh_gemm_epi.hpp — GEMM epilogues for accumulator tiles whose lanes hold four consecutive columns of one row, and the
// split-K reduce that applies them.
#pragma once
#include "vh_gemm.hpp"

namespace vh {

// The 4 x 4 words of a quad of lanes transposed: lane b of each quad gives x[j] to lane j and gets lane j's x[b].
VH_DEV void quad_transpose(uint32_t (&x)[4], int lane) {
    const bool b0 = lane & 1, b1 = lane & 2;
#pragma unroll
    for (int p = 0; p < 4; p += 2) {
        const int r = dpp<kDppXor1>(int(b0 ? x[p] : x[p + 1]));
        if (b0) x[p] = uint32_t(r); else x[p + 1] = uint32_t(r);
    }
#pragma unroll
    for (int p = 0; p < 2; ++p) {
        const int r = dpp<kDppXor2>(int(b1 ? x[p] : x[p + 2]));
        if (b1) x[p] = uint32_t(r); else x[p + 2] = uint32_t(r);
    }
}

VH_DEV bool split_f16x4(const f32x4v &r, f16x4v &hi, f16x4v &lo) {
    bool bad = false;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        _Float16 h, l;
        bad |= split_f16(r[e], h, l);
        hi[e] = h;
        lo[e] = l;
    }
    return bad;
}

VH_DEV bool aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

// Epilogue of one 16 x 16 tile of a product taken with W as the MFMA's A operand and the activations as its B: the lane
// then holds four consecutive columns C[row][c0 .. c0 + 3] in c (row = lane % 16, c0 = 4 (lane / 16) of the tile), so a
// RoPE or SwiGLU pair is in one lane and a store is 16 bytes of a row (8 of an f16 plane) instead of four 4-byte (2-byte)
// stores to four rows. The sums and the elementwise formulas are gemm_epilogue's. vec (epi_vec): rows and parameters may
// be accessed 16 bytes at a time where the four columns exist. All lanes of a wave call it (the v^T exchange).
template <int EPI>
VH_DEV void epi_tile(f32x4v c, const GemmArgs &g, int row, int c0, bool vec, int lane, bool &bad) {
    const bool rin = row < g.m, full = vec && c0 + 3 < g.n;
    if (g.bias) {
        if (full) {
            c += *reinterpret_cast<const f32x4v *>(g.bias + c0);
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) c[e] += c0 + e < g.n ? g.bias[c0 + e] : 0.f;
        }
    }
    if (EPI == EPI_SWIGLU || EPI == EPI_SWIGLU_H16) {
        if (!rin) return;
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            if (c0 + 2 * p >= g.n) continue;
            const float r = silu(c[2 * p]) * c[2 * p + 1];
            const int64_t idx = int64_t(row) * g.ldy + c0 / 2 + p;
            if (EPI == EPI_SWIGLU) {
                g.y[idx] = r;
            } else {
                _Float16 hi, lo;
                bad |= split_f16(r, hi, lo);
                g.h16[idx] = hi;
                g.h16[g.lo_off + idx] = lo;
            }
        }
        return;
    }
    if (EPI == EPI_ROPE || EPI == EPI_ROPE_H16) {
        const int b = row / g.seq, n = row - b * g.seq;
        if (c0 < g.rope_cols) {
            const int inner = g.rope_cols / 2, rhd = g.rope_hd ? g.rope_hd : g.hd;
            if (g.rope && rin) {
#pragma unroll
                for (int p = 0; p < 2; ++p) {
                    const int col = c0 + 2 * p, d = col % g.hd, head = (col % inner) / g.hd;
                    if (d < rhd && (g.rope_heads <= 0 || head < g.rope_heads)) {
                        const float *cs = g.rope + (int64_t(n) * (rhd / 2) + d / 2) * 2;
                        const float cc = cs[0], sn = cs[1], x0 = c[2 * p], x1 = c[2 * p + 1];
                        c[2 * p] = x0 * cc - x1 * sn;
                        c[2 * p + 1] = x1 * cc + x0 * sn;
                    }
                }
            }
            if (EPI == EPI_ROPE_H16) {
                f16x4v hi, lo;
                if (rin) {
                    bad |= split_f16x4(c, hi, lo);
                    const int64_t idx = int64_t(row) * g.rope_cols + c0;
                    *reinterpret_cast<f16x4v *>(g.h16 + idx) = hi;
                    *reinterpret_cast<f16x4v *>(g.h16 + g.lo_off + idx) = lo;
                }
                return;
            }
        } else if (EPI == EPI_ROPE_H16) {
            // v, transposed: [batch][head][d][key]; four lanes of a quad exchange so that each holds four keys of one d
            const int64_t vbase = int64_t(g.m) * g.rope_cols;
            const int vh = g.rope_cols / 2 / g.hd;
            f16x4v hi, lo;
            const bool ovf = split_f16x4(c, hi, lo);
            bad |= rin && c0 < g.n && ovf;
            if (g.seq % 4 == 0) {
                uint32_t x[4];
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    x[e] = uint32_t(__builtin_bit_cast(uint16_t, _Float16(hi[e]))) |
                           uint32_t(__builtin_bit_cast(uint16_t, _Float16(lo[e]))) << 16;
                quad_transpose(x, lane);
                const int col = c0 + (lane & 3), cv = col - g.rope_cols, k0 = n - (lane & 3);
                if (rin && col < g.n) {
                    const int64_t idx = vbase + ((int64_t(b) * vh + cv / g.hd) * g.hd + cv % g.hd) * g.ldvt + k0;
                    uint2 h, l;
                    h.x = (x[0] & 0xFFFFu) | (x[1] << 16); h.y = (x[2] & 0xFFFFu) | (x[3] << 16);
                    l.x = (x[0] >> 16) | (x[1] & 0xFFFF0000u); l.y = (x[2] >> 16) | (x[3] & 0xFFFF0000u);
                    *reinterpret_cast<uint2 *>(g.h16 + idx) = h;
                    *reinterpret_cast<uint2 *>(g.h16 + g.lo_off + idx) = l;
                }
            } else if (rin) {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int cv = c0 + e - g.rope_cols;
                    if (c0 + e < g.n) {
                        const int64_t idx = vbase + ((int64_t(b) * vh + cv / g.hd) * g.hd + cv % g.hd) * g.ldvt + n;
                        g.h16[idx] = hi[e];
                        g.h16[g.lo_off + idx] = lo[e];
                    }
                }
            }
            return;
        }
    }
    if (!rin) return;
    const int64_t idx = int64_t(row) * g.ldy + c0;
    if (EPI == EPI_GELU_H16) {
#pragma unroll
        for (int e = 0; e < 4; ++e) c[e] = g.gelu_erf ? gelu_erf_f(c[e]) : gelu_tanh_f(c[e]);
        f16x4v hi, lo;
        if (full) {
            bad |= split_f16x4(c, hi, lo);
            *reinterpret_cast<f16x4v *>(g.h16 + idx) = hi;
            *reinterpret_cast<f16x4v *>(g.h16 + g.lo_off + idx) = lo;
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (c0 + e < g.n) {
                    _Float16 h, l;
                    bad |= split_f16(c[e], h, l);
                    g.h16[idx + e] = h;
                    g.h16[g.lo_off + idx + e] = l;
                }
        }
        return;
    }
    auto at = [&](const float *p, float (&v)[4]) {
        if (full) {
            const f32x4v t = *reinterpret_cast<const f32x4v *>(p);
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = t[e];
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = c0 + e < g.n ? p[e] : 0.f;
        }
    };
    constexpr bool kAcc = EPI == EPI_ACC || EPI == EPI_GATED_ACC || EPI == EPI_MISH_ACC || EPI == EPI_ACC_SNAKE;
    float y[4] = {0.f, 0.f, 0.f, 0.f}, p0[4], p1[4];
    if (kAcc) at(g.y + idx, y);
    if (EPI == EPI_GATED_ACC) at(g.gate + c0, p0);
    if (EPI == EPI_SNAKE || EPI == EPI_ACC_SNAKE) { at(g.snake_a + c0, p0); at(g.snake_ib + c0, p1); }
    f32x4v o, o2;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        float v = c[e];
        if (EPI == EPI_ACC) v = y[e] + v;
        else if (EPI == EPI_GATED_ACC) v = fmaf(p0[e], v, y[e]);
        else if (EPI == EPI_GELU) v = gelu_tanh_f(v);
        else if (EPI == EPI_GELU_ERF) v = gelu_erf_f(v);
        else if (EPI == EPI_MISH) v = mish_f(v);
        else if (EPI == EPI_MISH_ACC) v = y[e] + mish_f(v);
        else if (EPI == EPI_SNAKE) {
            const float sn = sinf(v * p0[e]);
            v = v + p1[e] * sn * sn;
        } else if (EPI == EPI_ACC_SNAKE) {
            v = y[e] + v;
            const float sn = sinf(v * p0[e]);
            o2[e] = v + p1[e] * sn * sn;
        }
        o[e] = v;
    }
    if (full) {
        *reinterpret_cast<f32x4v *>(g.y + idx) = o;
        if (EPI == EPI_ACC_SNAKE) *reinterpret_cast<f32x4v *>(g.snake_y + idx) = o2;
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (c0 + e < g.n) {
                g.y[idx + e] = o[e];
                if (EPI == EPI_ACC_SNAKE) g.snake_y[idx + e] = o2[e];
            }
    }
}

// Whether the rows and parameter vectors of this launch are aligned for epi_tile's 16-byte accesses.
template <int EPI>
VH_DEV bool epi_vec(const GemmArgs &g) {
    if (EPI == EPI_GELU_H16) return g.ldy % 4 == 0 && g.lo_off % 4 == 0 && (reinterpret_cast<uintptr_t>(g.h16) & 7) == 0 && aligned16(g.bias);
    return g.ldy % 4 == 0 && aligned16(g.y) && aligned16(g.bias) && aligned16(g.gate) && aligned16(g.snake_a) && aligned16(g.snake_ib) &&
           aligned16(g.snake_y);
}

// The split-K partial slices ws[z][m][n] added in z order, then bias and the epilogue: one thread per four columns of a
// row. Eight slices' loads are in flight at once (past `splits` they read slice 0 and are left out). Bound by its launch
// and one round trip of loads. grid ceil(m ceil(n / 4) / 256).
template <int EPI>
__global__ __launch_bounds__(256) void k_gemm_splitk_reduce(GemmArgs g, int32_t splits) {
    const int nq = (g.n + 3) / 4;
    const int64_t t = int64_t(blockIdx.x) * 256 + threadIdx.x;
    if (t >= int64_t(g.m) * nq) return;
    const int row = int(t / nq), c0 = int(t % nq) * 4;
    const int64_t slice = int64_t(g.m) * g.n;
    const float *p = g.ws + int64_t(row) * g.n + c0;
    f32x4v v = {0.f, 0.f, 0.f, 0.f};
    for (int z0 = 0; z0 < splits; z0 += 8) {
        f32x4v x[8];
        if (g.n % 4 == 0) {
#pragma unroll
            for (int z = 0; z < 8; ++z) x[z] = *reinterpret_cast<const f32x4v *>(p + (z0 + z < splits ? z0 + z : 0) * slice);
        } else {
#pragma unroll
            for (int z = 0; z < 8; ++z)
#pragma unroll
                for (int e = 0; e < 4; ++e) x[z][e] = c0 + e < g.n ? p[(z0 + z < splits ? z0 + z : 0) * slice + e] : 0.f;
        }
#pragma unroll
        for (int z = 0; z < 8; ++z)
            if (z0 + z < splits) v += x[z];
    }
    bool bad = false;
    epi_tile<EPI>(v, g, row, c0, epi_vec<EPI>(g), 0, bad);
}
template <int EPI>
constexpr bool kReduceEpi = EPI == EPI_STORE || EPI == EPI_ACC || EPI == EPI_GATED_ACC || EPI == EPI_SWIGLU || EPI == EPI_SNAKE ||
                            EPI == EPI_GELU_ERF || EPI == EPI_ACC_SNAKE;

}  // namespace vh
