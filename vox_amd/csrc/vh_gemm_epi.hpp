// vh_gemm_epi.hpp — GEMM epilogues for accumulator tiles whose lanes hold four consecutive columns of one row, and the
// split-K reduce that applies them.
#pragma once
#include "vh_gemm.hpp"
#include "vh_launch.hpp"

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

// Four f32 values as f16 halves (split_f16x2).
VH_DEV void split4(const f32x4v &x, uint2 &hi, uint2 &lo) {
    split_f16x2(x[0], x[1], hi.x, lo.x);
    split_f16x2(x[2], x[3], hi.y, lo.y);
}
// The range check of the split, two instructions a value: |x| is finite and >= 65520 exactly when twice its magnitude
// bits less those of 65520, unsigned, is below the distance to infinity. ovf4 keeps the smallest such difference seen.
constexpr uint32_t kOvfBase = 0x477FF000u << 1, kOvfSpan = (0x7F800000u << 1) - (0x477FF000u << 1);
VH_DEV uint32_t ovf4(const f32x4v &x, uint32_t mn) {
#pragma unroll
    for (int e = 0; e < 4; ++e) mn = min(mn, (__float_as_uint(x[e]) << 1) - kOvfBase);
    return mn;
}
// Four epilogue values as f16 halves (element e of hi and lo in half e of the words); true when one is beyond the f16
// range. The asm split takes each value as the f32 it is: left to the compiler, the conversion to hi can fold into the
// arithmetic before it (one rounding) in one place and not in the other, and lo then misses hi by an ulp (measured in the
// GELU epilogue: 1.8e-6 relative against 4e-8).
VH_DEV bool split_f16x4(const f32x4v &r, uint2 &hi, uint2 &lo) {
    split4(r, hi, lo);
    return ovf4(r, 0xFFFFFFFFu) < kOvfSpan;
}

VH_DEV bool aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

// The elementwise epilogues: v = c + bias, y the row's value, p0 / p1 the gate or the Snake parameters; EPI_ACC_SNAKE's
// second result in o2[e].
template <int EPI>
VH_DEV float epi_value(float v, float y, float p0, float p1, f32x4v &o2, int e) {
    if (EPI == EPI_ACC) return y + v;
    if (EPI == EPI_GATED_ACC) return fmaf(p0, v, y);
    if (EPI == EPI_GELU) return gelu_tanh_f(v);
    if (EPI == EPI_GELU_ERF) return gelu_erf_f(v);
    if (EPI == EPI_MISH) return mish_f(v);
    if (EPI == EPI_MISH_ACC) return y + mish_f(v);
    if (EPI == EPI_SNAKE) {
        const float sn = sinf(v * p0);
        return v + p1 * sn * sn;
    }
    if (EPI == EPI_ACC_SNAKE) {
        const float u = y + v, sn = sinf(u * p0);
        o2[e] = u + p1 * sn * sn;
        return u;
    }
    return v;
}
// The outputs of the activation epilogues of row `row`, columns c0 .. c0 + 3 (row and c0 inside): GELU_H16 (n a multiple of
// 32) and SWIGLU_H16 (n of 64) into f16 planes of ldy columns, SWIGLU as f32 rows.
template <int EPI>
VH_DEV void halves_store(f32x4v c, const GemmArgs &g, int row, int c0, bool &bad) {
    if (EPI == EPI_SWIGLU) {
#pragma unroll
        for (int p = 0; p < 2; ++p)
            if (c0 + 2 * p < g.n) g.y[int64_t(row) * g.ldy + c0 / 2 + p] = silu(c[2 * p]) * c[2 * p + 1];
    } else if (EPI == EPI_SWIGLU_H16) {
        uint32_t hi, lo;
        const float u0 = silu(c[0]) * c[1], u1 = silu(c[2]) * c[3];
        split_f16x2(u0, u1, hi, lo);
        bad |= ovf4(f32x4v{u0, u1, 0.f, 0.f}, 0xFFFFFFFFu) < kOvfSpan;
        _Float16 *o = g.h16 + plane_off(row, c0 / 2, int(g.ldy));
        *reinterpret_cast<uint32_t *>(o) = hi;
        *reinterpret_cast<uint32_t *>(o + kPlaneLo) = lo;
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) c[e] = g.gelu_erf ? gelu_erf_f(c[e]) : gelu_tanh_f(c[e]);
        uint2 hi, lo;
        bad |= split_f16x4(c, hi, lo);
        _Float16 *o = g.h16 + plane_off(row, c0, int(g.ldy));
        *reinterpret_cast<uint2 *>(o) = hi;
        *reinterpret_cast<uint2 *>(o + kPlaneLo) = lo;
    }
}
// EPI_ROPE_H16's store of columns c0 .. c0 + 3 (already rotated) in qkv_off's layout; for v four lanes of a quad exchange so
// that each holds four keys of one dimension (every lane of the wave takes part).
VH_DEV void rope_h16_store(const f32x4v &c, const GemmArgs &g, int row, int c0, int lane, bool &bad) {
    const bool rin = row < g.m && c0 < g.n;
    const int inner = g.rope_cols / 2, heads = inner / kQkvHead, B = g.m / g.seq, b = row / g.seq, n = row - b * g.seq;
    uint2 hi, lo;
    const bool ovf = split_f16x4(c, hi, lo);
    bad |= rin && ovf;
    auto put = [&](int64_t idx, const uint2 &h, const uint2 &l) {
        *reinterpret_cast<uint2 *>(g.h16 + idx) = h;
        *reinterpret_cast<uint2 *>(g.h16 + idx + kPlaneLo) = l;
    };
    if (c0 < g.rope_cols) {
        const int sec = c0 >= inner, cq = c0 - sec * inner;
        if (rin) put(qkv_off(sec, b, cq / kQkvHead, n, cq % kQkvHead, B, heads, g.seq_pad), hi, lo);
        return;
    }
    const int cv = c0 - g.rope_cols;
    // element e: hi in the low half, lo in the high half
    uint32_t x[4] = {(hi.x & 0xFFFFu) | lo.x << 16, hi.x >> 16 | (lo.x & 0xFFFF0000u), (hi.y & 0xFFFFu) | lo.y << 16,
                     hi.y >> 16 | (lo.y & 0xFFFF0000u)};
    if (g.seq % 4 == 0) {
        quad_transpose(x, lane);
        if (rin) {
            const uint2 h = {(x[0] & 0xFFFFu) | (x[1] << 16), (x[2] & 0xFFFFu) | (x[3] << 16)};
            const uint2 l = {(x[0] >> 16) | (x[1] & 0xFFFF0000u), (x[2] >> 16) | (x[3] & 0xFFFF0000u)};
            put(qkv_off(2, b, cv / kQkvHead, n - (lane & 3), cv % kQkvHead + (lane & 3), B, heads, g.seq_pad), h, l);
        }
    } else if (rin) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int64_t idx = qkv_off(2, b, cv / kQkvHead, n, cv % kQkvHead + e, B, heads, g.seq_pad);
            g.h16[idx] = __builtin_bit_cast(_Float16, uint16_t(x[e]));
            g.h16[idx + kPlaneLo] = __builtin_bit_cast(_Float16, uint16_t(x[e] >> 16));
        }
    }
}

// Epilogue of one 16 x 16 tile of a product taken with W as the MFMA's A operand and the activations as its B: the lane
// then holds four consecutive columns C[row][c0 .. c0 + 3] in c (row = lane % 16, c0 = 4 (lane / 16) of the tile), so a
// RoPE or SwiGLU pair is in one lane and a store is 16 bytes of a row (8 of an f16 plane) instead of four 4-byte (2-byte)
// stores to four rows. The sums and the elementwise formulas are gemm_epilogue's. vec (epi_vec): rows and parameters may
// be accessed 16 bytes at a time where the four columns exist. All lanes of a wave call it (the exchange of v).
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
    if constexpr (EPI == EPI_GELU_H16 || EPI == EPI_SWIGLU_H16 || EPI == EPI_SWIGLU) {
        if (rin && c0 < g.n) halves_store<EPI>(c, g, row, c0, bad);
        return;
    }
    if constexpr (EPI == EPI_ROPE_H16) {
        if (c0 < g.rope_cols && g.rope && rin) {
            const int n = row % g.seq, inner = g.rope_cols / 2, rhd = g.rope_hd ? g.rope_hd : g.hd;
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
        rope_h16_store(c, g, row, c0, lane, bad);
        return;
    }
    if (!rin) return;
    const int64_t idx = int64_t(row) * g.ldy + c0;
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
    float y[4] = {0.f, 0.f, 0.f, 0.f}, p0[4] = {0.f, 0.f, 0.f, 0.f}, p1[4] = {0.f, 0.f, 0.f, 0.f};
    if (kAcc) at(g.y + idx, y);
    if (EPI == EPI_GATED_ACC) at(g.gate + c0, p0);
    if (EPI == EPI_SNAKE || EPI == EPI_ACC_SNAKE) { at(g.snake_a + c0, p0); at(g.snake_ib + c0, p1); }
    f32x4v o, o2;
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = epi_value<EPI>(c[e], y[e], p0[e], p1[e], o2, e);
    if (full) {
        *reinterpret_cast<f32x4v *>(g.y + idx) = o;
        if constexpr (EPI == EPI_ACC_SNAKE) *reinterpret_cast<f32x4v *>(g.snake_y + idx) = o2;
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (c0 + e < g.n) {
                g.y[idx + e] = o[e];
                if constexpr (EPI == EPI_ACC_SNAKE) g.snake_y[idx + e] = o2[e];
            }
    }
}

// Whether the rows and parameter vectors of this launch are aligned for epi_tile's 16-byte accesses.
template <int EPI>
VH_DEV bool epi_vec(const GemmArgs &g) {
    if (EPI == EPI_GELU_H16) return aligned16(g.bias);
    return g.ldy % 4 == 0 && aligned16(g.y) && aligned16(g.bias) && aligned16(g.gate) && aligned16(g.snake_a) && aligned16(g.snake_ib) &&
           aligned16(g.snake_y);
}

// The epilogue of a wave's TM x TN tiles with its operands (bias, gate, Snake parameters, the rows it adds to, the rotation
// pairs) loaded before the K loop, where nothing waits for them: read tile by tile after it, each tile's behind the store of
// the one before, they are a chain of round trips (2000 x 1024, K 1024 with the gated add in the DiT step: 27 us, with a
// plain store 18). load() and finish() take the wave's first row and column; the fast form needs columns in fours and 16-byte alignment (epi_vec),
// otherwise finish() runs epi_tile.
template <int EPI, int TM, int TN>
struct EpiOps {
    static constexpr bool kAcc = EPI == EPI_ACC || EPI == EPI_GATED_ACC || EPI == EPI_MISH_ACC || EPI == EPI_ACC_SNAKE;
    static constexpr bool kRope = EPI == EPI_ROPE_H16;
    static constexpr bool kP0 = EPI == EPI_GATED_ACC || EPI == EPI_SNAKE || EPI == EPI_ACC_SNAKE;
    static constexpr bool kP1 = EPI == EPI_SNAKE || EPI == EPI_ACC_SNAKE;
    f32x4v bias[TN], p0[kP0 ? TN : 1], p1[kP1 ? TN : 1], y[kAcc ? TM : 1][kAcc ? TN : 1], cs[kRope ? TM : 1][kRope ? TN : 1];
    bool fast;

    VH_DEV void load(const GemmArgs &g, int rbase, int cbase) {
        fast = epi_vec<EPI>(g) && g.n % 4 == 0;
        const int rhd = g.rope_hd ? g.rope_hd : g.hd;  // the table's floats per row
        if (kRope) fast = fast && g.hd % 4 == 0 && (!g.rope || (rhd % 4 == 0 && aligned16(g.rope)));
        if (!fast) return;
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            const int c = min(cbase + 16 * j, g.n - 4);
            bias[j] = f32x4v{0.f, 0.f, 0.f, 0.f};
            if (g.bias) bias[j] = *reinterpret_cast<const f32x4v *>(g.bias + c);
            if constexpr (EPI == EPI_GATED_ACC) p0[j] = *reinterpret_cast<const f32x4v *>(g.gate + c);
            if constexpr (kP1) {
                p0[j] = *reinterpret_cast<const f32x4v *>(g.snake_a + c);
                p1[j] = *reinterpret_cast<const f32x4v *>(g.snake_ib + c);
            }
        }
        if constexpr (kAcc) {
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j)
                    y[i][j] = *reinterpret_cast<const f32x4v *>(g.y + int64_t(min(rbase + 16 * i, g.m - 1)) * g.ldy + min(cbase + 16 * j, g.n - 4));
        }
        if constexpr (kRope) {
            if (g.rope) {
#pragma unroll
                for (int i = 0; i < TM; ++i) {
                    const int n = min(rbase + 16 * i, g.m - 1) % g.seq;
#pragma unroll
                    for (int j = 0; j < TN; ++j)
                        cs[i][j] = *reinterpret_cast<const f32x4v *>(g.rope + int64_t(n) * rhd + min((cbase + 16 * j) % g.hd, rhd - 4));
                }
            }
        }
    }

    template <class Acc>
    VH_DEV void finish(const Acc &acc, const GemmArgs &g, int rbase, int cbase, int lane, bool &bad) const {
        if (!fast) {
            const bool vec = epi_vec<EPI>(g);
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j) epi_tile<EPI>(acc[i][j], g, rbase + 16 * i, cbase + 16 * j, vec, lane, bad);
            return;
        }
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            const int c0 = cbase + 16 * j;
            bool rot = false;
            if constexpr (kRope) {
                const int rhd = g.rope_hd ? g.rope_hd : g.hd;  // the padding dims (d >= rhd) stay zero
                rot = g.rope && c0 < g.rope_cols && c0 % g.hd < rhd && (g.rope_heads <= 0 || c0 % (g.rope_cols / 2) / g.hd < g.rope_heads);
            }
#pragma unroll
            for (int i = 0; i < TM; ++i) {
                const int row = rbase + 16 * i;
                const bool in = row < g.m && c0 < g.n;
                f32x4v c = acc[i][j] + bias[j];
                if constexpr (kRope) {
                    const f32x4v t = cs[i][j];
                    if (rot) c = f32x4v{c[0] * t[0] - c[1] * t[1], c[1] * t[0] + c[0] * t[1], c[2] * t[2] - c[3] * t[3], c[3] * t[2] + c[2] * t[3]};
                }
                if constexpr (EPI == EPI_ROPE_H16) {
                    rope_h16_store(c, g, row, c0, lane, bad);
                } else if constexpr (EPI == EPI_GELU_H16 || EPI == EPI_SWIGLU_H16 || EPI == EPI_SWIGLU) {
                    if (in) halves_store<EPI>(c, g, row, c0, bad);
                } else {
                    f32x4v o2;
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const float y0 = kAcc ? y[kAcc ? i : 0][kAcc ? j : 0][e] : 0.f, a0 = kP0 ? p0[kP0 ? j : 0][e] : 0.f,
                                    a1 = kP1 ? p1[kP1 ? j : 0][e] : 0.f;
                        c[e] = epi_value<EPI>(c[e], y0, a0, a1, o2, e);
                    }
                    if (in) {
                        const int64_t idx = int64_t(row) * g.ldy + c0;
                        *reinterpret_cast<f32x4v *>(g.y + idx) = c;
                        if constexpr (EPI == EPI_ACC_SNAKE) *reinterpret_cast<f32x4v *>(g.snake_y + idx) = o2;
                    }
                }
            }
        }
    }
};

// Split K: a tile's four columns as partial sums into slice ws ([m][n]), no bias or epilogue.
VH_DEV void store_partial(const f32x4v &v, float *ws, const GemmArgs &g, int row, int c0) {
    if (row >= g.m) return;
    float *p = ws + int64_t(row) * g.n + c0;
    if (g.n % 4 == 0) {
        if (c0 < g.n) *reinterpret_cast<f32x4v *>(p) = v;
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (c0 + e < g.n) p[e] = v[e];
    }
}

// The split-K partial slices ws[z][m][n] added in z order, then bias and the epilogue: one thread per U columns of a row, eight
// slices' loads in flight at once (past `splits` they read slice 0 and are left out). U 4 where n is a multiple of 4; else one
// column (a gate | up pair of SWIGLU), since four columns then are sixteen 4-byte loads and a chain of scalar stores a thread
// (9 x 1026, K 3072 in 24 slices, product and reduce: 16.5 us with four columns, 11.1 with one). Bound by its launch and one
// round trip of loads. grid ceil(m ceil(n / U) / 256).
template <int EPI, int U>
__global__ __launch_bounds__(256) void k_gemm_splitk_reduce(GemmArgs g, int32_t splits) {
    static_assert(U == 4 || U == (EPI == EPI_SWIGLU ? 2 : 1), "four columns, or the epilogue's least");
    const int nq = (g.n + U - 1) / U;
    const int64_t t = int64_t(blockIdx.x) * 256 + threadIdx.x;
    if (t >= int64_t(g.m) * nq) return;
    const int row = int(t / nq), c0 = int(t % nq) * U;
    const int64_t slice = int64_t(g.m) * g.n;
    const float *p = g.ws + int64_t(row) * g.n + c0;
    f32x4v v = {0.f, 0.f, 0.f, 0.f};
    for (int z0 = 0; z0 < splits; z0 += 8) {
        f32x4v x[8];
#pragma unroll
        for (int z = 0; z < 8; ++z) {
            const float *q = p + (z0 + z < splits ? z0 + z : 0) * slice;
            if constexpr (U == 4) {
                x[z] = *reinterpret_cast<const f32x4v *>(q);
            } else {
                x[z] = f32x4v{q[0], U == 2 ? q[U - 1] : 0.f, 0.f, 0.f};
            }
        }
#pragma unroll
        for (int z = 0; z < 8; ++z)
            if (z0 + z < splits) v += x[z];
    }
    if constexpr (U == 4) {
        bool bad = false;
        epi_tile<EPI>(v, g, row, c0, epi_vec<EPI>(g), 0, bad);
    } else {
#pragma unroll
        for (int e = 0; e < U; ++e) v[e] += g.bias ? g.bias[c0 + e] : 0.f;
        if constexpr (EPI == EPI_SWIGLU) {
            g.y[int64_t(row) * g.ldy + c0 / 2] = silu(v[0]) * v[1];
        } else {
            constexpr bool kAcc = EPI == EPI_ACC || EPI == EPI_GATED_ACC || EPI == EPI_ACC_SNAKE, kSnake = EPI == EPI_SNAKE || EPI == EPI_ACC_SNAKE;
            const int64_t idx = int64_t(row) * g.ldy + c0;
            f32x4v o2 = {0.f, 0.f, 0.f, 0.f};
            g.y[idx] = epi_value<EPI>(v[0], kAcc ? g.y[idx] : 0.f, EPI == EPI_GATED_ACC ? g.gate[c0] : kSnake ? g.snake_a[c0] : 0.f,
                                      kSnake ? g.snake_ib[c0] : 0.f, o2, 0);
            if constexpr (EPI == EPI_ACC_SNAKE) g.snake_y[idx] = o2[0];
        }
    }
}
template <int EPI>
hipError_t launch_splitk_reduce(const GemmArgs &g, int splits, hipStream_t s) {
    constexpr int U = EPI == EPI_SWIGLU ? 2 : 1;
    const int u = g.n % 4 == 0 ? 4 : U;
    const dim3 grid(unsigned((int64_t(g.m) * ((g.n + u - 1) / u) + 255) / 256));
    if (u == 4) return launch(k_gemm_splitk_reduce<EPI, 4>, grid, dim3(256), 0, s, g, int32_t(splits));
    return launch(k_gemm_splitk_reduce<EPI, U>, grid, dim3(256), 0, s, g, int32_t(splits));
}
template <int EPI>
constexpr bool kReduceEpi = EPI == EPI_STORE || EPI == EPI_ACC || EPI == EPI_GATED_ACC || EPI == EPI_SWIGLU || EPI == EPI_SNAKE ||
                            EPI == EPI_GELU_ERF || EPI == EPI_ACC_SNAKE;

}  // namespace vh
