// vh_codec.hpp — Qwen3-TTS codec decoder kernels besides the GEMMs (qwen3.cpp:80-161, :366-481; the Vulkan shaders
// snake / hist / dwconv / ola / ringput / attnw of gpu_codec.cpp): streaming histories, the causal depthwise conv,
// the transposed conv's overlap-add with its tail (and the Snake of its output), the pre-transformer's RoPE + ring
// append and sliding-window attention over the ring, layer-scaled residual adds and the final clamp. The other Snakes
// are GEMM epilogues (EPI_SNAKE, EPI_ACC_SNAKE). Activations are time-major f32 rows.
#pragma once
#include "vh_common.hpp"
#include "vh_types.hpp"

namespace vh {

// A streaming history after a call of T rows: the last ctx rows of [old (ctx rows); x (T rows, stride ldx)] into
// dst (another buffer than old). qwen3.cpp:120, :136.
__global__ __launch_bounds__(256) void k_hist_shift(float *__restrict__ dst, const float *__restrict__ old,
                                                    const float *__restrict__ x, int64_t ldx, int32_t T, int32_t ctx,
                                                    int32_t C) {
    const int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x;
    if (i >= int64_t(ctx) * C) return;
    const int j = int(i / C), c = int(i % C), r = j + T;  // row r of the extended sequence
    dst[i] = r < ctx ? old[int64_t(r) * C + c] : x[int64_t(r - ctx) * ldx + c];
}

// dwconv_stream (qwen3.cpp:123-137): y[t][c] = b[c] + sum_k w[c][k] ext[t + k][c] over ext = [hist (K - 1 rows); x],
// taps in order. One thread per output.
// hist_next (may be null): also written, the next call's history (k_hist_shift's rows) by threads i < (K - 1) C.
__global__ __launch_bounds__(256) void k_dwconv_causal(const float *__restrict__ x, const float *__restrict__ hist,
                                                       const float *__restrict__ w, const float *__restrict__ b,
                                                       float *__restrict__ y, int32_t T, int32_t C, int32_t K,
                                                       float *__restrict__ hist_next) {
    const int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x;
    if (hist_next && i < int64_t(K - 1) * C) {
        const int j = int(i / C), c = int(i % C), r = j + T;  // row r of [hist; x]
        hist_next[i] = r < K - 1 ? hist[int64_t(r) * C + c] : x[int64_t(r - (K - 1)) * C + c];
    }
    if (i >= int64_t(T) * C) return;
    const int t = int(i / C), c = int(i % C), ctx = K - 1;
    float acc = b[c];
    for (int k = 0; k < K; ++k) {
        const int r = t + k;
        const float v = r < ctx ? hist[int64_t(r) * C + c] : x[int64_t(r - ctx) * C + c];
        acc += w[int64_t(c) * K + k] * v;
    }
    y[i] = acc;
}

// trans_stream's overlap-add (qwen3.cpp:139-161) from the GEMM output tmp [T][K co] (row k co + o of frame t): output
// row p (of T s + K - s) takes frame p / s at tap p % s and frame p / s - 1 at tap p % s + s (K <= 2 s), plus the old
// tail's row p; rows below T s go to y with the bias, the rest to the new tail (another buffer than the old one).
// sy, when set: Snake(y) (per-channel sa, sib) of those rows too, the first residual unit's input.
__global__ __launch_bounds__(256) void k_ola(const float *__restrict__ tmp, const float *__restrict__ tail_old,
                                             float *__restrict__ tail_new, const float *__restrict__ bias,
                                             float *__restrict__ y, int32_t T, int32_t s, int32_t K, int32_t co,
                                             float *__restrict__ sy, const float *__restrict__ sa, const float *__restrict__ sib) {
    const int tr = K - s;
    const int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x;
    if (i >= (int64_t(T) * s + tr) * co) return;
    const int64_t p = i / co;
    const int o = int(i % co);
    const int64_t t = p / s;
    const int k = int(p - t * s);
    float v = p < tr ? tail_old[p * co + o] : 0.f;
    if (t < T && k < K) v += tmp[(t * K + k) * co + o];
    if (t >= 1 && k + s < K) v += tmp[((t - 1) * K + k + s) * co + o];
    if (p < int64_t(T) * s) {
        const float yv = v + bias[o];
        y[p * co + o] = yv;
        if (sy) {
            const float sn = sinf(yv * sa[o]);
            sy[p * co + o] = yv + sib[o] * sn * sn;
        }
    } else {
        tail_new[(p - int64_t(T) * s) * co + o] = v;
    }
}

// nn::ConvT's overlap-add with padding (nn.cpp:217-245) in gather form, from the GEMM output z [T][K co] (row k co + o
// of input frame t): output row r of To takes z[t][r + pad - t s] for every frame t with 0 <= r + pad - t s < K, summed
// in increasing t (the order the reference adds them in), then the bias (or nothing). One thread per output element.
__global__ __launch_bounds__(256) void k_convt_gather(const float *__restrict__ z, const float *__restrict__ bias,
                                                      float *__restrict__ y, int32_t T, int32_t To, int32_t s, int32_t K,
                                                      int32_t pad, int32_t co) {
    const int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x;
    if (i >= int64_t(To) * co) return;
    const int64_t r = i / co;
    const int o = int(i - r * co);
    const int64_t q = r + pad;
    const int64_t lo_num = q - K + 1;
    const int64_t t_lo = lo_num <= 0 ? 0 : (lo_num + s - 1) / s;
    const int64_t t_hi = min(int64_t(T) - 1, q / s);
    float v = 0.f;
    for (int64_t t = t_lo; t <= t_hi; ++t) v += z[(t * K + (q - t * s)) * co + o];
    y[i] = bias ? v + bias[o] : v;
}

// The pre-transformer's attention of one call, from the q | k | v rows [F][ld] of its frames: the q / k rotation (rope_apply,
// kernels.cpp:740-757: pairs (d, d + hd / 2)) with the host table rope [F][hd / 2][2] of positions pos0 + i; the append of row
// i's key and value to ring slot (pos0 + i) % R of the layer's f32 ring [R][kv_heads hd]; and the sliding-window attention of
// row i (kernels.cpp:809-828 with the window of :814): keys of positions (p - W, p], scores scale (q . k), softmax, sum p v. The
// call's own keys are rotated again by each block that needs them, from the rows, so no block waits for another's append,
// and the appended slots are in no row's window (R >= W + F - 1). The first position pos0 is read from device memory (*pos), so a
// captured call replays at any position. W <= 1024, hd <= 128, hd % 4 == 0, F <= 16.
// One block per (row, head): a thread takes a key for the scores, then a dimension and every (256 / DT)th key for the output;
// the ring's keys and values are on their way before anything waits. Bound by that latency: one wave reading the values eight
// positions at a time took 6.5 us for a window of 72, after 3.8 us for the rotation and append in a launch of its own; 10.3 ->
// 6.0 us.
constexpr int kCodecRows = 16;
template <int DT>
__global__ __launch_bounds__(256) void k_codec_attn(const float *__restrict__ qkv, int32_t ld, float *ring_k, float *ring_v,
                                                    const float *__restrict__ rope, int32_t R, int32_t heads, int32_t kvh, int32_t hd,
                                                    const int64_t *__restrict__ pos, int32_t W, float scale, float *__restrict__ ao) {
    constexpr int G = 256 / DT, VC = 24;  // key groups of the output, keys of a group in flight
    __shared__ float p[1024], red[4], part[G][DT];
    __shared__ __align__(16) float q[128], kc[kCodecRows][128];
    const int i = blockIdx.x, h = blockIdx.y, tid = threadIdx.x, d = tid % DT, grp = tid / DT;
    const int qd = heads * hd, kd = kvh * hd, hk = h / (heads / kvh), off = hk * hd, half = hd / 2;
    const int64_t pos0 = *pos;
    const int64_t last = pos0 + i, first = last - W + 1 > 0 ? last - W + 1 : 0;
    const int n = int(last - first + 1), s0 = int(first % R), nring = n - 1 - i > 0 ? n - 1 - i : 0;  // keys before the call's
    const int r0 = i + 1 - (n - nring);  // the first of the call's rows in the window
    auto slot_of = [&](int j) { return s0 + j < R ? s0 + j : s0 + j - R; };
    auto value = [&](int j) {
        return j < nring ? ring_v[int64_t(slot_of(j)) * kd + off + d] : qkv[int64_t(r0 + j - nring) * ld + qd + kd + off + d];
    };
    f32x4 kr[DT / 4];  // this thread's key, if the ring's
    if (tid < nring) {
        const f32x4 *k = reinterpret_cast<const f32x4 *>(ring_k + int64_t(slot_of(tid)) * kd + off);
#pragma unroll
        for (int e = 0; e < DT / 4; ++e) kr[e] = k[min(e, hd / 4 - 1)];
    }
    float v[VC];
    if (d < hd) {
#pragma unroll
        for (int c = 0; c < VC; ++c) v[c] = grp + G * c < n ? value(grp + G * c) : 0.f;
    }
    for (int e = tid; e < (i + 2) * half; e += 256) {  // the call's keys up to row i, then q
        const int r = e / half, x = e % half;
        const bool key = r <= i;
        const float *src = key ? qkv + int64_t(r) * ld + qd + off : qkv + int64_t(i) * ld + h * hd;
        const float *cs = rope + int64_t(key ? r : i) * hd;
        const float a = src[x], b = src[x + half], c = cs[2 * x], sn = cs[2 * x + 1];
        float *o = key ? kc[r] : q;
        o[x] = a * c - b * sn;
        o[x + half] = b * c + a * sn;
    }
    __syncthreads();
    if (h % (heads / kvh) == 0 && tid < hd) {  // row i's slot, by the first query head of each kv head
        const int64_t slot = last % R;
        ring_k[slot * kd + off + tid] = kc[i][tid];
        ring_v[slot * kd + off + tid] = qkv[int64_t(i) * ld + qd + kd + off + tid];
    }
    const f32x4 *qv = reinterpret_cast<const f32x4 *>(q);
    float mx = -INFINITY;
    for (int j = tid; j < n; j += 256) {
        float dot = 0.f;
        auto term = [&](const f32x4 &a, const f32x4 &b) { dot += b[0] * a[0] + b[1] * a[1] + b[2] * a[2] + b[3] * a[3]; };
        if (j < nring && j == tid) {
#pragma unroll
            for (int e = 0; e < DT / 4; ++e)
                if (e < hd / 4) term(kr[e], qv[e]);
        } else {
            const f32x4 *k = j < nring ? reinterpret_cast<const f32x4 *>(ring_k + int64_t(slot_of(j)) * kd + off)
                                       : reinterpret_cast<const f32x4 *>(kc[r0 + j - nring]);
            for (int e = 0; e < hd / 4; ++e) term(k[e], qv[e]);
        }
        p[j] = scale * dot;
        mx = fmaxf(mx, p[j]);
    }
    mx = wave_max(mx);
    if (tid % 64 == 0) red[tid / 64] = mx;
    __syncthreads();
    mx = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    float sum = 0.f;
    for (int j = tid; j < n; j += 256) {
        p[j] = expf(p[j] - mx);
        sum += p[j];
    }
    sum = wave_sum(sum);
    __syncthreads();  // every wave has read red
    if (tid % 64 == 0) red[tid / 64] = sum;
    __syncthreads();
    const float inv = 1.0f / ((red[0] + red[1]) + (red[2] + red[3]));
    float acc = 0.f;
    if (d < hd) {
#pragma unroll
        for (int c = 0; c < VC; ++c) acc += grp + G * c < n ? p[grp + G * c] * v[c] : 0.f;
        for (int j = grp + G * VC; j < n; j += G) acc += p[j] * value(j);
    }
    part[grp][d] = acc;
    __syncthreads();
    if (tid < hd) {
        float o = part[0][tid];
#pragma unroll
        for (int g = 1; g < G; ++g) o += part[g][tid];
        ao[int64_t(i) * heads * hd + h * hd + tid] = o * inv;
    }
}

// h += s[e] t over rows of H (the layer scales of kernels.cpp:830, :838: the projection scaled, then added).
__global__ __launch_bounds__(256) void k_scale_acc(float *__restrict__ h, const float *__restrict__ t,
                                                   const float *__restrict__ s, int64_t n, int32_t H) {
    const int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x;
    if (i >= n) return;
    h[i] += t[i] * s[int(i % H)];
}

// The final clamp to [-1, 1] (qwen3.cpp:478).
__global__ __launch_bounds__(256) void k_clamp1(float *__restrict__ y, int64_t n) {
    const int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x;
    if (i >= n) return;
    y[i] = fminf(1.0f, fmaxf(-1.0f, y[i]));
}

}  // namespace vh
