// comp_emit.h — the compressor's emitted row (cuda/compressor.cu:107-339),
// shared by the per-step kernels (compressor.hip) and the prompt-chunk kernel
// (chunk.hip), which take the window's rows from different places.
#pragma once

#include "ds4hip_common.h"

#include <cmath>

namespace ds4hip {

constexpr float kNegInf = -1.0e30f;   // cuda/compressor.cu:53
constexpr float kRmsEps = 1.0e-6f;    // cuda/compressor.cu:54
constexpr int kNRot = 64;             // cuda/compressor.cu:55

struct RopeArgs {
    float theta_scale, freq_scale, ext_factor, attn_factor, corr_low, corr_high;
    int pos;
};

// cuda/rope.cu:214-250 (host) for n_rot = 64
inline RopeArgs rope_args(int il, int pos) {
    const bool compressed = il >= 2;
    RopeArgs R;
    const float base = compressed ? 160000.0f : 10000.0f;
    R.freq_scale = compressed ? 1.0f / 16.0f : 1.0f;
    R.ext_factor = compressed ? 1.0f : 0.0f;
    R.attn_factor = 1.0f;
    if (R.ext_factor != 0.0f) R.attn_factor /= 1.0f + 0.1f * logf(1.0f / R.freq_scale);
    R.corr_low = R.corr_high = 0.0f;
    if (R.ext_factor != 0.0f) {
        const float pi = 3.14159265358979323846f;
        auto corr_dim = [&](float t) {
            return (float)kNRot * logf(65536.0f / (t * 2.0f * pi)) / (2.0f * logf(base));
        };
        R.corr_low = fmaxf(0.0f, floorf(corr_dim(32.0f)));
        R.corr_high = fminf((float)(kNRot - 1), ceilf(corr_dim(1.0f)));
    }
    R.theta_scale = powf(base, -2.0f / (float)kNRot);
    R.pos = pos;
    return R;
}

// The emitted row from a window's state rows: pool, RMSNorm, tail RoPE, FP8
// round trip. Src gives the window as the state holds it: kv(row, column) and
// score(row, column), rows 0 .. 2 ratio - 1 (ratio 4) or 0 .. ratio - 1. One
// workgroup of 512 threads; thread j owns column j (< head_dim <= 512).
template <class Src>
__device__ inline void emit_row(const Src &src, const float *__restrict__ w_norm, float *__restrict__ emit_out,
                                int head_dim, int ratio, int is_attn, RopeArgs R) {
    __shared__ float pooled[512];
    __shared__ float red[8];
    const int j = threadIdx.x;
    // ---- pool (cuda/compressor.cu:107-164)
    float v = 0.0f;
    if (j < head_dim) {
        float mx = kNegInf;
        if (ratio == 4) {
            for (int r = 0; r < 4; ++r) {
                mx = fmaxf(mx, src.score(r, j));
                mx = fmaxf(mx, src.score(4 + r, head_dim + j));
            }
            if (mx > kNegInf * 0.5f) {
                float den = 0.0f, sum = 0.0f;
                for (int r = 0; r < 4; ++r) {
                    const float wp = expf(src.score(r, j) - mx);
                    const float wc = expf(src.score(4 + r, head_dim + j) - mx);
                    den += wp + wc;
                    sum += wp * src.kv(r, j);
                    sum += wc * src.kv(4 + r, head_dim + j);
                }
                v = den > 0.0f ? sum / den : 0.0f;
            }
        } else {
            // ratio 128: 32 rows at a time, so that the loads of a batch are in
            // flight together (row by row, an emit took 32 us with the state in
            // cache; now 14), and rolled: the code is fetched once per emit
#pragma unroll 1
            for (int b = 0; b < 128; b += 32) {
                float sc[32];
#pragma unroll
                for (int r = 0; r < 32; ++r) sc[r] = src.score(b + r, j);
#pragma unroll
                for (int r = 0; r < 32; ++r) mx = fmaxf(mx, sc[r]);
            }
            if (mx > kNegInf * 0.5f) {
                float den = 0.0f, sum = 0.0f;
#pragma unroll 1
                for (int b = 0; b < 128; b += 32) {
                    float sc[32], k[32];
#pragma unroll
                    for (int r = 0; r < 32; ++r) {
                        sc[r] = src.score(b + r, j);
                        k[r] = src.kv(b + r, j);
                    }
#pragma unroll
                    for (int r = 0; r < 32; ++r) {
                        const float w = expf(sc[r] - mx);
                        den += w;
                        sum += w * k[r];
                    }
                }
                v = den > 0.0f ? sum / den : 0.0f;
            }
        }
    }
    // ---- RMSNorm (cuda/compressor.cu:174-219)
    float ss = v * v;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) ss += __shfl_xor(ss, off);
    if ((j & 63) == 0) red[j >> 6] = ss;
    __syncthreads();
    float tot = 0.0f;
    for (int w = 0; w < 8; ++w) tot += red[w];
    const float scale = 1.0f / sqrtf(tot / (float)head_dim + kRmsEps);
    if (j < head_dim) pooled[j] = v * scale * w_norm[j];
    __syncthreads();
    // ---- tail RoPE at the window start (cuda/compressor.cu:325-331, rope.cu:136-201)
    const int n_nope = head_dim - kNRot;
    float out = j < head_dim ? pooled[j] : 0.0f;
    if (j >= n_nope && j < head_dim) {
        const int p = (j - n_nope) >> 1;   // pair index
        float te = (float)R.pos;
        for (int k = 0; k < p; ++k) te *= R.theta_scale;
        const float ti = R.freq_scale * te;
        float theta = ti, ms = R.attn_factor;
        if (R.ext_factor != 0.0f) {
            const float y = ((float)p - R.corr_low) / fmaxf(0.001f, R.corr_high - R.corr_low);
            const float mix = (1.0f - fminf(1.0f, fmaxf(0.0f, y))) * R.ext_factor;
            theta = ti * (1.0f - mix) + te * mix;
            ms *= 1.0f + 0.1f * logf(1.0f / R.freq_scale);
        }
        float c, s;
        sincosf(theta, &s, &c);   // one argument reduction
        c *= ms;
        s *= ms;
        const float x0 = pooled[n_nope + 2 * p], x1 = pooled[n_nope + 2 * p + 1];
        out = ((j - n_nope) & 1) ? x0 * s + x1 * c : x0 * c - x1 * s;
    }
    // ---- FP8 round trip of the non-RoPE prefix (attention compressor only)
    if (is_attn && j < n_nope) {
        float a = fabsf(out);
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) a = fmaxf(a, __shfl_xor(a, off));
        const int e = fp8_block_exp(a);
        float q = fminf(fmaxf(ldexpf(out, -e), -448.0f), 448.0f);
        const uint32_t code = e4m3_encode(q);
        const uint32_t mag = code & 0x7Fu;
        float val;
        if (mag < 8) {
            val = (float)mag * 0.001953125f;
        } else {
            const uint32_t bits = ((mag >> 3) + 120u) << 23 | (mag & 7u) << 20;
            val = __uint_as_float(bits);
        }
        out = ldexpf((code & 0x80u) ? -val : val, e);
    }
    if (j < head_dim) emit_out[j] = out;
}

}  // namespace ds4hip
