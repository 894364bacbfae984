// indexer.hip — lightning-indexer scores and exact top-k selection.
//
// Scores (cuda/indexer_allowed.cu:68-171): score[c] = sum_h w[h] relu(q_h . k_c),
// computed with the reference kernel's own operations so that scores and the
// selected positions are bit-identical to it. The reference runs one block per
// key, thread h = head h:
//   dot_h = fma chain over d ascending from 0.0f (`dot += q * k`, contracted);
//   relu `dot < 0 ? 0 : dot`; partial_h = dot_h * w[h] (a rounded product);
//   each 32-head warp adds its partials with an xor butterfly (16, 8, 4, 2, 1),
//   warp 0 combines the warp sums with an xor butterfly over 8 lanes (4, 2, 1;
//   lanes past the last warp hold 0.0f).
// The dot chains run on the matrix cores: v_mfma_f32_16x16x4_f32 adds its
// four products to the accumulator one fma at a time, k ascending (checked bit
// for bit against fmaf, denormals, infinities and cancellation included), so
// 32 of them over d are the reference's chain. A butterfly's lane-0 result is
// a balanced binary tree, which is added with the same pairs: heads h and
// h + 16 are two accumulators of a lane, the rest are lane exchanges.
// head_dim < 128 takes one thread per key, the tree fed in leaf order (heads
// bit-reversed: h, h + 16, h + 8, h + 24, ...) to a carry chain (HeadTree).
// Floating-point contraction is off in this file: every product and sum
// rounds where the reference's does.
//
// Selection (cuda/indexer_allowed.cu:200-279): top_k rounds of argmax with
// ties to the lowest index select exactly the top_k entries in
// (score desc, index asc) order. This is computed as an exact radix select on
// order-preserving 32-bit keys (11 + 11 + 10 bits; histograms built by all
// workgroups with LDS + global atomics), which yields the threshold key T,
// the number above it and how many ties at T to take; one workgroup then
// walks the candidates in index order and emits the 0/1 mask or the
// ascending position list.

#include "ds4hip_common.h"
#include "../../include/ds4hip.h"

#include <algorithm>
#include <cstdlib>

using namespace ds4hip;

#pragma clang fp contract(off)

namespace {

constexpr int kMaxHeads = 64;
constexpr int kMaxDim = 128;
constexpr int kBins = 2048;
constexpr int kSmallSelect = 16384;   // candidates one workgroup selects in LDS (the batched select's limit)

__device__ inline unsigned ord_key(float s) {
    unsigned u = __float_as_uint(s);
    if (u == 0x80000000u) u = 0;                 // -0 ranks as +0
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

template <int kKind>   // 0 f32, 1 f16, 2 bf16
__device__ inline float key_elem(const void *keys, size_t i) {
    if (kKind == 0) return static_cast<const float *>(keys)[i];
    if (kKind == 1) return f16_bits_to_f32(static_cast<const uint16_t *>(keys)[i]);
    return bf16_to_f32(static_cast<const uint16_t *>(keys)[i]);
}

// The reference's head sum (see the top of the file), fed one leaf at a time
// in leaf order: leaf t, one head's product, of warp t / 32. An odd leaf index
// closes a pair with the level below, like a binary counter's carry.
struct HeadTree {
    static constexpr int kLevels = 5;
    float l[kLevels];
    float w0 = 0.0f, w1 = 0.0f;
    // branch-free (t is uniform, but branches here cost the caller's
    // registers): every level's sum is formed and selects keep the right ones
    __device__ inline void push(int t, float v) {
        bool carry = true;   // v still travels up
#pragma unroll
        for (int k = 0; k < kLevels; ++k) {
            const bool odd = (t >> k) & 1;
            const float up = l[k] + v;
            l[k] = (carry && !odd) ? v : l[k];
            carry = carry && odd;
            v = up;
        }
        const bool w_is_1 = (t >> kLevels) & 1;
        w0 = (carry && !w_is_1) ? v : w0;
        w1 = (carry && w_is_1) ? v : w1;
    }
    // warp 0's 8-lane butterfly over (w0, w1, 0, ..., 0): lane 0 gets
    // ((w0 + 0) + 0) + ((w1 + 0) + 0); x + 0 + 0 == x + 0
    __device__ inline float result() const { return (w0 + 0.0f) + (w1 + 0.0f); }
};

// Head of leaf t in the 5-level order: bits 0..4 reversed within the warp.
__device__ inline int head_of_leaf(int t) {
    return (t & ~31) | (int)(__builtin_bitreverse32((unsigned)(t & 31)) >> 27);
}
// relu and the rounded product of one head (cuda/indexer_allowed.cu:89-90)
__device__ inline float head_partial(float dot, float w) {
    if (dot < 0.0f) dot = 0.0f;
    return dot * w;
}

// ---- head_dim 128: scores on the fp32 matrix cores -----------------------------------------

constexpr int kTileKeys = 16;             // keys per 16x16x4 tile
constexpr int kRowStride = kMaxDim + 4;   // staged row in LDS: the 16 rows x 4 lane groups of a step on all banks

// Rows [r0, r0 + 16) of 128 elements (rows past `last` repeat it), two
// 16-byte loads (fp32) or one per thread of a 256-thread workgroup, widened
// to fp32 in LDS rows by put. `wide`: the base is 16-byte aligned; else the
// elements are read one by one.
template <int kKind>
struct TileLoad {
    static constexpr int kPer = kKind == 0 ? 4 : 8;                       // elements per 16 bytes
    static constexpr int kLoads = kTileKeys * kMaxDim / kPer / 256;       // 2 or 1
    uint4_t raw[kLoads];
    __device__ inline void load(const void *base, long long r0, long long last, bool wide) {
#pragma unroll
        for (int u = 0; u < kLoads; ++u) {
            const int v = (int)threadIdx.x + 256 * u;
            const long long r = r0 + v / (kMaxDim / kPer);
            const size_t i = (size_t)(r < last ? r : last) * kMaxDim + (v % (kMaxDim / kPer)) * kPer;
            if (kKind == 0) {
                const uint32_t *p = static_cast<const uint32_t *>(base) + i;
                raw[u] = wide ? *reinterpret_cast<const uint4_t *>(p) : uint4_t{p[0], p[1], p[2], p[3]};
            } else {
                const uint16_t *p = static_cast<const uint16_t *>(base) + i;
                if (wide) raw[u] = *reinterpret_cast<const uint4_t *>(p);
                else
#pragma unroll
                    for (int k = 0; k < 4; ++k) raw[u][k] = (uint32_t)p[2 * k] | (uint32_t)p[2 * k + 1] << 16;
            }
        }
    }
    __device__ inline void put(float *rows) const {
#pragma unroll
        for (int u = 0; u < kLoads; ++u) {
            const int v = (int)threadIdx.x + 256 * u;
            float *d = rows + (v / (kMaxDim / kPer)) * kRowStride + (v % (kMaxDim / kPer)) * kPer;
            float f[kPer];
#pragma unroll
            for (int e = 0; e < kPer; ++e) {
                const uint16_t h = (uint16_t)((raw[u][e * 4 / kPer] >> (16 * (e & 1))) & 0xFFFF);
                f[e] = kKind == 0 ? __uint_as_float(raw[u][e & 3]) : (kKind == 1 ? f16_bits_to_f32(h) : bf16_to_f32(h));
            }
#pragma unroll
            for (int e = 0; e < kPer; e += 4)
                *reinterpret_cast<float4_t *>(d + e) = float4_t{f[e], f[e + 1], f[e + 2], f[e + 3]};
        }
    }
};

// Sum over the lanes l % 16 of a value per lane, with the butterfly's offsets
// 8, 4, 2, 1 (row rotations: after the 8 step a lane's value repeats every 8
// lanes, so a rotation by 4 pairs the lanes of an xor by 4; then quads).
__device__ inline float lanes16_sum(float v) {
    v = v + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x128, 0xF, 0xF, false));
    v = v + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x124, 0xF, 0xF, false));
    v = v + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x4E, 0xF, 0xF, false));
    return v + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xB1, 0xF, 0xF, false));
}

// One sequence's keys and where its scores go.
struct ScoreSeq {
    const float *q, *w;      // [n_head][128], [n_head]
    const void *keys;
    long long row0;          // first key row
    float *scores;           // of key 0
    int n;
};

// Scores keys [c0, end) of one sequence by a workgroup of four waves, 16 a
// time: wave t takes heads 16 t .. 16 t + 15 (32 registers of query operands
// and one accumulator), and the products meet in LDS for the tree. Heads past
// n_head read the last one's query and add +0.0f, as the reference's idle threads do.
// store(key, score) is called by the lane that finished the key.
//
// What bounds it: the fp32 matrix rate, 15 ns per 16 keys x 16 heads x 4 dims
// and SIMD, to which every vector instruction adds its own time (fp32 MFMAs
// and VALU use the same units, measured). So the keys are widened once per
// workgroup into LDS rows, from which LDS reads bring the step operands; the
// next keys' loads and stores ride along, with one barrier per 16 keys. The
// query goes through LDS too, as whole rows: operand-wise 4-byte loads of it
// took 9 us of a 35k-key launch. Measured (64 heads, kernel alone): 131072
// bf16 keys 46.0 -> 34.1 us against one fma chain per thread, 35k fp32 keys
// of 16 sequences 22.4 -> 11.1 us against four chained lanes per key, and
// against a lane per head 5.2 / 8.5 / 11.7 / 18.2 -> 4.5 / 4.6 / 5.8 / 6.8 us
// at 1100 / 3000 / 6000 / 10000 keys, so one form serves every size.
//
// lds: kScoreLds floats, holding the query rows while they become operands,
// then the key tiles, the products and (hist) the caller's level-1 histogram,
// which is cleared here.
constexpr int kTileLds = kTileKeys * kRowStride;
constexpr int kScoreLds = 4 * kTileLds;                     // 33 KB: four workgroups per CU
constexpr int kPartAt = 2 * kTileLds, kHistAt = kPartAt + 2 * 4 * 4 * 64;
static_assert(kHistAt + kBins <= kScoreLds, "score LDS");
template <int kKind, class F>
__device__ inline void score_keys(const ScoreSeq &S, int n_head, int c0, int end, float *lds, bool hist, F store) {
    const int lane = threadIdx.x & 63, col = lane & 15, g = lane >> 4, t = threadIdx.x >> 6;
    const bool wide = (reinterpret_cast<uintptr_t>(S.keys) & 15) == 0;
    const long long last = S.row0 + S.n - 1;
    TileLoad<kKind> next;
    next.load(S.keys, S.row0 + c0, last, wide);
    const int h = 16 * t + col;
    const bool live = h < n_head;
    const float w = live ? S.w[h] : 0.0f;
    // this wave's 16 query rows through its quarter of lds (whole rows per
    // load: strided 4-byte loads of the operands cost more than the scoring)
    float q[kMaxDim / 4];
    {
        float *mine = lds + t * kTileLds;
        const bool wq = (reinterpret_cast<uintptr_t>(S.q) & 15) == 0;
        float4_t v[kTileKeys * kMaxDim / 4 / 64];
#pragma unroll
        for (int u = 0; u < kTileKeys * kMaxDim / 4 / 64; ++u) {
            const int i = lane + 64 * u, r = min(16 * t + i / (kMaxDim / 4), n_head - 1);
            const float *p = S.q + (size_t)r * kMaxDim + 4 * (i % (kMaxDim / 4));
            v[u] = wq ? *reinterpret_cast<const float4_t *>(p) : float4_t{p[0], p[1], p[2], p[3]};
        }
#pragma unroll
        for (int u = 0; u < kTileKeys * kMaxDim / 4 / 64; ++u) {
            const int i = lane + 64 * u;
            *reinterpret_cast<float4_t *>(mine + (i / (kMaxDim / 4)) * kRowStride + 4 * (i % (kMaxDim / 4))) = v[u];
        }
#pragma unroll
        for (int i = 0; i < kMaxDim / 4; ++i) q[i] = mine[col * kRowStride + 4 * i + g];
    }
    __syncthreads();   // lds changes its use
    unsigned *lh = reinterpret_cast<unsigned *>(lds + kHistAt);
    if (hist)
        for (int i = threadIdx.x; i < kBins; i += 256) lh[i] = 0;
    next.put(lds);
    if (c0 + kTileKeys < end) next.load(S.keys, S.row0 + c0 + kTileKeys, last, wide);
    __syncthreads();
    for (int buf = 0; c0 < end; c0 += kTileKeys, buf ^= 1) {
        const float *kr = lds + buf * kTileLds + col * kRowStride + g;
        float *part = lds + kPartAt + buf * (4 * 4 * 64) + lane;   // [wave][i][lane]
        float k[kMaxDim / 4];
#pragma unroll
        for (int i = 0; i < kMaxDim / 4; ++i) k[i] = kr[4 * i];
        if (c0 + kTileKeys < end) {
            next.put(lds + (buf ^ 1) * kTileLds);
            if (c0 + 2 * kTileKeys < end) next.load(S.keys, S.row0 + c0 + 2 * kTileKeys, last, wide);
        }
        float4_t acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int i = 0; i < kMaxDim / 4; ++i) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(k[i], q[i], acc, 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 4; ++i)   // key 4 g + i
            part[(4 * t + i) * 64] = __int_as_float(__float_as_int(head_partial(acc[i], w)) & (live ? ~0 : 0));
        // the only barrier: the other buffers are written again after the
        // next one, by when their readers are past it
        __syncthreads();
        // wave t finishes key 4 g + t of each lane group
        const float w0 = lanes16_sum(part[t * 64] + part[(4 + t) * 64]);
        const float w1 = lanes16_sum(part[(8 + t) * 64] + part[(12 + t) * 64]);
        const int c = c0 + 4 * g + t;
        // warp 0's 8-lane butterfly over (w0, w1, 0, ..., 0)
        if (col == 0 && c < S.n) store(c, (w0 + 0.0f) + (w1 + 0.0f));
    }
}

// Keys per workgroup (a multiple of 16) for n keys in all: one tile each up
// to four workgroups per CU (what the LDS holds), beyond that more tiles
// each, which spreads the query's staging over them.
constexpr int kScoreBlocks = 1024;
int score_keys_per_block(long long n) { return 16 * (int)((n + 16 * kScoreBlocks - 1) / (16 * kScoreBlocks)); }

// Any head_dim <= 128: the key row is zero-padded to 128 in registers and
// the query is read with the same padding from LDS.
template <int kKind>
__device__ inline float score_any(const float *qs, const float *ws, const void *keys, int c,
                                  int n_head, int head_dim) {
    float k[kMaxDim];
#pragma unroll
    for (int d = 0; d < kMaxDim; ++d)
        k[d] = d < head_dim ? key_elem<kKind>(keys, (size_t)c * head_dim + d) : 0.0f;
    HeadTree tree;
    const int n_leaves = (n_head + 31) & ~31;
    for (int t = 0; t < n_leaves; ++t) {
        const int h = head_of_leaf(t);
        float p = 0.0f;
        if (h < n_head) {
            const float *qh = qs + h * head_dim;
            float dot = 0.0f;
#pragma unroll
            for (int d = 0; d < kMaxDim; ++d)
                if (d < head_dim) dot = fmaf(qh[d], k[d], dot);
            p = head_partial(dot, ws[h]);
        }
        tree.push(t, p);
    }
    return tree.result();
}

// Scores of one sequence and, with hist, the level-1 histogram of the first
// n_cand. kFull: head_dim == 128, keys_per_blk keys per workgroup; else one
// thread per key with the query in LDS.
template <int kKind, bool kFull>
__global__ __launch_bounds__(256) void score_kernel(const float *__restrict__ q,
                                                    const float *__restrict__ w,
                                                    const void *__restrict__ keys, int n_comp,
                                                    int n_head, int head_dim,
                                                    float *__restrict__ scores,
                                                    unsigned *__restrict__ hist, int n_cand, int keys_per_blk) {
    // kFull: lh is the histogram part of its LDS; else it follows the query
    __shared__ __attribute__((aligned(16))) float lds[kFull ? kScoreLds : kMaxHeads * kMaxDim + kMaxHeads + kBins];
    unsigned *lh = reinterpret_cast<unsigned *>(lds + (kFull ? kHistAt : kMaxHeads * kMaxDim + kMaxHeads));
    if (kFull) {
        const ScoreSeq S{q, w, keys, 0, scores, n_comp};
        const int c0 = blockIdx.x * keys_per_blk;
        score_keys<kKind>(S, n_head, c0, min(c0 + keys_per_blk, n_comp), lds, hist != nullptr, [&](int c, float s) {
            scores[c] = s;
            if (hist && c < n_cand) atomicAdd(&lh[ord_key(s) >> 21], 1u);
        });
    } else {
        float *qs = lds, *ws = lds + kMaxHeads * kMaxDim;
        if (hist)
            for (int i = threadIdx.x; i < kBins; i += 256) lh[i] = 0;
        stage_to_lds(qs, q, n_head * head_dim);
        for (int i = threadIdx.x; i < n_head; i += 256) ws[i] = w[i];
        __syncthreads();
        const int c = blockIdx.x * 256 + threadIdx.x;
        if (c < n_comp) {
            const float s = score_any<kKind>(qs, ws, keys, c, n_head, head_dim);
            scores[c] = s;
            if (hist && c < n_cand) atomicAdd(&lh[ord_key(s) >> 21], 1u);
        }
    }
    if (hist) {
        __syncthreads();
        for (int i = threadIdx.x; i < kBins; i += 256)
            if (lh[i]) atomicAdd(&hist[i], lh[i]);
    }
}

__global__ void zero_u32_kernel(unsigned *p, int n) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) p[i] = 0;
}

// Inclusive prefix sum over the 256 threads of a workgroup (4 waves).
__device__ inline unsigned block_incl_scan(unsigned v, unsigned *wsum) {
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const unsigned u = __shfl_up(v, off);
        if (lane >= off) v += u;
    }
    if (lane == 63) wsum[wv] = v;
    __syncthreads();
    unsigned before = 0;
    for (int i = 0; i < wv; ++i) before += wsum[i];
    __syncthreads();
    return v + before;
}

// Finds, in histogram h (nb bins, high bin = larger keys), the bin holding the
// need-th largest key and the count strictly above that bin (need == 0:
// the top bin, nothing above).
// Called by every thread of a 256-thread workgroup: thread t sums bins
// [nb-1-t*per, nb-1-(t+1)*per), a block scan finds the thread whose range
// crosses need, and that thread walks its <= 8 bins.
__device__ void find_bin(const unsigned *h, int nb, unsigned need, unsigned *s_bin,
                         unsigned *s_above, unsigned *scratch) {
    const int t = threadIdx.x;
    const int per = nb / 256;
    unsigned local = 0;
    for (int i = 0; i < per; ++i) local += h[nb - 1 - (t * per + i)];
    const unsigned incl = block_incl_scan(local, scratch);
    const unsigned excl = incl - local;
    if (need == 0) {
        if (t == 0) {
            *s_bin = (unsigned)(nb - 1);
            *s_above = 0;
        }
    } else if (excl < need && incl >= need) {
        unsigned run = excl;
        int bin = nb - 1 - t * per;
        for (int i = 0; i < per - 1; ++i, --bin) {
            if (run + h[bin] >= need) break;
            run += h[bin];
        }
        *s_bin = (unsigned)bin;
        *s_above = run;
    }
    __syncthreads();
}

// Threshold key T (the need0-th largest candidate key) and the number of
// candidates equal to T that are taken (lowest indices first).
__device__ void threshold(const unsigned *hists, unsigned need0, unsigned *T, unsigned *need_eq,
                          unsigned *scratch, unsigned *s_bin, unsigned *s_above) {
    unsigned need = need0;
    find_bin(hists, kBins, need, s_bin, s_above, scratch);
    unsigned t = *s_bin << 21;
    need -= *s_above;
    __syncthreads();
    find_bin(hists + kBins, kBins, need, s_bin, s_above, scratch);
    t |= *s_bin << 10;
    need -= *s_above;
    __syncthreads();
    find_bin(hists + 2 * kBins, 1024, need, s_bin, s_above, scratch);
    t |= *s_bin;
    need -= *s_above;
    *T = t;
    *need_eq = need;
}

// Stage 2 / 3 histogram: recompute the selection state from the previous
// histograms, then histogram the next bit field of keys matching the prefix.
template <int kStage>
__global__ __launch_bounds__(256) void hist_next_kernel(const float *__restrict__ scores,
                                                        int n_cand, unsigned need0,
                                                        unsigned *__restrict__ hists) {
    __shared__ unsigned lh[kBins];
    __shared__ unsigned scratch[256];
    __shared__ unsigned s_bin, s_above;
    unsigned *h1 = hists, *h2 = hists + kBins, *h3 = hists + 2 * kBins;
    find_bin(h1, kBins, need0, &s_bin, &s_above, scratch);
    unsigned prefix = s_bin << 21, need = need0 - s_above;
    int shift = 10, nb = kBins;
    if (kStage == 3) {
        __syncthreads();
        find_bin(h2, kBins, need, &s_bin, &s_above, scratch);
        prefix |= s_bin << 10;
        shift = 0;
        nb = 1024;
    }
    for (int i = threadIdx.x; i < nb; i += 256) lh[i] = 0;
    __syncthreads();
    const unsigned mask_hi = kStage == 2 ? 0xFFE00000u : 0xFFFFFC00u;
    for (int c = blockIdx.x * 256 + threadIdx.x; c < n_cand; c += gridDim.x * 256) {
        const unsigned k = ord_key(scores[c]);
        if ((k & mask_hi) == prefix) atomicAdd(&lh[(k >> shift) & (nb - 1)], 1u);
    }
    __syncthreads();
    unsigned *dst = kStage == 2 ? h2 : h3;
    for (int i = threadIdx.x; i < nb; i += 256)
        if (lh[i]) atomicAdd(&dst[i], lh[i]);
}

constexpr int kChunk = 1024;   // positions per emit workgroup (256 threads x 4)

// Per chunk: candidates strictly above T and equal to T.
__global__ __launch_bounds__(256) void count_kernel(const float *__restrict__ scores, int n_cand,
                                                    unsigned need0,
                                                    const unsigned *__restrict__ hists,
                                                    unsigned *__restrict__ chunk_gt,
                                                    unsigned *__restrict__ chunk_eq) {
    __shared__ unsigned scratch[256];
    __shared__ unsigned s_bin, s_above, red[2][4];
    unsigned T, need_eq;
    threshold(hists, need0, &T, &need_eq, scratch, &s_bin, &s_above);
    unsigned gt = 0, eq = 0;
    for (int i = 0; i < 4; ++i) {
        const int c = blockIdx.x * kChunk + i * 256 + threadIdx.x;
        if (c < n_cand) {
            const unsigned k = ord_key(scores[c]);
            gt += k > T;
            eq += k == T;
        }
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        gt += __shfl_xor(gt, off);
        eq += __shfl_xor(eq, off);
    }
    if ((threadIdx.x & 63) == 0) {
        red[0][threadIdx.x >> 6] = gt;
        red[1][threadIdx.x >> 6] = eq;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        chunk_gt[blockIdx.x] = red[0][0] + red[0][1] + red[0][2] + red[0][3];
        chunk_eq[blockIdx.x] = red[1][0] + red[1][1] + red[1][2] + red[1][3];
    }
}

// Block-wide exclusive scan of 256 values (one per thread); returns the total.
__device__ unsigned block_excl_scan(unsigned v, unsigned *buf, unsigned *excl) {
    const int t = threadIdx.x;
    buf[t] = v;
    __syncthreads();
    for (int off = 1; off < 256; off <<= 1) {
        const unsigned u = t >= off ? buf[t - off] : 0;
        __syncthreads();
        buf[t] += u;
        __syncthreads();
    }
    *excl = buf[t] - v;
    const unsigned total = buf[255];
    __syncthreads();
    return total;
}

// Per chunk: every candidate above T, ties at T in index order while the
// global tie rank < need_eq, and every position >= n_cand (the forced recent
// window). Writes the 0/1 mask and/or the ascending position list.
__global__ __launch_bounds__(256) void emit_kernel(const float *__restrict__ scores, int n_comp,
                                                   int n_cand, unsigned need0,
                                                   const unsigned *__restrict__ hists,
                                                   const unsigned *__restrict__ chunk_gt,
                                                   const unsigned *__restrict__ chunk_eq,
                                                   int32_t *__restrict__ mask,
                                                   int32_t *__restrict__ pos_out) {
    __shared__ unsigned scratch[256], buf[256];
    __shared__ unsigned s_bin, s_above;
    unsigned T, need_eq;
    threshold(hists, need0, &T, &need_eq, scratch, &s_bin, &s_above);
    // selections and ties of the earlier chunks
    unsigned sel_b = 0, eq_b = 0;
    for (int c2 = threadIdx.x; c2 < (int)blockIdx.x; c2 += 256) {
        eq_b += chunk_eq[c2];
        sel_b += chunk_gt[c2];
    }
    unsigned ex;
    const unsigned eq_before = block_excl_scan(eq_b, buf, &ex);
    const unsigned gt_before = block_excl_scan(sel_b, buf, &ex);
    // ties taken by earlier chunks = min(need_eq, ties before)
    const unsigned ties_taken_before = eq_before < need_eq ? eq_before : need_eq;
    const unsigned sel_before = gt_before + ties_taken_before;
    // this thread's 4 consecutive positions
    const int base = blockIdx.x * kChunk + threadIdx.x * 4;
    unsigned k4[4];
    unsigned my_eq = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int c = base + i;
        k4[i] = (c < n_cand) ? ord_key(scores[c]) : 0;
        my_eq += (c < n_cand) && k4[i] == T;
    }
    unsigned eq_ex;
    block_excl_scan(my_eq, buf, &eq_ex);
    unsigned rank = eq_before + eq_ex;
    bool take[4];
    unsigned my_sel = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int c = base + i;
        bool t = false;
        if (c < n_cand) {
            if (k4[i] > T) t = true;
            else if (k4[i] == T) { t = rank < need_eq; ++rank; }
        } else if (c < n_comp) {
            t = true;
        }
        take[i] = t;
        my_sel += t;
    }
    unsigned sel_ex;
    block_excl_scan(my_sel, buf, &sel_ex);
    unsigned o = sel_before + sel_ex;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int c = base + i;
        if (c >= n_comp) break;
        if (mask) mask[c] = take[i] ? 1 : 0;
        if (take[i] && pos_out) pos_out[o] = c;
        o += take[i];
    }
}

__global__ void fill_kernel(int32_t *out, int n, int32_t v, int iota) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
        out[i] = iota ? i : v;
}

__global__ void scale_kernel(float *y, int n, float s) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) y[i] *= s;
}

int launch_scores(const float *q, const float *w, const void *keys, int kind, int n_comp,
                  int n_head, int head_dim, float *scores, unsigned *hist, int n_cand,
                  hipStream_t st) {
    const bool full = head_dim == kMaxDim;
    const int kpb = full ? score_keys_per_block(n_comp) : 256;
    const dim3 grid((n_comp + kpb - 1) / kpb);
    switch (kind) {
    case 0:
        if (full) hipLaunchKernelGGL((score_kernel<0, true>), grid, dim3(256), 0, st, q, w, keys, n_comp, n_head, head_dim, scores, hist, n_cand, kpb);
        else hipLaunchKernelGGL((score_kernel<0, false>), grid, dim3(256), 0, st, q, w, keys, n_comp, n_head, head_dim, scores, hist, n_cand, kpb);
        break;
    case 1:
        if (full) hipLaunchKernelGGL((score_kernel<1, true>), grid, dim3(256), 0, st, q, w, keys, n_comp, n_head, head_dim, scores, hist, n_cand, kpb);
        else hipLaunchKernelGGL((score_kernel<1, false>), grid, dim3(256), 0, st, q, w, keys, n_comp, n_head, head_dim, scores, hist, n_cand, kpb);
        break;
    default:
        if (full) hipLaunchKernelGGL((score_kernel<2, true>), grid, dim3(256), 0, st, q, w, keys, n_comp, n_head, head_dim, scores, hist, n_cand, kpb);
        else hipLaunchKernelGGL((score_kernel<2, false>), grid, dim3(256), 0, st, q, w, keys, n_comp, n_head, head_dim, scores, hist, n_cand, kpb);
        break;
    }
    return hip_status(hipGetLastError());
}

// scores + selection. mask and/or pos_out; n_recent trailing positions are
// always selected and take part in no comparison.
size_t select_large_scratch_words(int n_comp);
size_t select_scratch_bytes(int n_comp) {
    const size_t chunks = (size_t)(n_comp > 0 ? n_comp : 1) / kChunk + 1;
    return std::max((3 * kBins + 2 * chunks), select_large_scratch_words(n_comp)) * sizeof(unsigned);
}

int launch_select_large(const float *scores, int n_comp, int n_cand, unsigned need0, unsigned *scratch,
                        int32_t *mask, int32_t *pos_out, hipStream_t st);
size_t select_large_scratch_words(int n_comp);
constexpr int kLargeSelectMax = 262144;   // candidates of the two-launch select (its LDS bitmaps)

int score_select(const float *q, const float *w, const void *keys, int kind, int n_comp,
                 int n_head, int head_dim, int top_k, int n_recent, float *scores,
                 unsigned *scratch, int32_t *mask, int32_t *pos_out, hipStream_t st) {
    if (!q || !w || !keys || !scores || !scratch || n_head <= 0 || n_head > kMaxHeads ||
        head_dim <= 0 || head_dim > kMaxDim || n_recent < 0 || (!mask && !pos_out))
        return kEINVAL;
    if (n_comp <= 0) return 0;
    if (top_k <= 0) {
        if (mask) hipLaunchKernelGGL(fill_kernel, dim3((n_comp + 255) / 256), dim3(256), 0, st, mask, n_comp, 0, 0);
        return hip_status(hipGetLastError());
    }
    if (n_comp <= top_k) {
        int rc = launch_scores(q, w, keys, kind, n_comp, n_head, head_dim, scores, nullptr, 0, st);
        if (rc) return rc;
        if (mask) hipLaunchKernelGGL(fill_kernel, dim3((n_comp + 255) / 256), dim3(256), 0, st, mask, n_comp, 1, 0);
        if (pos_out) hipLaunchKernelGGL(fill_kernel, dim3((n_comp + 255) / 256), dim3(256), 0, st, pos_out, n_comp, 0, 1);
        return hip_status(hipGetLastError());
    }
    const int recent = n_recent < top_k ? n_recent : top_k;
    const int n_cand = n_comp - recent;
    // Few candidates and positions only (the model's decode: a few thousand
    // compressed rows): the batched pair with one sequence, the scores and
    // one workgroup's LDS radix select, two launches instead of six;
    // the same scores and the same selection rule.
    if (!mask && head_dim == kMaxDim && n_cand <= kSmallSelect) {
        const long long row0 = 0;
        return ds4hip_indexer_topk_positions_batch(q, w, keys, kind, &row0, &n_comp, 1, n_head, head_dim, top_k,
                                                   n_recent, scores, pos_out, top_k, st);
    }
    const unsigned need0 = (unsigned)(top_k - recent);
    const int n_chunks = (n_comp + kChunk - 1) / kChunk;
    unsigned *hists = scratch;
    unsigned *chunk_gt = scratch + 3 * kBins;
    unsigned *chunk_eq = chunk_gt + n_chunks;
    // up to kLargeSelectMax candidates (16-byte aligned scores): the level-1
    // histogram in the score kernel, then the two-launch select
    if (n_cand <= kLargeSelectMax && (reinterpret_cast<uintptr_t>(scores) & 15) == 0) {
        // level-1 histogram, list counter and bitmap start at zero
        const int nz = kBins + 1 + (n_cand + 31) / 32;
        hipLaunchKernelGGL(zero_u32_kernel, dim3((nz + 255) / 256), dim3(256), 0, st, scratch, nz);
        int rc = launch_scores(q, w, keys, kind, n_comp, n_head, head_dim, scores, scratch, n_cand, st);
        if (rc) return rc;
        return launch_select_large(scores, n_comp, n_cand, need0, scratch, mask, pos_out, st);
    }
    hipLaunchKernelGGL(zero_u32_kernel, dim3(24), dim3(256), 0, st, hists, 3 * kBins);
    int rc = launch_scores(q, w, keys, kind, n_comp, n_head, head_dim, scores, hists, n_cand, st);
    if (rc) return rc;
    const int g = (n_cand + 256 * 8 - 1) / (256 * 8) + 1;
    hipLaunchKernelGGL(hist_next_kernel<2>, dim3(g), dim3(256), 0, st, scores, n_cand, need0, hists);
    hipLaunchKernelGGL(hist_next_kernel<3>, dim3(g), dim3(256), 0, st, scores, n_cand, need0, hists);
    hipLaunchKernelGGL(count_kernel, dim3(n_chunks), dim3(256), 0, st, scores, n_cand, need0, hists,
                       chunk_gt, chunk_eq);
    hipLaunchKernelGGL(emit_kernel, dim3(n_chunks), dim3(256), 0, st, scores, n_comp, n_cand, need0,
                       hists, chunk_gt, chunk_eq, mask, pos_out);
    return hip_status(hipGetLastError());
}

}  // namespace

extern "C" int ds4hip_indexer_allowed_short_circuit_i32(int32_t *out_i32, int n_comp, int top_k,
                                                        void *stream) {
    // cuda/indexer_allowed.cu:283-305: n_comp <= 0 -> nothing; n_comp > top_k
    // is a caller error (the reference aborts; here it is reported).
    if (n_comp <= 0) return 0;
    if (!out_i32 || n_comp > top_k) return ds4hip_set_last_error(kEINVAL);
    hipLaunchKernelGGL(fill_kernel, dim3((n_comp + 127) / 128), dim3(128), 0, (hipStream_t)stream,
                       out_i32, n_comp, 1, 0);
    return ds4hip_set_last_error(hip_status(hipGetLastError()));
}

extern "C" int ds4hip_scale_inplace_f32(float *y, int n, float scale, void *stream) {
    if (n <= 0) return 0;
    if (!y) return ds4hip_set_last_error(kEINVAL);
    hipLaunchKernelGGL(scale_kernel, dim3((n + 63) / 64), dim3(64), 0, (hipStream_t)stream, y, n, scale);
    return ds4hip_set_last_error(hip_status(hipGetLastError()));
}

extern "C" size_t ds4hip_indexer_select_scratch_bytes(int n_comp) { return select_scratch_bytes(n_comp); }

// The reference launchers take only a score scratch; the selection
// histograms live in the library's per-stream scratch (no allocation once it
// has grown to the size a stream needs).
static int with_hists(int (*fn)(unsigned *, void *), void *ctx, int n_comp, hipStream_t st) {
    void *h = nullptr;
    const int e = stream_scratch(st, select_scratch_bytes(n_comp), &h);
    if (e) return e;
    return fn(static_cast<unsigned *>(h), ctx);
}

struct TopkCall {
    const float *q, *w;
    const void *keys;
    int kind, n_comp, n_head, head_dim, top_k;
    int32_t *allowed;
    float *scores;
    hipStream_t st;
};

extern "C" int ds4hip_indexer_score_topk_i32(const float *q, const float *weights,
                                             const uint16_t *index_comp, int n_comp, int n_head,
                                             int head_dim, int top_k, int32_t *allowed_out,
                                             float *scratch_scores, void *stream) {
    if (n_comp <= 0 || n_head <= 0 || head_dim <= 0) return 0;   // cuda/indexer_allowed.cu:330-331
    TopkCall c{q, weights, index_comp, 1, n_comp, n_head, head_dim, top_k, allowed_out,
               scratch_scores, (hipStream_t)stream};
    return ds4hip_set_last_error(with_hists(
        [](unsigned *h, void *p) {
            auto *c = static_cast<TopkCall *>(p);
            return score_select(c->q, c->w, c->keys, c->kind, c->n_comp, c->n_head, c->head_dim,
                                c->top_k, 0, c->scores, h, c->allowed, nullptr, c->st);
        },
        &c, n_comp, (hipStream_t)stream));
}

extern "C" int ds4hip_indexer_score_topk_f32_i32(const float *q, const float *weights,
                                                 const float *index_comp_f32, int n_comp,
                                                 int n_head, int head_dim, int top_k,
                                                 int32_t *allowed_out, float *scratch_scores,
                                                 void *stream) {
    if (n_comp <= 0 || n_head <= 0 || head_dim <= 0) return 0;
    TopkCall c{q, weights, index_comp_f32, 0, n_comp, n_head, head_dim, top_k, allowed_out,
               scratch_scores, (hipStream_t)stream};
    return ds4hip_set_last_error(with_hists(
        [](unsigned *h, void *p) {
            auto *c = static_cast<TopkCall *>(p);
            return score_select(c->q, c->w, c->keys, c->kind, c->n_comp, c->n_head, c->head_dim,
                                c->top_k, 0, c->scores, h, c->allowed, nullptr, c->st);
        },
        &c, n_comp, (hipStream_t)stream));
}

extern "C" int ds4hip_indexer_topk_positions(const float *q, const float *weights,
                                             const void *keys, int key_kind, int n_comp,
                                             int n_head, int head_dim, int top_k, int n_recent,
                                             float *scratch_scores, void *scratch_select,
                                             int32_t *allowed_mask, int32_t *positions_out,
                                             void *stream) {
    if (key_kind < 0 || key_kind > 2) return ds4hip_set_last_error(kEINVAL);
    return ds4hip_set_last_error(score_select(
        q, weights, keys, key_kind, n_comp, n_head, head_dim, top_k, n_recent, scratch_scores,
        static_cast<unsigned *>(scratch_select), allowed_mask, positions_out, (hipStream_t)stream));
}

// ---- batched selection (several sequences, one launch per phase) -------------------------
//
// Scores: the key rows of all sequences are concatenated; block ranges per
// sequence come from a prefix table in the kernel arguments, so each block
// scores keys of one sequence with that sequence's query and weights.
// Selection: one 1024-thread workgroup per sequence holds the ordered keys of
// its candidates in LDS (up to kSelMax) and runs a 4 x 8-bit radix select,
// then emits the positions in ascending order (same rule as above: the top
// (score desc, index asc) plus the forced recent window).

namespace {

constexpr int kMaxSeq = 16;
constexpr int kSelMax = 16384;

struct BatchArgs {
    const float *q;            // [n_seq][n_head][128]
    const float *w;            // [n_seq][n_head]
    const void *keys;          // key rows, sequence s at row key0[s]
    float *scores;             // same indexing as the key rows
    int32_t *pos_out;          // [n_seq][pos_stride]
    int n_seq, n_head, top_k, n_recent, pos_stride, keys_per_blk;
    long long key0[kMaxSeq];
    int n_comp[kMaxSeq];
    int blk0[kMaxSeq + 1];     // first score block of each sequence
};

// The sequence of score workgroup blockIdx.x, and its first key there.
__device__ inline ScoreSeq batch_seq(const BatchArgs &A, int keys_per_blk, int &c0) {
    int s = 0;
#pragma unroll
    for (int i = 1; i < kMaxSeq; ++i)
        if (i < A.n_seq && (int)blockIdx.x >= A.blk0[i]) s = i;
    ScoreSeq S{};
    int first = 0;
#pragma unroll
    for (int i = 0; i < kMaxSeq; ++i)
        if (i == s) {
            S.n = A.n_comp[i];
            S.row0 = A.key0[i];
            first = A.blk0[i];
        }
    S.q = A.q + (size_t)s * A.n_head * kMaxDim;
    S.w = A.w + (size_t)s * A.n_head;
    S.keys = A.keys;
    S.scores = A.scores + S.row0;
    c0 = ((int)blockIdx.x - first) * keys_per_blk;
    return S;
}

template <int kKind>
__global__ __launch_bounds__(256) void score_batch_kernel(const BatchArgs A) {
    __shared__ __attribute__((aligned(16))) float lds[kScoreLds];
    int c0;
    const ScoreSeq S = batch_seq(A, A.keys_per_blk, c0);
    score_keys<kKind>(S, A.n_head, c0, min(c0 + A.keys_per_blk, S.n), lds, false,
                      [&](int c, float s) { S.scores[c] = s; });
}

__device__ inline unsigned scan1024_excl(unsigned v, unsigned *wsum, unsigned *total) {
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    unsigned x = v;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const unsigned u = __shfl_up(x, off);
        if (lane >= off) x += u;
    }
    if (lane == 63) wsum[wv] = x;
    __syncthreads();
    unsigned before = 0, tot = 0;
    for (int i = 0; i < 16; ++i) {
        const unsigned t = wsum[i];
        before += i < wv ? t : 0;
        tot += t;
    }
    __syncthreads();
    *total = tot;
    return before + x - v;
}

// Inclusive prefix sum over the 64 lanes of a wave.
__device__ inline unsigned wave_scan_incl(unsigned x) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const unsigned y = __shfl_up(x, off);
        x += lane >= off ? y : 0u;
    }
    return x;
}

// Exclusive prefix sum over a 1024-thread workgroup of small per-thread
// values (below 32): within a wave from ballots of the values' bit planes (no
// lane shuffles), then the 16 wave totals through LDS with one barrier. ws is
// this scan's own 16 words (not reused by another scan of the launch).
__device__ inline unsigned scan1024_small(unsigned v, unsigned *ws, unsigned *total) {
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    unsigned below = 0, wtot = 0;
#pragma unroll
    for (int b = 0; b < 5; ++b) {
        const unsigned long long m = __ballot((v >> b) & 1u);
        below += __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u)) << b;
        wtot += (unsigned)__popcll(m) << b;
    }
    if (lane == 0) ws[wv] = wtot;
    __syncthreads();
    unsigned before = 0, tot = 0;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const unsigned x = ws[i];
        before += i < wv ? x : 0u;
        tot += x;
    }
    *total = tot;
    return before + below;
}

// One 1024-thread workgroup selects of scores[0, n), n > top_k (see the top of
// this section), and writes the positions to out.
__device__ inline void select_body(const float *__restrict__ scores, int n, int top_k, int n_recent,
                                   int32_t *__restrict__ out) {
    __shared__ unsigned keys[kSelMax];
    __shared__ __attribute__((aligned(16))) unsigned hist[2][256];
    __shared__ unsigned wemit[2][16];
    const int t = threadIdx.x;
    const int recent = n_recent < top_k ? n_recent : top_k;
    const int n_cand = n - recent;
    const unsigned need0 = (unsigned)(top_k - recent);
    // four loads in flight per thread (clamped, not branched): a strided copy
    // loop would wait for each load in turn
    for (int b = 0; b < n_cand; b += 4096) {
        unsigned v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) v[u] = ord_key(scores[min(b + 1024 * u + t, n_cand - 1)]);
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (b + 1024 * u + t < n_cand) keys[b + 1024 * u + t] = v[u];
    }
    // radix select of the need0-th largest key, 8 bits at a time. Two
    // histograms alternate by pass, so a pass is two barriers: every wave
    // reads the whole histogram (4 bins per lane) and finds the threshold
    // bin itself with a lane scan; the next pass's histogram is cleared
    // meanwhile (its last reads were before this pass's first barrier).
    if (t < 256) hist[0][t] = 0;
    unsigned prefix = 0, pmask = 0, need = need0;
    for (int shift = 24, p = 0; shift >= 0 && need > 0; shift -= 8, ++p) {
        unsigned *h = hist[p & 1];
        __syncthreads();
        for (int i = t; i < n_cand; i += 1024) {
            const unsigned k = keys[i];
            if ((k & pmask) == prefix) atomicAdd(&h[(k >> shift) & 255], 1u);
        }
        __syncthreads();
        if (t < 256) hist[(p + 1) & 1][t] = 0;
        const int lane = t & 63;
        // lane l: bins 255 - 4l down to 252 - 4l
        const uint4_t c4 = *reinterpret_cast<const uint4_t *>(h + 252 - 4 * lane);
        const unsigned ls = c4[0] + c4[1] + c4[2] + c4[3];
        const unsigned cum = wave_scan_incl(ls);
        const int L = __builtin_ctzll(__ballot(cum >= need));
        unsigned acc = cum - ls, bin = 0, above = 0;
        bool found = false;
#pragma unroll
        for (int i = 3; i >= 0; --i) {
            const unsigned v = c4[i];
            if (!found && acc + v >= need) {
                found = true;
                bin = (unsigned)(252 - 4 * lane + i);
                above = acc;
            }
            acc += v;
        }
        prefix |= (unsigned)__builtin_amdgcn_readlane((int)bin, L) << shift;
        pmask |= 255u << shift;
        need -= (unsigned)__builtin_amdgcn_readlane((int)above, L);
    }
    if (need0 == 0) __syncthreads();   // the keys' stores, otherwise ordered by the passes' barriers
    // need0 == 0 leaves T above every key
    const unsigned T = need0 ? prefix : 0xFFFFFFFFu;
    const unsigned need_eq = need0 ? need : 0;
    // emit in index order: thread t owns a contiguous range
    const int per = (n_cand + 1023) / 1024;
    const int b0 = t * per, b1 = min(b0 + per, n_cand);
    unsigned n_eq = 0;
    for (int i = b0; i < b1; ++i) n_eq += keys[i] == T;
    unsigned tot_eq;
    // per <= 16 keys per thread: the counts are small
    unsigned eq_rank = scan1024_small(n_eq, wemit[0], &tot_eq);
    unsigned n_sel = 0;
    {
        unsigned r = eq_rank;
        for (int i = b0; i < b1; ++i) {
            const unsigned k = keys[i];
            if (k > T) ++n_sel;
            else if (k == T) { n_sel += r < need_eq; ++r; }
        }
    }
    unsigned tot_sel;
    unsigned o = scan1024_small(n_sel, wemit[1], &tot_sel);
    {
        unsigned r = eq_rank;
        for (int i = b0; i < b1; ++i) {
            const unsigned k = keys[i];
            bool take = k > T;
            if (k == T) { take = r < need_eq; ++r; }
            if (take) out[o++] = i;
        }
    }
    for (int i = t; i < recent; i += 1024) out[tot_sel + i] = n_cand + i;
}

__global__ __launch_bounds__(1024) void select_batch_kernel(const BatchArgs A) {
    const int s = blockIdx.x;
    int n = 0;
    long long k0 = 0;
#pragma unroll
    for (int i = 0; i < kMaxSeq; ++i)
        if (i == s) {
            n = A.n_comp[i];
            k0 = A.key0[i];
        }
    int32_t *out = A.pos_out + (size_t)s * A.pos_stride;
    if (n <= A.top_k) {
        for (int i = threadIdx.x; i < n; i += 1024) out[i] = i;
        return;
    }
    select_body(A.scores + k0, n, A.top_k, A.n_recent, out);
}

// ---- the tokens of a prompt chunk: one key list that grows along the chunk -----------------

struct ChunkSelArgs {
    const float *q, *w;        // [n][n_head][128], [n][n_head]
    const float *keys;         // fp32 rows
    float *scores;             // [n][stride]
    int32_t *pos_out;          // [n][top_k]
    int n_head, top_k, stride, keys_per_blk;
    int n0, p0, ratio;         // keys before the chunk, its first position, tokens per key
    __device__ inline int keys_of(int t) const { return n0 + (p0 + t + 1) / ratio - p0 / ratio; }
};

__global__ __launch_bounds__(256) void score_chunk_kernel(const ChunkSelArgs A) {
    __shared__ __attribute__((aligned(16))) float lds[kScoreLds];
    const int t = blockIdx.y, n = A.keys_of(t), c0 = (int)blockIdx.x * A.keys_per_blk;
    if (n <= A.top_k || c0 >= n) return;
    const ScoreSeq S{A.q + (size_t)t * A.n_head * kMaxDim, A.w + (size_t)t * A.n_head, A.keys, 0,
                     A.scores + (size_t)t * A.stride, n};
    score_keys<0>(S, A.n_head, c0, min(c0 + A.keys_per_blk, n), lds, false, [&](int c, float s) { S.scores[c] = s; });
}

__global__ __launch_bounds__(1024) void select_chunk_kernel(const ChunkSelArgs A) {
    const int t = blockIdx.x, n = A.keys_of(t);
    if (n <= A.top_k) return;
    select_body(A.scores + (size_t)t * A.stride, n, A.top_k, 0, A.pos_out + (size_t)t * A.top_k);
}

// ---- two-launch selection of a long candidate list ----------------------------------------
//
// After the score kernel's level-1 histogram (key bits 31..21):
//  compact (one workgroup per 1024 candidates, coalesced): keys above the
//    level-1 threshold bin set their bit in a global bitmap; keys in the bin
//    are appended, unordered, to a global list of (key, index) pairs (one
//    counter add per wave);
//  finish (one 1024-thread workgroup): levels 2 (bits 20..10) and 3 (bits
//    9..0) of the radix select over the listed keys give the exact threshold
//    key T and the number of ties at T to take; listed keys above T join the
//    bitmap (copied to LDS), keys equal to T go to a tie bitmap whose
//    popcount scan ranks them by index, and the need_eq lowest join too; a
//    popcount scan of the bitmap writes the positions in ascending order (and
//    / or the 0/1 mask), then the forced recent window.
// Two launches instead of four, and the full score list is read once more
// instead of three times. The list has room for every candidate, so a
// threshold bin of any size is handled (a large one only costs list reads).
constexpr int kLargeBits = 262144;   // candidates the finishing workgroup's LDS bitmaps cover
constexpr int kFinishPairs = 8192;   // listed keys it copies to LDS (a longer list is read from memory)

__global__ __launch_bounds__(256) void compact_kernel(const float *__restrict__ scores, int n_cand,
                                                      unsigned need0, const unsigned *__restrict__ hist1,
                                                      unsigned *__restrict__ bitmap,
                                                      unsigned *__restrict__ list_n,
                                                      unsigned *__restrict__ list_key,
                                                      int *__restrict__ list_idx) {
    __shared__ unsigned scratch[256];
    __shared__ unsigned s_bin, s_above;
    if (need0 == 0) return;
    find_bin(hist1, kBins, need0, &s_bin, &s_above, scratch);
    const unsigned b1 = s_bin;
    const int c = blockIdx.x * kChunk + 4 * threadIdx.x;
    unsigned k[4];
    if (c + 3 < n_cand) {
        const float4_t v = *reinterpret_cast<const float4_t *>(scores + c);
#pragma unroll
        for (int j = 0; j < 4; ++j) k[j] = ord_key(v[j]);
    } else {
#pragma unroll
        for (int j = 0; j < 4; ++j) k[j] = c + j < n_cand ? ord_key(scores[c + j]) : 0;
    }
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    // in-bin keys: per-wave ballots, one counter add per workgroup (a counter
    // add per wave would serialize ~1000 same-address atomics)
    __shared__ unsigned s_wcnt[4][4], s_base;
    unsigned long long bal[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const bool live = c + j < n_cand;
        const unsigned hb = k[j] >> 21;
        if (live && hb > b1) atomicOr(&bitmap[(c + j) >> 5], 1u << ((c + j) & 31));
        bal[j] = __ballot(live && hb == b1);
        if (lane == 0) s_wcnt[wv][j] = (unsigned)__popcll(bal[j]);
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned tot = 0;
        for (int w = 0; w < 4; ++w)
            for (int j = 0; j < 4; ++j) {
                const unsigned n = s_wcnt[w][j];
                s_wcnt[w][j] = tot;   // exclusive prefix in (wave, j) order
                tot += n;
            }
        s_base = tot ? atomicAdd(list_n, tot) : 0;
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < 4; ++j)
        if ((bal[j] >> lane) & 1) {
            const unsigned o = s_base + s_wcnt[wv][j] + (unsigned)__popcll(bal[j] & ((1ULL << lane) - 1));
            list_key[o] = k[j];
            list_idx[o] = c + j;
        }
}

__global__ __launch_bounds__(1024) void finish_kernel(int n_comp, int n_cand, unsigned need0,
                                                      const unsigned *__restrict__ hist1,
                                                      const unsigned *__restrict__ bitmap,
                                                      const unsigned *__restrict__ list_n,
                                                      const unsigned *__restrict__ list_key,
                                                      const int *__restrict__ list_idx,
                                                      int32_t *__restrict__ mask,
                                                      int32_t *__restrict__ pos_out) {
    __shared__ unsigned sel[kLargeBits / 32];
    __shared__ unsigned tie[kLargeBits / 32];
    __shared__ unsigned hist[kBins];
    __shared__ unsigned lkey[kFinishPairs];
    __shared__ int lidx[kFinishPairs];
    __shared__ unsigned wsum[16];
    __shared__ unsigned s_bin, s_above;
    const int t = threadIdx.x;
    const int n_words = (n_cand + 31) / 32;
    // the independent loads first (bitmap, level-1 histogram, list length),
    // so their latencies overlap; then the list, once
    const unsigned np = need0 ? *list_n : 0;
    if (need0)
        for (int i = t; i < kBins; i += 1024) hist[i] = hist1[i];
    for (int i = t; i < n_words; i += 1024) {
        sel[i] = need0 ? bitmap[i] : 0;
        tie[i] = 0;
    }
    const bool in_lds = np <= (unsigned)kFinishPairs;
    if (in_lds)
        for (unsigned i = t; i < np; i += 1024) {
            lkey[i] = list_key[i];
            lidx[i] = list_idx[i];
        }
    __syncthreads();
    const unsigned *keys_l = in_lds ? lkey : list_key;
    const int *idx_l = in_lds ? lidx : list_idx;
    // the bin of histogram h (nb bins, high bin = larger keys) that holds the
    // need-th largest key, and the count above it (thread t owns nb / 1024
    // bins from the top)
    auto find = [&](const unsigned *h, int nb, unsigned need) {
        const int per = nb / 1024;
        unsigned v = 0;
        for (int i = 0; i < per; ++i) v += h[nb - 1 - t * per - i];
        unsigned tot;
        const unsigned ex = scan1024_excl(v, wsum, &tot);
        if (ex < need && ex + v >= need) {
            unsigned run = ex;
            int b = nb - 1 - t * per;
            for (int i = 0; i < per - 1; ++i, --b) {
                if (run + h[b] >= need) break;
                run += h[b];
            }
            s_bin = (unsigned)b;
            s_above = run;
        }
        __syncthreads();
    };
    const int wpt = (n_words + 1023) / 1024;   // thread t owns words [t * wpt, (t + 1) * wpt)
    const int w0 = t * wpt, w1 = min(w0 + wpt, n_words);
    if (need0 > 0) {
        find(hist, kBins, need0);
        const unsigned b1 = s_bin;
        unsigned need = need0 - s_above;
        unsigned pref = b1 << 21, pmask = 0xFFE00000u;
        for (int lvl = 0; lvl < 2; ++lvl) {
            const int shift = lvl == 0 ? 10 : 0, nb = lvl == 0 ? kBins : 1024;
            __syncthreads();   // the previous level's readers of s_bin are done
            for (int i = t; i < nb; i += 1024) hist[i] = 0;
            __syncthreads();
            for (unsigned i = t; i < np; i += 1024) {
                const unsigned k = keys_l[i];
                if ((k & pmask) == pref) atomicAdd(&hist[(k >> shift) & (nb - 1)], 1u);
            }
            __syncthreads();
            find(hist, nb, need);
            pref |= s_bin << shift;
            pmask |= (unsigned)(nb - 1) << shift;
            need -= s_above;
        }
        const unsigned T = pref, need_eq = need;
        for (unsigned i = t; i < np; i += 1024) {
            const unsigned k = keys_l[i];
            const int c = idx_l[i];
            if (k > T) atomicOr(&sel[c >> 5], 1u << (c & 31));
            else if (k == T) atomicOr(&tie[c >> 5], 1u << (c & 31));
        }
        __syncthreads();
        // the need_eq ties of lowest index
        unsigned nt = 0;
        for (int w = w0; w < w1; ++w) nt += __popc(tie[w]);
        unsigned tot;
        unsigned rank = scan1024_excl(nt, wsum, &tot);
        for (int w = w0; w < w1; ++w) {
            unsigned bits = tie[w], add = 0;
            while (bits && rank < need_eq) {
                const unsigned low = bits & (0u - bits);
                add |= low;
                bits ^= low;
                ++rank;
            }
            sel[w] |= add;   // this thread's words only
        }
        __syncthreads();
    }
    unsigned ns = 0;
    for (int w = w0; w < w1; ++w) ns += __popc(sel[w]);
    unsigned tot;
    unsigned o = scan1024_excl(ns, wsum, &tot);
    for (int w = w0; w < w1; ++w) {
        unsigned bits = sel[w];
        if (mask)
            for (int b = 0; b < 32 && w * 32 + b < n_cand; ++b) mask[w * 32 + b] = (bits >> b) & 1u;
        if (pos_out)
            while (bits) {
                const int b = __builtin_ctz(bits);
                bits &= bits - 1;
                pos_out[o++] = w * 32 + b;
            }
    }
    for (int i = t; i < n_comp - n_cand; i += 1024) {
        if (pos_out) pos_out[need0 + i] = n_cand + i;
        if (mask) mask[n_cand + i] = 1;
    }
}

// scratch: [hist1 kBins][list_n 1][bitmap words][list keys n_cand][list idx n_cand] (u32)
size_t select_large_scratch_words(int n_comp) {
    const size_t n = (size_t)(n_comp > 0 ? n_comp : 1);
    return kBins + 1 + (n + 31) / 32 + 2 * n;
}

int launch_select_large(const float *scores, int n_comp, int n_cand, unsigned need0, unsigned *scratch,
                        int32_t *mask, int32_t *pos_out, hipStream_t st) {
    unsigned *hist1 = scratch, *list_n = scratch + kBins, *bitmap = list_n + 1;
    const int n_words = (n_cand + 31) / 32;
    unsigned *list_key = bitmap + n_words;
    int *list_idx = reinterpret_cast<int *>(list_key + n_cand);
    hipLaunchKernelGGL(compact_kernel, dim3((n_cand + kChunk - 1) / kChunk), dim3(256), 0, st, scores, n_cand,
                       need0, hist1, bitmap, list_n, list_key, list_idx);
    hipLaunchKernelGGL(finish_kernel, dim3(1), dim3(1024), 0, st, n_comp, n_cand, need0, hist1, bitmap, list_n,
                       list_key, list_idx, mask, pos_out);
    return hip_status(hipGetLastError());
}

}  // namespace

extern "C" int ds4hip_indexer_topk_positions_batch(
        const float *q, const float *weights, const void *keys, int key_kind,
        const long long *key_row0_host, const int *n_comp_host, int n_seq, int n_head,
        int head_dim, int top_k, int n_recent, float *scratch_scores, int32_t *positions_out,
        int pos_stride, void *stream) {
    if (!q || !weights || !keys || !key_row0_host || !n_comp_host || !scratch_scores ||
        !positions_out || key_kind < 0 || key_kind > 2 || n_seq <= 0 || n_seq > kMaxSeq ||
        n_head <= 0 || n_head > kMaxHeads || head_dim != kMaxDim || top_k <= 0 || n_recent < 0 ||
        pos_stride < top_k)
        return ds4hip_set_last_error(kEINVAL);
    BatchArgs A;
    A.q = q;
    A.w = weights;
    A.keys = keys;
    A.scores = scratch_scores;
    A.pos_out = positions_out;
    A.n_seq = n_seq;
    A.n_head = n_head;
    A.top_k = top_k;
    A.n_recent = n_recent;
    A.pos_stride = pos_stride;
    long long n_scored = 0;
    for (int s = 0; s < n_seq; ++s)
        if (n_comp_host[s] > top_k) n_scored += n_comp_host[s];
    const int keys_per_blk = A.keys_per_blk = score_keys_per_block(n_scored);
    int blk = 0;
    for (int s = 0; s < kMaxSeq; ++s) {
        const int n = s < n_seq ? n_comp_host[s] : 0;
        if (n < 0 || (n > top_k && n - (n_recent < top_k ? n_recent : top_k) > kSelMax))
            return ds4hip_set_last_error(kEINVAL);
        A.n_comp[s] = n;
        A.key0[s] = s < n_seq ? key_row0_host[s] : 0;
        A.blk0[s] = blk;
        // only sequences that need a selection are scored
        if (s < n_seq && n > top_k) blk += (n + keys_per_blk - 1) / keys_per_blk;
    }
    A.blk0[kMaxSeq] = blk;
    const hipStream_t st = (hipStream_t)stream;
    if (blk > 0) {
        const dim3 g(blk), b(256);
        switch (key_kind) {
        case 0:
            hipLaunchKernelGGL(score_batch_kernel<0>, g, b, 0, st, A);
            break;
        case 1:
            hipLaunchKernelGGL(score_batch_kernel<1>, g, b, 0, st, A);
            break;
        default:
            hipLaunchKernelGGL(score_batch_kernel<2>, g, b, 0, st, A);
            break;
        }
    }
    hipLaunchKernelGGL(select_batch_kernel, dim3(n_seq), dim3(1024), 0, st, A);
    return ds4hip_set_last_error(hip_status(hipGetLastError()));
}

int ds4hip_indexer_chunk_max_keys() { return kSelMax; }

int ds4hip_indexer_chunk_topk(const float *q, const float *weights, const float *keys, int n_tok, int p0, int ratio,
                              int n_keys0, int n_head, int top_k, float *scores, int score_stride,
                              int32_t *positions, hipStream_t st) {
    ChunkSelArgs A{q, weights, keys, scores, positions, n_head, top_k, score_stride, 0, n_keys0, p0, ratio};
    const int n_last = n_keys0 + (p0 + n_tok) / ratio - p0 / ratio;
    if (n_last <= top_k) return 0;
    if (n_last > kSelMax || n_last > score_stride) return kEINVAL;
    A.keys_per_blk = score_keys_per_block((long long)n_last * n_tok);
    hipLaunchKernelGGL(score_chunk_kernel, dim3((n_last + A.keys_per_blk - 1) / A.keys_per_blk, n_tok), dim3(256), 0,
                       st, A);
    hipLaunchKernelGGL(select_chunk_kernel, dim3(n_tok), dim3(1024), 0, st, A);
    return hip_status(hipGetLastError());
}
