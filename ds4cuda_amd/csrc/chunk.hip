// chunk.hip — Step 12 of a prompt chunk (up to 128 tokens of one layer) over
// the FP8 session: compressors, emitted rows, indexer query and selection for
// all tokens in a few launches, with the results of the token-by-token loop
// (cuda/forward_batch.cu:264-284) bit for bit.
//
// The only values that carry from one token to the next are the compressor's
// state rows, and those are projections of the tokens themselves. So:
//   project: every token's projections (kv, gate, their indexer forms, the
//            indexer query and head weights);
//   emit:    every window that closes inside the chunk, its rows taken from
//            the projections or, for tokens before the chunk, from the state;
//   finish:  the state rows as the last token leaves them, the indexer
//            queries' RoPE;
//   then the FP8 push of the emitted rows, and the tokens' selections.

#include "comp_emit.h"
#include "ds4hip_common.h"
#include "rope.h"
#include "../../include/ds4hip.h"
#include "../../include/ds4hip_session.h"

#include <algorithm>

using namespace ds4hip;

namespace {

constexpr int kEmbd = 4096, kLora = 1024;       // inputs of the projections
constexpr int kIdxHeads = 64, kIdxDim = DS4HIP_INDEXER_HEAD_DIM;

// ---- projections -------------------------------------------------------------------------
//
// Y[t][r] = W[r] . x[t] (f16 W, fp32 x) with the sums of the one-token matvec
// (wave_rows_dot and the wave's butterfly): lane l of 64 runs an fma chain over
// the 8-element pieces l, l + 64, ... of the row, then xor offsets 32 .. 1 add
// the lanes. A 16x16x4 fp32 MFMA is four steps of such a chain for 16 rows x
// 16 tokens, so each of the 64 chains is an accumulator tile of its own, and
// the tiles are added with the butterfly's pairs.
//
// Wave w of a workgroup runs chains 4 u .. 4 u + 3 for u = w, w + 4, w + 8,
// w + 12: offsets 32 and 16 (u ^ 8, u ^ 4) stay inside the wave, offsets 8 and
// 4 (u ^ 2, u ^ 1) are waves w ^ 2 and w ^ 1, offsets 2 and 1 the four chains.
// Lane group g loads chain 4 u + g's piece; lane exchanges turn four such
// registers into the operands of the four chains.
//
// Bound by the fp32 matrix rate (15 ns per MFMA and SIMD; 2.4 M of them for
// 128 tokens of a ratio-4 layer with its indexer query: 35 us over the chip)
// and the L2 latency of the pieces that two waves per SIMD leave uncovered.
// Measured there: 98 us with 32 rows x 16 tokens a workgroup, 126 us with 16 x
// 16 (three waves per SIMD, half as much again from L2), 115 us with 16 x 32,
// 230 us with 32 x 32 (one wave per SIMD); one matvec launch per token and
// matrix took 21 us a token. Up to 16 tokens take 16 x 16, where twice the
// workgroups stream the weights; the line is a token tile's. Whole chunks with
// 32 and 16 rows: 16 tokens without a selection 68.0 and 66.7 us, with one 90.1
// and 92.3; 17 tokens 99.2 and 104.1, 64 tokens 141.7 and 149.9.

__device__ inline void lanes_to_steps(uint32_t (&v)[4]) {
    // lane group g holds v[i] of chain g; afterwards v[j] of group g is
    // element g of chain j: a 16x16x4 operand of chain j
    auto a = __builtin_amdgcn_permlane32_swap(v[0], v[2], false, false);
    auto b = __builtin_amdgcn_permlane32_swap(v[1], v[3], false, false);
    auto c = __builtin_amdgcn_permlane16_swap(a[0], b[0], false, false);
    auto d = __builtin_amdgcn_permlane16_swap(a[1], b[1], false, false);
    v[0] = c[0];
    v[1] = c[1];
    v[2] = d[0];
    v[3] = d[1];
}

struct ProjJob {
    const uint16_t *w;    // [rows][K] f16
    const float *x;       // [n][K]
    float *y;             // [n][ld]
    const uint16_t *ape;  // f16 [ratio][rows], added at the token's position, or NULL
    float scale;          // times the sum (1: none)
    int ld, k_is_lora;
};
constexpr int kMaxJobs = 6;
struct ProjArgs {
    ProjJob j[kMaxJobs];
    int blk0[kMaxJobs + 1];   // first row tile of each job, and their count
    int n, p0, ratio;
};

// A lane's raw pieces of one step of the pipeline: its row's eight f16 weights
// per row tile and its token's eight inputs.
template <int kR>
struct Pieces {
    uint4_t w[kR];
    float4_t x[2];
    __device__ inline void load(const uint16_t *const (&wp)[kR], const float *xp, bool x_wide, int e0) {
#pragma unroll
        for (int r = 0; r < kR; ++r) w[r] = *reinterpret_cast<const uint4_t *>(wp[r] + e0);
        const float *p = xp + e0;
#pragma unroll
        for (int h = 0; h < 2; ++h)
            x[h] = x_wide ? *reinterpret_cast<const float4_t *>(p + 4 * h)
                          : float4_t{p[4 * h], p[4 * h + 1], p[4 * h + 2], p[4 * h + 3]};
    }
};

// One wave's chains of a (16 kR) x 16 tile: kJ pieces per chain. sum[i]:
// chains i of its four groups added (offsets 32, 16). x_wide: x is 16-byte
// aligned (else four 4-byte loads). The pieces are loaded two steps ahead:
// with two waves per SIMD nothing else covers the L2 latency.
template <int kJ, int kR>
__device__ inline void chain_tiles(const uint16_t *const (&w)[kR], const float *x, bool x_wide, int wave,
                                   float4_t (&sum)[4][kR]) {
    static_assert(kJ % 2 == 0, "the two buffers alternate by piece");
    const int g = (threadIdx.x & 63) >> 4;
    // step q = kJ s + j: piece j of group s, groups in the order w, w + 8, w + 4, w + 12
    auto elem = [&](int q) {
        const int sq = (q / kJ) & 3, j = q % kJ;
        return (4 * (wave + ((sq & 1) << 3) + ((sq >> 1) << 2)) + g + 64 * j) * 8;
    };
    float4_t half[4][kR];
    Pieces<kR> buf[2];
    buf[0].load(w, x, x_wide, elem(0));
    buf[1].load(w, x, x_wide, elem(1));
#pragma unroll 1
    for (int s = 0; s < 4; ++s) {
        float4_t acc[4][kR];
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int r = 0; r < kR; ++r) acc[i][r] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int j = 0; j < kJ; ++j) {
            Pieces<kR> &cur = buf[j & 1];
            uint32_t a[kR][2][4], b[2][4];
#pragma unroll
            for (int r = 0; r < kR; ++r)
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    a[r][e >> 2][e & 3] =
                        __float_as_uint(f16_bits_to_f32((uint16_t)((cur.w[r][e >> 1] >> (16 * (e & 1))) & 0xFFFF)));
#pragma unroll
            for (int e = 0; e < 8; ++e) b[e >> 2][e & 3] = __float_as_uint(cur.x[e >> 2][e & 3]);
            cur.load(w, x, x_wide, elem(kJ * s + j + 2));   // past the last step: group 0 again, unused
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int h = 0; h < 2; ++h) {
#pragma unroll
                for (int r = 0; r < kR; ++r) lanes_to_steps(a[r][h]);
                lanes_to_steps(b[h]);
#pragma unroll
                for (int r = 0; r < kR; ++r)
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        acc[i][r] = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(a[r][h][i]),
                                                                         __uint_as_float(b[h][i]), acc[i][r], 0, 0, 0);
            }
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int r = 0; r < kR; ++r) {
                if (s == 0) sum[i][r] = acc[i][r];
                if (s == 1) sum[i][r] = sum[i][r] + acc[i][r];
                if (s == 2) half[i][r] = acc[i][r];
                if (s == 3) sum[i][r] = sum[i][r] + (half[i][r] + acc[i][r]);
            }
    }
}

template <int kR>
__global__ __launch_bounds__(256, 2) void chunk_project_kernel(const ProjArgs A) {
    __shared__ float red[4][4][kR][4][64];   // [wave][chain][row tile][register][lane]
    // the token tiles of a row tile run on one XCD (workgroups go to the eight
    // in turn), so its L2 reads those weights once: 107 -> 98 us for 128 tokens
    const int tok_tiles = (A.n + 15) / 16;
    const int row_tile = (int)blockIdx.x / (8 * tok_tiles) * 8 + (int)blockIdx.x % 8;
    if (row_tile >= A.blk0[kMaxJobs]) return;
    int jb = 0;
#pragma unroll
    for (int i = 1; i < kMaxJobs; ++i)
        if (row_tile >= A.blk0[i]) jb = i;
    const ProjJob J = A.j[jb];
    const int K = J.k_is_lora ? kLora : kEmbd;
    const int row0 = (row_tile - A.blk0[jb]) * 16 * kR, tok0 = (int)blockIdx.x / 8 % tok_tiles * 16;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint16_t *w[kR];
#pragma unroll
    for (int r = 0; r < kR; ++r) w[r] = J.w + (size_t)(row0 + 16 * r + (lane & 15)) * K;
    const float *x = J.x + (size_t)min(tok0 + (lane & 15), A.n - 1) * K;
    float4_t sum[4][kR];
    const bool wide = (reinterpret_cast<uintptr_t>(J.x) & 15) == 0;
    if (J.k_is_lora) chain_tiles<kLora / 512, kR>(w, x, wide, wave, sum);
    else chain_tiles<kEmbd / 512, kR>(w, x, wide, wave, sum);
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int r = 0; r < kR; ++r)
#pragma unroll
            for (int e = 0; e < 4; ++e) red[wave][i][r][e][lane] = sum[i][r][e];
    __syncthreads();
    // wave `wave` finishes register `wave` of every row tile: row 4 (lane / 16) +
    // wave, token lane % 16
    const int tok = tok0 + (lane & 15);
#pragma unroll
    for (int r = 0; r < kR; ++r) {
        float c[4];
#pragma unroll
        for (int i = 0; i < 4; ++i)
            c[i] = (red[0][i][r][wave][lane] + red[2][i][r][wave][lane]) +
                   (red[1][i][r][wave][lane] + red[3][i][r][wave][lane]);
        float v = (c[0] + c[2]) + (c[1] + c[3]);
        const int row = row0 + 16 * r + 4 * (lane >> 4) + wave;
        if (tok >= A.n) continue;
        if (J.ape) v = v + f16_bits_to_f32(J.ape[(size_t)((A.p0 + tok) % A.ratio) * J.ld + row]);
        if (J.scale != 1.0f) v = v * J.scale;
        J.y[(size_t)tok * J.ld + row] = v;
    }
}

// ---- emitted rows and states ---------------------------------------------------------------

struct CompJob {
    const float *kv, *score;       // projections [n][width], the score with its APE row
    float *state_kv, *state_score;
    const float *w_norm;
    float *emit;                   // emitted rows [n_emit][head_dim]
    int head_dim, width, is_attn;
};
struct EmitArgs {
    CompJob j[2];
    int n, p0, ratio, n_emit, n_jobs;
    RopeArgs rope;
};

// Window `win` (positions [ratio win, ratio win + ratio)) as the state holds it
// when it closes: rows of the chunk's tokens from the projections, earlier
// ones from the state at the chunk's start, whose rows 4 .. 7 (ratio 4) hold
// the window of position p0 and rows 0 .. 3 the one before.
struct ChunkSrc {
    const CompJob &J;
    int p0, ratio, win;
    __device__ inline size_t at(int r, bool &chunk) const {
        const int rr = ratio == 4 ? (r & 3) : r;
        const int of = ratio == 4 && r < 4 ? win - 1 : win;
        const int pos = of * ratio + rr;
        chunk = pos >= p0;
        if (chunk) return (size_t)(pos - p0) * J.width;
        return (size_t)(ratio == 4 ? (of == p0 / 4 ? 4 + rr : rr) : r) * J.width;
    }
    __device__ inline float kv(int r, int c) const {
        bool chunk;
        const size_t o = at(r, chunk);
        return (chunk ? J.kv : J.state_kv)[o + c];
    }
    __device__ inline float score(int r, int c) const {
        bool chunk;
        const size_t o = at(r, chunk);
        return (chunk ? J.score : J.state_score)[o + c];
    }
};

// Workgroup (m, job): the m-th window that closes in the chunk.
__global__ __launch_bounds__(512) void chunk_emit_kernel(const EmitArgs A) {
    const CompJob &J = A.j[blockIdx.y];
    const int win = A.p0 / A.ratio + (int)blockIdx.x;
    RopeArgs R = A.rope;
    R.pos = win * A.ratio;
    emit_row(ChunkSrc{J, A.p0, A.ratio, win}, J.w_norm, J.emit + (size_t)blockIdx.x * J.head_dim, J.head_dim, A.ratio,
             J.is_attn, R);
}

// The state rows the chunk's tokens leave. Ratio 128: each of the at most 128
// tokens has a row of its own (element i of the n rows). Ratio 4, column i: a
// token's row at its position's place, and once a window has closed, its rows
// (4 .. 7) copied to 0 .. 3.
__device__ inline void finish_state(const CompJob &J, int n, int p0, int ratio, int n_emit, int i) {
    if (ratio != 4) {
        const size_t o = (size_t)((p0 + i / J.width) % ratio) * J.width + i % J.width;
        J.state_kv[o] = J.kv[i];
        J.state_score[o] = J.score[i];
        return;
    }
    const int c = i;
    const int last = p0 + n - 1, closed = p0 / 4 + n_emit - 1;   // the last window that closed
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const size_t lo = (size_t)r * J.width + c, hi = (size_t)(4 + r) * J.width + c;
        if (n_emit) {
            const int pos = 4 * closed + r;
            const size_t o = (size_t)(pos - p0) * J.width + c;
            const float kv = pos >= p0 ? J.kv[o] : J.state_kv[hi];
            const float sc = pos >= p0 ? J.score[o] : J.state_score[hi];
            J.state_kv[lo] = kv;
            J.state_score[lo] = sc;
        }
        const int pos = last - ((last - r) & 3);   // the last position with this row
        if (pos >= p0) {
            const size_t o = (size_t)(pos - p0) * J.width + c;
            J.state_kv[hi] = J.kv[o];
            J.state_score[hi] = J.score[o];
        }
    }
}

// Workgroups [0, state_blks): state columns; the rest: the indexer queries'
// forward tail RoPE, a pair per thread.
struct FinishArgs {
    EmitArgs e;
    float *q_idx;             // [n][heads * 128], NULL: no RoPE
    RopeParams rope;
    int col_blk1, state_blks; // first workgroup of job 1, workgroups of both
};
__global__ __launch_bounds__(256) void chunk_finish_kernel(const FinishArgs A) {
    if ((int)blockIdx.x < A.state_blks) {
        const int jb = (int)blockIdx.x >= A.col_blk1 ? 1 : 0;
        const CompJob &J = A.e.j[jb];
        const int c = ((int)blockIdx.x - (jb ? A.col_blk1 : 0)) * 256 + (int)threadIdx.x;
        if (c < (A.e.ratio == 4 ? 1 : A.e.n) * J.width) finish_state(J, A.e.n, A.e.p0, A.e.ratio, A.e.n_emit, c);
        return;
    }
    constexpr int kHalf = kNRot / 2;
    const int i = ((int)blockIdx.x - A.state_blks) * 256 + (int)threadIdx.x;
    const int head = i / kHalf, t = i % kHalf, tok = head / kIdxHeads;
    if (tok >= A.e.n) return;
    float *x = A.q_idx + (size_t)head * kIdxDim + (kIdxDim - kNRot) + 2 * t;
    float y0, y1;
    rope_pair(x[0], x[1], t, A.e.p0 + tok, A.rope, y0, y1);
    x[0] = y0;
    x[1] = y1;
}

// ---- the step's scratch ----------------------------------------------------------------------

size_t up256(size_t b) { return (b + 255) & ~(size_t)255; }

struct ChunkWs {
    float *kv, *score, *ikv, *iscore, *emit, *q_idx, *w_idx, *scores;
    uint8_t *select;
    int score_stride;
    size_t bytes;
};
// cap_keys: the layer's indexer capacity (0: no indexer)
ChunkWs chunk_ws(void *base, int n, int ratio, int cap_keys) {
    ChunkWs W{};
    size_t off = 0;
    auto take = [&](size_t floats) {
        float *p = base ? reinterpret_cast<float *>(static_cast<uint8_t *>(base) + off) : nullptr;
        off += up256(floats * 4);
        return p;
    };
    const int width = (ratio == 4 ? 2 : 1) * DS4HIP_HEAD_DIM;
    W.kv = take((size_t)n * width);
    W.score = take((size_t)n * width);
    W.emit = take((size_t)(n / ratio + 1) * DS4HIP_HEAD_DIM);
    if (cap_keys > 0) {
        W.ikv = take((size_t)n * 2 * kIdxDim);
        W.iscore = take((size_t)n * 2 * kIdxDim);
        W.q_idx = take((size_t)n * kIdxHeads * kIdxDim);
        W.w_idx = take((size_t)n * kIdxHeads);
        // tokens past the chunk selection's key limit select one by one, with
        // the same scratch (in stream order) for their scores
        W.score_stride = (std::min(cap_keys, ds4hip_indexer_chunk_max_keys()) + 63) & ~63;
        W.scores = take(std::max((size_t)n * W.score_stride, (size_t)cap_keys));
        if (cap_keys > ds4hip_indexer_chunk_max_keys())
            W.select = reinterpret_cast<uint8_t *>(take(ds4hip_indexer_select_scratch_bytes(cap_keys) / 4 + 1));
    }
    W.bytes = off;
    return W;
}

template <int kR>
void launch_project(const ProjArgs &A, int blocks, hipStream_t st) {
    hipLaunchKernelGGL(chunk_project_kernel<kR>, dim3((blocks + 7) / 8 * 8 * ((A.n + 15) / 16)), dim3(256), 0, st, A);
}

int chunk_step(ds4hip_session_state *s, int il, int p0, int n, const float *attn_norm, const float *q_lora,
               const ds4hip_chunk_layer *w, int32_t *sel, int *n_comp_tok, int *n_sel_tok, void *ws, size_t ws_bytes,
               hipStream_t st) {
    if (!s || !s->arena_base || il < 0 || il >= DS4HIP_N_LAYER || n <= 0 || n > DS4HIP_CHUNK_MAX || p0 < 0 ||
        !n_comp_tok || !n_sel_tok || !attn_norm || !w || !ws)
        return kEINVAL;
    ds4hip_layer_state *L = &s->layers[il];
    const int ratio = L->compress_ratio;
    const bool idx = L->has_indexer;
    if (!ratio || !w->comp_kv || !w->comp_gate || !w->comp_ape || !w->comp_norm) return kEINVAL;
    if (idx && (!w->idx_kv || !w->idx_gate || !w->idx_ape || !w->idx_norm || w->top_k <= 0)) return kEINVAL;
    const int n_emit = (p0 + n) / ratio - p0 / ratio;
    if (L->n_comp + n_emit > L->cap_comp || (idx && L->n_index_comp + n_emit > L->cap_comp)) return DS4HIP_ENOSPC;
    const bool select = idx && L->n_index_comp + n_emit > w->top_k;
    if (select && (!q_lora || !w->idx_q_b || !w->idx_proj || !sel)) return kEINVAL;
    const ChunkWs W = chunk_ws(ws, n, ratio, idx ? L->cap_comp : 0);
    if (ws_bytes < W.bytes) return kEINVAL;

    ProjArgs P{};
    P.n = n;
    P.p0 = p0;
    P.ratio = ratio;
    const int width = (ratio == 4 ? 2 : 1) * DS4HIP_HEAD_DIM;
    const bool big = n > 16;
    const int rows_blk = big ? 32 : 16;
    int jobs = 0, blk = 0;
    auto job = [&](const uint16_t *wt, const float *x, float *y, const uint16_t *ape, float scale, int rows, int lora) {
        P.j[jobs] = ProjJob{wt, x, y, ape, scale, rows, lora};
        P.blk0[jobs++] = blk;
        blk += rows / rows_blk;
    };
    job(w->comp_kv, attn_norm, W.kv, nullptr, 1.0f, width, 0);
    job(w->comp_gate, attn_norm, W.score, w->comp_ape, 1.0f, width, 0);
    if (idx) {
        job(w->idx_kv, attn_norm, W.ikv, nullptr, 1.0f, 2 * kIdxDim, 0);
        job(w->idx_gate, attn_norm, W.iscore, w->idx_ape, 1.0f, 2 * kIdxDim, 0);
    }
    if (select) {
        job(w->idx_proj, attn_norm, W.w_idx, nullptr, (float)(1.0 / sqrt((double)(kIdxDim * kIdxHeads))), kIdxHeads, 0);
        job(w->idx_q_b, q_lora, W.q_idx, nullptr, 1.0f, kIdxHeads * kIdxDim, 1);
    }
    for (int i = jobs; i <= kMaxJobs; ++i) P.blk0[i] = blk;
    if (big) launch_project<2>(P, blk, st);
    else launch_project<1>(P, blk, st);
    int rc = hip_status(hipGetLastError());
    if (rc) return rc;

    FinishArgs F{};
    EmitArgs &E = F.e;
    E.n = n;
    E.p0 = p0;
    E.ratio = ratio;
    E.n_emit = n_emit;
    E.n_jobs = idx ? 2 : 1;
    E.rope = rope_args(il, 0);
    E.j[0] = CompJob{W.kv, W.score, L->attn_state_kv, L->attn_state_score, w->comp_norm, W.emit, DS4HIP_HEAD_DIM, width, 1};
    if (idx)   // the keys go straight to the session's key rows
        E.j[1] = CompJob{W.ikv, W.iscore, L->index_state_kv, L->index_state_score, w->idx_norm,
                         L->index_comp_kv + (size_t)L->n_index_comp * kIdxDim, kIdxDim, 2 * kIdxDim, 0};
    if (n_emit) {
        hipLaunchKernelGGL(chunk_emit_kernel, dim3(n_emit, E.n_jobs), dim3(512), 0, st, E);
        if ((rc = hip_status(hipGetLastError()))) return rc;
    }
    F.col_blk1 = ((ratio == 4 ? 1 : n) * width + 255) / 256;
    F.state_blks = F.col_blk1 + (idx ? (2 * kIdxDim + 255) / 256 : 0);
    int blocks = F.state_blks;
    if (select) {
        F.q_idx = W.q_idx;
        F.rope = rope_params(kNRot, il, false);
        blocks += (n * kIdxHeads * (kNRot / 2) + 255) / 256;
    }
    hipLaunchKernelGGL(chunk_finish_kernel, dim3(blocks), dim3(256), 0, st, F);
    if ((rc = hip_status(hipGetLastError()))) return rc;
    if (n_emit &&
        (rc = ds4hip_fp8_kv_quantize_append(W.emit, n_emit, DS4HIP_HEAD_DIM, DS4HIP_N_ROT, s->codes, s->sexp, s->tail,
                                            L->row_base + L->n_comp, nullptr, st)))
        return rc;
    const int n_idx0 = L->n_index_comp;
    auto keys_of = [&](int t) { return n_idx0 + (p0 + t + 1) / ratio - p0 / ratio; };
    for (int t = 0; t < n; ++t) {
        n_comp_tok[t] = n_sel_tok[t] = L->n_comp + (p0 + t + 1) / ratio - p0 / ratio;
        if (idx && keys_of(t) > w->top_k) n_sel_tok[t] = w->top_k;
    }
    if (select) {
        // the keys a token sees, not those the session could hold, decide its form
        int together = 0;
        while (together < n && keys_of(together) <= ds4hip_indexer_chunk_max_keys()) ++together;
        if (together)
            rc = ds4hip_indexer_chunk_topk(W.q_idx, W.w_idx, L->index_comp_kv, together, p0, ratio, n_idx0, kIdxHeads,
                                           w->top_k, W.scores, W.score_stride, sel, st);
        for (int t = together; t < n && !rc; ++t)
            if (keys_of(t) > w->top_k)
                rc = ds4hip_indexer_topk_positions(W.q_idx + (size_t)t * kIdxHeads * kIdxDim, W.w_idx + (size_t)t * kIdxHeads,
                                                   L->index_comp_kv, 0, keys_of(t), kIdxHeads, kIdxDim, w->top_k, 0,
                                                   W.scores, W.select, nullptr, sel + (size_t)t * w->top_k, st);
    }
    if (rc) return rc;
    L->n_comp += n_emit;
    if (idx) L->n_index_comp += n_emit;
    return 0;
}

}  // namespace

extern "C" size_t ds4hip_session_chunk_step_workspace_bytes(const ds4hip_session_state *s, int il, int n_tok) {
    if (!s || il < 0 || il >= DS4HIP_N_LAYER || n_tok <= 0 || n_tok > DS4HIP_CHUNK_MAX) return 0;
    const ds4hip_layer_state *L = &s->layers[il];
    if (!L->compress_ratio) return 0;
    return chunk_ws(nullptr, n_tok, L->compress_ratio, L->has_indexer ? L->cap_comp : 0).bytes;
}

extern "C" int ds4hip_session_chunk_step(ds4hip_session_state *s, int il, int p0, int n_tok, const float *attn_norm,
                                         const float *q_lora_norm, const ds4hip_chunk_layer *w, int32_t *sel,
                                         int *n_comp_tok, int *n_sel_tok, void *workspace, size_t workspace_bytes,
                                         void *stream) {
    return ds4hip_set_last_error(chunk_step(s, il, p0, n_tok, attn_norm, q_lora_norm, w, sel, n_comp_tok, n_sel_tok,
                                            workspace, workspace_bytes, (hipStream_t)stream));
}

extern "C" int ds4hip_session_push_raw_rows(ds4hip_session_state *s, int il, const float *kv, int n_rows,
                                            void *stream) {
    if (!s || !s->arena_base || il < 0 || il >= DS4HIP_N_LAYER || !kv || n_rows < 0 || n_rows > s->layers[il].cap_raw)
        return ds4hip_set_last_error(kEINVAL);
    ds4hip_layer_state *L = &s->layers[il];
    const int first = std::min(n_rows, L->cap_raw - L->raw_head);   // rows before the ring wraps
    const long long ring = L->row_base + L->cap_comp;
    int rc = first ? ds4hip_fp8_kv_quantize_append(kv, first, DS4HIP_HEAD_DIM, DS4HIP_N_ROT, s->codes, s->sexp, s->tail,
                                                   ring + L->raw_head, nullptr, stream)
                   : 0;
    if (!rc && n_rows > first)
        rc = ds4hip_fp8_kv_quantize_append(kv + (size_t)first * DS4HIP_HEAD_DIM, n_rows - first, DS4HIP_HEAD_DIM,
                                           DS4HIP_N_ROT, s->codes, s->sexp, s->tail, ring, nullptr, stream);
    if (rc) return rc;
    L->raw_head = (L->raw_head + n_rows) % L->cap_raw;
    L->n_raw = std::min(L->n_raw + n_rows, L->cap_raw);
    return 0;
}
