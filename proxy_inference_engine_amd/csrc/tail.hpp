// tail.hpp -- the end of _inference (engine/inference_engine.py:254,268-271) with the greedy sampler
// (samplers/__init__.py:37-38): logprobs = f32(logits) - logsumexp(f32(logits)); token = first argmax.
//
// Behind the lm_head GEMV, whose epilogue (EPI_LOGITS) leaves per-wave (max, sum exp(x - max), first argmax) partials: k_logits_finish, in which every workgroup merges
// the partials (a few thousand, L2-resident) and writes its slice of the fp32 logprobs.  Behind any other product: k_logits_rows, one launch or, behind k_logits_tiles, two (logits_row.hpp).
#pragma once
#include "common.hpp"
#include "logits_row.hpp"
#include "w4_gemv.hpp"  // LogitStat, DecState

constexpr int TAIL_FINISH_BLOCKS = 64;

// whole rows at once, grid (rows, parts); tiles (nullable): what k_logits_tiles left of them.  lens (nullable): the rows' context lengths, moved on by the token that this step appended
template <class T>
__global__ void __launch_bounds__(LOGITS_ROW_THREADS) k_logits_rows(const u16 *logits, int V, const RowStat *tiles, float *logprobs, int *tokens, int *lens) {
    const size_t at = (size_t)blockIdx.x * V;
    float lse;
    int token;
    logits_row_stats<T>(logits + at, V, tiles ? tiles + (size_t)blockIdx.x * LOGITS_TILES : nullptr, lse, token);
    logits_row_write<T>(logits + at, V, lse, blockIdx.y, gridDim.y, logprobs + at);
    if (blockIdx.y == 0 && threadIdx.x == 0) {
        tokens[blockIdx.x] = token;
        if (lens && lens[blockIdx.x] > 0) ++lens[blockIdx.x];
    }
}

constexpr int TAIL_MAX_STATS = 4096;  // 256 threads x 16 register-resident partials

template <class T>
__global__ void __launch_bounds__(256) k_logits_finish(const u16 *logits, int V, const LogitStat *stats, int n_stats, float *logprobs,
                                                       int *token, DecState *state, int *history, int hist_cap, const unsigned *err_word, int *lens) {
    __shared__ float s_max[4], s_sum[4];
    __shared__ int s_arg[4];
    logits += (size_t)blockIdx.y * V, stats += (size_t)blockIdx.y * n_stats, logprobs += (size_t)blockIdx.y * V, token += blockIdx.y;  // batch row
    // every workgroup merges all partials: 16 independent 16-byte loads per thread, then two register passes
    LogitStat st[16];
#pragma unroll
    for (int k = 0; k < 16; ++k) {
        const int i = threadIdx.x + 256 * k;
        const uint4 raw = *reinterpret_cast<const uint4 *>(stats + (i < n_stats ? i : n_stats - 1));
        st[k].max = i < n_stats ? __builtin_bit_cast(float, raw.x) : -INFINITY;
        st[k].sumexp = i < n_stats ? __builtin_bit_cast(float, raw.y) : 0.0f;
        st[k].argmax = i < n_stats ? (int)raw.z : 0x7fffffff;
    }
    float mx = -INFINITY;
    int arg = 0x7fffffff;
#pragma unroll
    for (int k = 0; k < 16; ++k)
        if (st[k].max > mx || (st[k].max == mx && st[k].argmax < arg)) mx = st[k].max, arg = st[k].argmax;
    const float wmax = wave_max(mx);
    int cand = (mx == wmax) ? arg : 0x7fffffff;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) cand = min(cand, __shfl_xor(cand, o, 64));
    const int wave = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) s_max[wave] = wmax, s_arg[wave] = cand;
    __syncthreads();
    float M = s_max[0];
    int tok = s_arg[0];
#pragma unroll
    for (int w = 1; w < 4; ++w)
        if (s_max[w] > M || (s_max[w] == M && s_arg[w] < tok)) M = s_max[w], tok = s_arg[w];
    float se = 0.0f;
#pragma unroll
    for (int k = 0; k < 16; ++k) se += st[k].sumexp > 0.0f ? st[k].sumexp * expf(st[k].max - M) : 0.0f;
    se = wave_sum(se);
    if ((threadIdx.x & 63) == 0) s_sum[wave] = se;
    __syncthreads();
    const float lse = M + logf((s_sum[0] + s_sum[1]) + (s_sum[2] + s_sum[3]));
    const int slice = (((V + gridDim.x - 1) / gridDim.x) + 7) & ~7;  // 8 logits per thread and pass
    const int begin = blockIdx.x * slice, end = min(V, begin + slice);
    for (int i = begin + threadIdx.x * 8; i < end; i += 256 * 8) {
        if (i + 8 <= end && (V & 7) == 0) {
            const uint4 v = *reinterpret_cast<const uint4 *>(logits + i);
            float4 o0 = make_float4(lo_f32<T>(v.x) - lse, hi_f32<T>(v.x) - lse, lo_f32<T>(v.y) - lse, hi_f32<T>(v.y) - lse);
            float4 o1 = make_float4(lo_f32<T>(v.z) - lse, hi_f32<T>(v.z) - lse, lo_f32<T>(v.w) - lse, hi_f32<T>(v.w) - lse);
            *reinterpret_cast<float4 *>(logprobs + i) = o0;
            *reinterpret_cast<float4 *>(logprobs + i + 4) = o1;
        } else {
            for (int k = i; k < min(i + 8, end); ++k) logprobs[k] = T::to_f32(logits[k]) - lse;
        }
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        if (err_word && *err_word != 0u) tok = -1;  // the persistent launch gave up a bounded wait (sticky): no plausible-looking id from garbage
        *token = tok;
        if (lens && lens[blockIdx.y] > 0) ++lens[blockIdx.y];  // (batch rows: k_logits_rows)
        if (state) {
            const int next_pos = state->pos + 1;  // the position the chosen token will occupy
            if (history && next_pos < hist_cap) history[next_pos] = tok;  // device-side token history (PromptCache.computed_ids)
            state->token = tok;   // greedy auto-feed of the next step
            state->pos = next_pos;  // cache.offset += 1 (reusable.py:139)
        }
    }
}

// `rows` logit vectors [rows, V] at once (the multi-sequence decode step, the op-level API).  tiles: LOGITS_TILES a row of scratch, needed where logits_in_tiles says so (nullptr: not in tiles)
static inline int logits_tail_rows_launch(int dtype, const u16 *logits, int V, int rows, RowStat *tiles, float *logprobs, int *tokens, hipStream_t st, int *lens = nullptr) {
    if (dtype != PIE_BF16 && dtype != PIE_F16) return pie::fail(PIE_E_ARG, "logits tail: dtype must be PIE_BF16 or PIE_F16");
    if (tiles) {
        const dim3 gt(LOGITS_TILES, rows);
        if (dtype == PIE_BF16) hipLaunchKernelGGL((k_logits_tiles<BF16, u16>), gt, dim3(LOGITS_TILE_THREADS), 0, st, logits, V, tiles);
        else hipLaunchKernelGGL((k_logits_tiles<F16, u16>), gt, dim3(LOGITS_TILE_THREADS), 0, st, logits, V, tiles);
        PIE_LAUNCH_CHECK();
    }
    const dim3 g(rows, logits_row_parts(rows));
    if (dtype == PIE_BF16) hipLaunchKernelGGL(k_logits_rows<BF16>, g, dim3(LOGITS_ROW_THREADS), 0, st, logits, V, tiles, logprobs, tokens, lens);
    else hipLaunchKernelGGL(k_logits_rows<F16>, g, dim3(LOGITS_ROW_THREADS), 0, st, logits, V, tiles, logprobs, tokens, lens);
    PIE_LAUNCH_CHECK();
    return PIE_OK;
}

// one row whose partials the lm_head GEMV left
static inline int logits_tail_launch(int dtype, const u16 *logits, int V, const LogitStat *stats, int n_stats, float *logprobs,
                                     int *token, DecState *state, int *history, int hist_cap, hipStream_t st, const unsigned *err_word = nullptr) {
    if (dtype != PIE_BF16 && dtype != PIE_F16) return pie::fail(PIE_E_ARG, "logits tail: dtype must be PIE_BF16 or PIE_F16");
    if (n_stats > TAIL_MAX_STATS) return pie::fail(PIE_E_SHAPE, "logits tail: too many partials");
    if (dtype == PIE_BF16)
        hipLaunchKernelGGL(k_logits_finish<BF16>, dim3(TAIL_FINISH_BLOCKS), dim3(256), 0, st, logits, V, stats, n_stats, logprobs, token, state, history, hist_cap, err_word, (int *)nullptr);
    else
        hipLaunchKernelGGL(k_logits_finish<F16>, dim3(TAIL_FINISH_BLOCKS), dim3(256), 0, st, logits, V, stats, n_stats, logprobs, token, state, history, hist_cap, err_word, (int *)nullptr);
    PIE_LAUNCH_CHECK();
    return PIE_OK;
}
