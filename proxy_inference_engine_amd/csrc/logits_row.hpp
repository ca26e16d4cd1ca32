// logits_row.hpp -- log-softmax normaliser and greedy token of whole logit rows, in one launch or in two (engine/inference_engine.py:254,268-271, samplers/__init__.py:37-38).
//
// Every workgroup of a row reads the whole row (from L2: a row's workgroups share an XCD where the rows come in eights), keeps one running (max, sum, first index of the max) per thread and
// merges them once; then it writes its share of the log-probabilities.  What bounds it is the launch and one workgroup's exponentials, 32 a thread of 32768 logits.  16-bit rows of 32768, traced,
// us: 8 rows 6.9, 32 rows 8.0; with expf, a dozen instructions, 9.9 and 11.  Few rows of many more logits come in tiles, a launch in front of this one (logits_in_tiles): 128256 logits, traced,
// us, 8 rows 17.3 -> 8.6, 32 rows 21.2 -> 13.0; tiles of 32768 7.6 and 9.0.
#pragma once
#include "common.hpp"

constexpr int LOGITS_ROW_THREADS = 1024;

// eight consecutive logits (16-byte aligned), as they lie and as numbers
template <class L> struct LogitOctet;
template <> struct LogitOctet<u16> {
    uint4 q;
    __device__ __forceinline__ void load(const u16 *p) { q = *reinterpret_cast<const uint4 *>(p); }
    template <class T>
    __device__ __forceinline__ void get(float (&v)[8]) const {
        const u32 w[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
        for (int j = 0; j < 4; ++j) v[2 * j] = lo_f32<T>(w[j]), v[2 * j + 1] = hi_f32<T>(w[j]);
    }
};
template <> struct LogitOctet<float> {
    float4 a, b;
    __device__ __forceinline__ void load(const float *p) { a = reinterpret_cast<const float4 *>(p)[0], b = reinterpret_cast<const float4 *>(p)[1]; }
    template <class T>
    __device__ __forceinline__ void get(float (&v)[8]) const { v[0] = a.x, v[1] = a.y, v[2] = a.z, v[3] = a.w, v[4] = b.x, v[5] = b.y, v[6] = b.z, v[7] = b.w; }
};
// exp(x) for x <= 0: 2^t (1 + r), t = x log2 e as rounded, r = x - t ln 2 what the roundings left out.  (2^t alone is off by up to |x| 2^-24, alike for like logits: a sum of terms far below
// the maximum takes it whole.)  From -104 down e^x is below the smallest number there is, and -inf would make r a NaN.  A NaN counts nothing.
__device__ __forceinline__ float logits_exp(float x) {
    constexpr float LN2 = 0.69314718055994531f, REST = (float)(0.69314718055994531 - (double)LN2);
    x = fmaxf(x, -104.0f);
    const float t = x * 1.4426950408889634f, e = __builtin_amdgcn_exp2f(t);
    return fmaf(e, fmaf(-t, REST, fmaf(-t, LN2, x)), e);
}
template <class T> __device__ __forceinline__ float logit_f32(u16 x) { return T::to_f32(x); }
template <class T> __device__ __forceinline__ float logit_f32(float x) { return x; }

// -> maximum M of the n logits from row on, sum of exp(logit - M) and the first index of the maximum (the first logit's is at), in every thread of the workgroup.  A NaN counts nothing, in an infinite maximum's row neither does
// what is finite; a row of nothing above -inf has token INT_MAX.
template <class T, int NT, class L>
__device__ __forceinline__ void logits_stats(const L *row, int V, int first, float &M, float &S, int &token) {
    constexpr int WAVES = NT / 64, U = 4;  // U octets of a thread in flight
    __shared__ float s_max[WAVES], s_sum[WAVES];
    __shared__ int s_arg[WAVES];
    float m = -INFINITY, s = 0.0f;
    int arg = 0x7fffffff;
    auto take = [&](const float (&v)[8], int at, int step, int n) {  // the first n of v: logits at, at + step, ...
        float top = v[0];
#pragma unroll
        for (int j = 1; j < 8; ++j)
            if (j < n) top = fmaxf(top, v[j]);
        if (top > m) {
            s *= logits_exp(m - top), m = top;
#pragma unroll
            for (int j = 7; j >= 0; --j)
                if (j < n && v[j] == top) arg = at + j * step;
        }
        if (m > -INFINITY) {
            float e[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) e[j] = j < n ? logits_exp(v[j] - m) : 0.0f;
            s += ((e[0] + e[1]) + (e[2] + e[3])) + ((e[4] + e[5]) + (e[6] + e[7]));
        }
    };
    if ((V & 7) == 0 && ((size_t)row & 15) == 0) {
        for (int base = threadIdx.x * 8; base < V; base += U * NT * 8) {
            LogitOctet<L> q[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int i = base + u * NT * 8;
                q[u].load(row + (i < V ? i : V - 8));
            }
            __builtin_amdgcn_sched_barrier(0);  // (the loads stay together: sunk to their uses each waits out its own latency)
#pragma unroll
            for (int u = 0; u < U; ++u)
                if (base + u * NT * 8 < V) {
                    float v[8];
                    q[u].template get<T>(v);
                    take(v, base + u * NT * 8, 1, 8);
                }
        }
    } else {
        for (int i = threadIdx.x; i < V; i += NT * 8) {
            float v[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) v[j] = logit_f32<T>(row[min(i + j * NT, V - 1)]);
            take(v, i, NT, min(8, (V - 1 - i) / NT + 1));
        }
    }
    const int wave = threadIdx.x >> 6;
    const float wm = wave_max(m);
    int cand = m == wm ? arg : 0x7fffffff;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) cand = min(cand, __shfl_xor(cand, o, 64));
    const float ws = wave_sum(s > 0.0f ? s * logits_exp(m - wm) : 0.0f);
    if ((threadIdx.x & 63) == 0) s_max[wave] = wm, s_sum[wave] = ws, s_arg[wave] = cand;
    __syncthreads();
    // every wave merges the waves', one a lane (and adds them as a tree)
    const int lane = threadIdx.x & 63, w = lane & (WAVES - 1);
    const float wmax = s_max[w];
    M = wave_max(wmax);
    token = wmax == M ? s_arg[w] : 0x7fffffff;
#pragma unroll
    for (int o = WAVES / 2; o > 0; o >>= 1) token = min(token, __shfl_xor(token, o, 64));
    S = wave_sum(lane < WAVES && s_sum[w] > 0.0f ? s_sum[w] * logits_exp(wmax - M) : 0.0f);
    if (token != 0x7fffffff) token += first;
}

// Rows in 64 tiles, for a launch of their own
constexpr int LOGITS_TILES = 64, LOGITS_TILE_THREADS = 256;
struct RowStat {  // of a tile (of an empty one: -inf, 0, INT_MAX)
    float max, sum;
    int arg, pad;
};
template <class T, class L>
__global__ void __launch_bounds__(LOGITS_TILE_THREADS) k_logits_tiles(const L *logits, int V, RowStat *stats) {  // grid (tiles, rows)
    const int len = ((V + LOGITS_TILES - 1) / LOGITS_TILES + 7) & ~7, begin = blockIdx.x * len;
    RowStat s;
    s.pad = 0;
    logits_stats<T, LOGITS_TILE_THREADS>(logits + (size_t)blockIdx.y * V + begin, min(V - begin, len), begin, s.max, s.sum, s.arg);
    if (threadIdx.x == 0) stats[blockIdx.y * LOGITS_TILES + blockIdx.x] = s;
}

// -> log(sum exp(row)) and the row's first maximum, in every thread: of the row's tiles where a launch in front of this one left them, else of the row
template <class T, class L>
__device__ __forceinline__ void logits_row_stats(const L *row, int V, const RowStat *tiles, float &lse, int &token) {
    float M, S;
    if (tiles) {  // (every wave merges them, one a lane)
        const RowStat s = tiles[threadIdx.x & 63];
        M = wave_max(s.max), token = s.max == M ? s.arg : 0x7fffffff;
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) token = min(token, __shfl_xor(token, o, 64));
        S = wave_sum(s.sum > 0.0f ? s.sum * logits_exp(s.max - M) : 0.0f);
    } else logits_stats<T, LOGITS_ROW_THREADS>(row, V, 0, M, S, token);
    lse = M + logf(S);
}

// logprobs = row - lse over share `part` of `parts`
template <class T, class L>
__device__ __forceinline__ void logits_row_write(const L *row, int V, float lse, int part, int parts, float *logprobs) {
    const int share = ((V + parts - 1) / parts + 7) & ~7, begin = part * share, end = min(V, begin + share);
    if ((V & 7) == 0 && (((size_t)row | (size_t)logprobs) & 15) == 0) {
        for (int i = begin + threadIdx.x * 8; i < end; i += LOGITS_ROW_THREADS * 8) {
            LogitOctet<L> q;
            float v[8];
            q.load(row + i), q.template get<T>(v);
            *reinterpret_cast<float4 *>(logprobs + i) = make_float4(v[0] - lse, v[1] - lse, v[2] - lse, v[3] - lse);
            *reinterpret_cast<float4 *>(logprobs + i + 4) = make_float4(v[4] - lse, v[5] - lse, v[6] - lse, v[7] - lse);
        }
    } else {
        for (int i = begin + threadIdx.x; i < end; i += LOGITS_ROW_THREADS) logprobs[i] = logit_f32<T>(row[i]) - lse;
    }
}

// workgroups per row: a workgroup on every CU while the rows are few, so that a CU's writes are a fraction of a row (all read all of it)
static inline int logits_row_parts(int rows) { return rows >= 256 ? 1 : rows <= 16 ? 16 : 256 / rows; }
// A row's exponentials are taken by each of its workgroups, by tiles only once but in two launches (fp32: 9.5 us whatever the row is, until the tiles fill the chip): worth it for rows of a large
// vocabulary that are not many.  One launch / two, us, fp32: 49152 logits, 8 rows 8.7 / 9.4; 65536, 8 rows 10.2 / 9.5, 48 rows 12.8 / 12.8; 128256, 1 row 15.7 / 9.7, 64 rows 23.3 / 20.7,
// 128 rows 34.3 / 36.7; 262144, 8 rows 29.8 / 9.7.  Rows that are no multiple of eight logits are loaded one by one and cost two fifths more: 50257, 8 rows 11.9 / 9.6, 64 rows 14.2 / 16.1.
static inline bool logits_in_tiles(int rows, int V) {
    const int work = V & 7 ? V + V / 5 * 2 : V;
    return work >= 60000 && rows <= work / 1500;
}
