// rows_gemm.hip -- the Linear of the layer-stack models: y[M, N] = x[M, K] . W[N, K]^T with the consumer's element-wise work in the epilogue.
//
// Few rows (a decode step, a short portion): the weights are read once and everything else is small.  A workgroup of eight waves owns
// 16 * NW output features; KW waves split K between them (NW * KW = 8).  A wave streams 1-KiB pieces of the W16M tiles (w16_gemm.hpp: 32
// features x 64 columns in MFMA operand order) -- half a tile row group per instruction, four 256-byte runs -- straight into the A operand of
// v_mfma_f32_16x16x32_bf16; the B operand is the matching 16 B of up to 16 rows of x, read through L2.  One row of x uses one of the 16 columns,
// which costs nothing: the matrix cores are idle either way.  The K-split partial sums meet in LDS.
//
// The same kernel runs batched over heads (per-head up- / down-projections), over a list of unlike matrices, grouped over the active experts of a mixture (row lists), and for
// any M (blockIdx.z walks 16 * NT rows at a time).  Long rows of x that several rows share a pass with go through LDS instead (k_rows_lds).
#include <algorithm>

#include "stack_types.hpp"

size_t w16m_size(int N, int K);

typedef __attribute__((ext_vector_type(8))) __bf16 mf_bf16x8;
typedef __attribute__((ext_vector_type(8))) _Float16 mf_f16x8;
typedef __attribute__((ext_vector_type(4))) float mf_f32x4;
typedef __attribute__((ext_vector_type(4))) u32 mf_u32x4;

namespace {

// What blockIdx.y selects: the matrix, its live rows, and how result rows map to x rows.
struct RowsWork {
    const char *w;
    const void *x;
    void *y;
    int N, K, ldx, ldy, count, row0;
    const int *rows;  // x row of local row i (nullptr: row0 + i)
    int xoff, yoff;
};
// b: blockIdx.y; last: the shared expert's
__device__ __forceinline__ bool rows_select(const RowsArgs &a, RowsWork &k, int b, int last) {
    k.w = a.m.w, k.x = a.m.x, k.y = a.m.y, k.N = a.m.N, k.K = a.m.K, k.ldx = a.m.ldx, k.ldy = a.m.ldy;
    k.count = a.M, k.row0 = 0, k.rows = a.rows, k.xoff = k.yoff = 0;
    if (a.n_mats) {
        const RowsMat &m = a.mats[b];
        k.w = m.w, k.x = m.x, k.y = m.y, k.N = m.N, k.K = m.K, k.ldx = m.ldx, k.ldy = m.ldy;
        return true;
    }
    if (a.shared.w && b == last) {
        k.w = a.shared.w, k.x = a.shared.x, k.y = a.shared.y, k.N = a.shared.N, k.K = a.shared.K, k.ldx = a.shared.ldx, k.ldy = a.shared.ldy;
        return true;
    }
    if (a.active) {
        const int e = a.active[b];
        if (e < 0) return false;
        k.row0 = a.offset[e], k.count = a.offset[e + 1] - k.row0;
        if (a.gather) k.rows = a.list + k.row0;
        k.w += (size_t)e * a.w_batch;
        return true;
    }
    k.w += (size_t)b * a.w_batch, k.xoff = b * a.x_batch, k.yoff = b * a.y_batch;
    return true;
}

template <class E>
__device__ __forceinline__ mf_f32x4 rows_mfma(mf_u32x4 w, mf_u32x4 x, mf_f32x4 acc) {
    if constexpr (__is_same(E, ElemF16)) return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(mf_f16x8, w), __builtin_bit_cast(mf_f16x8, x), acc, 0, 0, 0);
    else return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(mf_bf16x8, w), __builtin_bit_cast(mf_bf16x8, x), acc, 0, 0, 0);
}
__host__ __device__ __forceinline__ bool rows_paired(int epi) { return epi == ROWS_SILU_MUL || epi == ROWS_CLIP_MUL || epi == ROWS_GELU_MUL || epi == ROWS_SWIGLU; }

// One finished value (m: result row inside the group, n: feature); pair: the value of feature n + 1 (rows_paired)
template <class E>
__device__ __forceinline__ void rows_finish(const RowsArgs &a, const RowsWork &k, int m, int n, float v, float pair) {
    typedef typename E::type T;
    const size_t row = (size_t)(k.row0 + m);
    switch (a.epi) {
        case ROWS_STORE: ((T *)k.y)[row * k.ldy + k.yoff + n] = E::pack(v); break;
        case ROWS_SCALE_F32: ((float *)k.y)[row * k.ldy + k.yoff + n] = v * a.scale; break;
        case ROWS_RELU2: {
            const float r = fmaxf(v, 0.0f);
            ((T *)k.y)[row * k.ldy + n] = E::pack(r * r);
            break;
        }
        case ROWS_XIELU: ((T *)k.y)[row * k.ldy + n] = E::pack(xielu<sizeof(T) == 4>(v, a.act_alpha, a.act_limit)); break;
        case ROWS_SILU_MUL:
            if (!(n & 1)) ((T *)k.y)[row * k.ldy + (n >> 1)] = E::pack(v / (1.0f + expf(-v)) * pair);
            break;
        case ROWS_CLIP_MUL:
            if (!(n & 1)) ((T *)k.y)[row * k.ldy + (n >> 1)] = E::pack(clipped_glu(v, pair, a.act_alpha, a.act_limit));
            break;
        case ROWS_GELU_MUL:
            if (!(n & 1)) {
                if (a.bias) v += BF16::to_f32(a.bias[n]), pair += BF16::to_f32(a.bias[n + 1]);
                ((T *)k.y)[row * k.ldy + (n >> 1)] = E::pack(gelu_tanh<sizeof(T) == 4>(v) * pair);
            }
            break;
        case ROWS_GELU_SIDE: ((T *)k.y)[row * k.ldy + n] = E::pack(gelu_tanh<sizeof(T) == 4>(v) * BF16::to_f32(token_vector(a.side, row)[n])); break;
        case ROWS_SOFTCAP: ((float *)k.y)[row * k.ldy + n] = a.act_limit * stack_tanh<sizeof(T) == 4>(v * a.scale / a.act_limit); break;
        case ROWS_LINEAR:
        case ROWS_SWIGLU:
            if constexpr (sizeof(T) == 2) {  // (the Llama's Linears: 16-bit stacks only)
                auto once = [&](float z, int at) {
                    const T r = E::pack(z);
                    return a.bias ? E::pack(E::load(&r) + E::load((const T *)a.bias + at)) : r;
                };
                const T g = once(v, n);
                if (a.epi == ROWS_LINEAR) ((T *)k.y)[row * k.ldy + n] = g;
                else if (!(n & 1)) {
                    const float z = E::load(&g);
                    const T s = E::pack(z / (1.0f + expf(-z))), u = once(pair, n + 1);
                    ((T *)k.y)[row * k.ldy + (n >> 1)] = E::pack(E::load(&s) * E::load(&u));
                }
            }
            break;
        case ROWS_SPLIT:
            if (n < a.split) ((T *)k.y)[row * k.ldy + n] = E::pack(v);
            else a.y2[row * a.ldy2 + n - a.split] = v;
            break;
        case ROWS_RESIDUAL: {
            float *xp = a.res + row * a.ld_res + n;
            const float x = *xp + point_norm(a.post, n, v);
            *xp = x;
            ((T *)a.h)[row * a.ldh + n] = E::pack(point_norm(a.next, n, x));
            break;
        }
    }
}

__host__ __device__ __forceinline__ int rows_riders(const RowsArgs &a) { return (a.append.M > 0) + (a.cache.M > 0) + (a.rotate.M > 0); }
static void rows_slice(RowsArgs &a, unsigned x, int batches) {  // x: gridDim.x
    const int M = std::max(a.append.M, std::max(a.cache.M, a.rotate.M));
    a.ride_slices = M > 0 && batches < 65000 ? std::min(4, (M + (int)x - 1) / (int)x) : 1;
}
// the last blockIdx.y's, ride_slices each: what rides along, a row to a workgroup where rows and workgroups allow it (two rows one after the other outlast a small product: heads of [512, 128] beside 32 rows'
// append 9.8 us, in two slices and with the norm weights asked for early 8.3)
template <class E, int THREADS>
__device__ __forceinline__ bool rows_ride(const RowsArgs &a, float *red) {
    int i = (int)(gridDim.y - 1 - blockIdx.y);
    if (i >= rows_riders(a) * a.ride_slices) return false;
    if (blockIdx.z) return true;
    const int slice = i % a.ride_slices;
    i /= a.ride_slices;
    const bool append = a.append.M > 0 && i == 0;
    i -= a.append.M > 0;
    const bool cache = a.cache.M > 0 && i == 0;
    const int M = append ? a.append.M : cache ? a.cache.M : a.rotate.M;
    for (int m = blockIdx.x + slice * gridDim.x; m < M; m += gridDim.x * a.ride_slices) {
        if (append) latent_append_row<E, ElemF32, THREADS>(a.append, m, red);
        else if (cache) latent_cache_row<E, THREADS>(a.cache, m, red);
        else rotate_row<E, THREADS>(a.rotate, m);
        __syncthreads();
    }
    return true;
}

// NT: blocks of 16 rows of x; KW: waves along K; NN: blocks of 16 features per wave (two share the x operands); MERGE: x = the merged key splits of head
// blockIdx.y (RowsArgs::merge), put together in LDS by every workgroup of the head; NORM: RowsArgs::x_norm (every workgroup sees its rows whole)
template <class E, int NT, int KW, int NN, bool MERGE = false, bool NORM = false>
__global__ void __launch_bounds__(512) k_rows_w16m(const RowsArgs a) {
    constexpr int NW = 8 / KW, U = NT >= 4 ? 2 : 4;
    constexpr int ST = 20;  // floats per (row, 16 features) line of the reduction image
    __shared__ __attribute__((aligned(16))) float s_red[8 * NN * NT * 16 * ST];
    __shared__ float s_ss[NORM ? 8 : 1][16];
    static_assert(!NORM || NT == 1, "norms: sixteen rows");
    if (rows_ride<ElemBF16, 512>(a, s_red)) return;
    __shared__ __attribute__((aligned(16))) u16 s_x[MERGE ? MERGE_ROWS * (MERGE_LDR + 64) : 8];
    const int ldx_lds = a.merge.ldr + 64;
    if constexpr (MERGE) {
        __shared__ float s_f[MERGE_ROWS][64];
        const int H = a.merge.H, M = a.merge.M, w = threadIdx.x >> 6;
        if (w < M) s_f[w][threadIdx.x & 63] = latent_split_weight(a.merge, (size_t)w * H + blockIdx.y, threadIdx.x & 63);
        __syncthreads();
        const int quads = ldx_lds / 4;
        for (int i = threadIdx.x; i < M * quads; i += 512) {
            const int m = i / quads, r = i % quads * 4;
            float4 v = make_float4(0, 0, 0, 0);  // (columns past the latent meet zero weights: zeros)
            if (r < a.merge.ldr) v = latent_merge4(a.merge, (size_t)m * H + blockIdx.y, r, [&](int s) { return s_f[m][s]; });
            *(uint2 *)(s_x + m * ldx_lds + r) = make_uint2(pack2<BF16>(v.x, v.y), pack2<BF16>(v.z, v.w));
        }
        __syncthreads();
    }
    RowsWork k;
    if (!rows_select(a, k, blockIdx.y, (int)gridDim.y - 1)) return;
    const int i0 = blockIdx.z * 16 * NT;
    if (i0 >= k.count) return;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wn = wave / KW, wk = wave % KW;
    const int t16 = (blockIdx.x * NW + wn) * NN;  // this wave's first block of 16 output features
    if ((int)blockIdx.x * NW * NN * 16 >= k.N) return;
    const int c = lane & 15, kq = lane >> 4;
    const int groups = (k.K + 63) >> 6, steps = 2 * groups;
    const bool live = t16 * 16 < k.N;  // (NN = 2: both blocks lie in one 32-row tile, which is stored whole)

    float ss = 0.0f;
    mf_f32x4 acc[NN][NT];
#pragma unroll
    for (int n = 0; n < NN; ++n)
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[n][t] = (mf_f32x4){0.0f, 0.0f, 0.0f, 0.0f};
    if (live) {
        const char *wp = k.w + (size_t)(t16 >> 1) * groups * 4096 + ((kq >> 1) * 1024 + ((kq & 1) * 32 + (t16 & 1) * 16 + c) * 16);
        const u16 *xp[NT];
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            int i = i0 + 16 * t + c;
            i = i < k.count ? i : k.count - 1;  // rows past the end repeat the last one (never stored)
            const int xr = k.rows ? k.rows[i] : k.row0 + i;
            xp[t] = MERGE ? s_x + xr * ldx_lds + 8 * kq : (const u16 *)k.x + (size_t)xr * k.ldx + k.xoff + 8 * kq;
        }
        auto fetch = [&](int s, mf_u32x4(&wv)[U][NN], mf_u32x4(&xv)[U][NT]) {
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int ss = s + u * KW, cl = ss < steps ? ss : steps - 1;
#pragma unroll
                for (int n = 0; n < NN; ++n) wv[u][n] = __builtin_nontemporal_load((const mf_u32x4 *)(wp + (size_t)cl * 2048 + n * 256));
#pragma unroll
                for (int t = 0; t < NT; ++t) xv[u][t] = *(const mf_u32x4 *)(xp[t] + 32 * cl);
            }
            __builtin_amdgcn_sched_barrier(0);
        };
        auto multiply = [&](int s, const mf_u32x4(&wv)[U][NN], const mf_u32x4(&xv)[U][NT]) {
#pragma unroll
            for (int u = 0; u < U; ++u)
#pragma unroll
                for (int n = 0; n < NN; ++n) {
                    mf_u32x4 w = wv[u][n];
                    if (s + u * KW >= steps) w = (mf_u32x4){0u, 0u, 0u, 0u};
                    if constexpr (NORM)
                        if (n == 0 && s + u * KW < steps && 32 * (s + u * KW) + 8 * kq < k.K)  // (what lies behind the row belongs to others; a row's padding to 8 is zero)
#pragma unroll
                            for (int i = 0; i < 4; ++i) ss = fmaf(lo_f32<BF16>(xv[u][0][i]), lo_f32<BF16>(xv[u][0][i]), fmaf(hi_f32<BF16>(xv[u][0][i]), hi_f32<BF16>(xv[u][0][i]), ss));
#pragma unroll
                    for (int t = 0; t < NT; ++t) acc[n][t] = rows_mfma<E>(w, xv[u][t], acc[n][t]);
                }
        };
        // (each half round's loads in a piece, no half round past the end (within the last one, steps past it read the last tile again): the compiler's waits count them exactly.  us, one row, with its own order and a last round of loads for nothing / this: [5120, 3072] 10.4 / 9.0,
        // [16384, 3072] 19.5 / 18.1, [6144, 4096] 12.3 / 11.9, [4096, 4096] 8.0 / 8.0)
        mf_u32x4 w0[U][NN], w1[U][NN], x0[U][NT], x1[U][NT];
        constexpr int R = U * KW;
        int s = wk;
        fetch(s, w0, x0);
        for (; s + 2 * R < steps; s += 2 * R) {
            fetch(s + R, w1, x1);
            multiply(s, w0, x0);
            fetch(s + 2 * R, w0, x0);
            multiply(s + R, w1, x1);
        }
        if (s + R < steps) {
            fetch(s + R, w1, x1);
            multiply(s, w0, x0);
            multiply(s + R, w1, x1);
        } else
            multiply(s, w0, x0);
    }
    if constexpr (NORM) {
        ss = xor32_sum(xor16_sum(ss));
        if (kq == 0) s_ss[wave][c] = ss;
    }
    // lane (kq, c) holds features 4 kq .. + 3 of row c
#pragma unroll
    for (int n = 0; n < NN; ++n)
#pragma unroll
        for (int t = 0; t < NT; ++t) *(mf_f32x4 *)(s_red + (((wave * NN + n) * NT + t) * 16 + c) * ST + 4 * kq) = acc[n][t];
    __syncthreads();
    const bool paired = rows_paired(a.epi);
    for (int id = threadIdx.x; id < NW * NN * NT * 256; id += 512) {
        const int nl = id & 15, ml = (id >> 4) % (16 * NT), wn2 = id / (256 * NT), w = wn2 / NN, nn = wn2 % NN;
        const int n = ((int)blockIdx.x * NW * NN + wn2) * 16 + nl, m = i0 + ml;
        if (n >= k.N || m >= k.count) continue;
        if (paired && (nl & 1)) continue;
        const float *r = s_red + (((w * KW * NN + nn) * NT + (ml >> 4)) * 16 + (ml & 15)) * ST + nl;
        float v = 0.0f, p = 0.0f;
#pragma unroll
        for (int q = 0; q < KW; ++q) v += r[q * NN * NT * 16 * ST];
        if (paired)
#pragma unroll
            for (int q = 0; q < KW; ++q) p += r[q * NN * NT * 16 * ST + 1];
        if constexpr (NORM) {
            float sum = 0.0f;
#pragma unroll
            for (int q = 0; q < KW; ++q) sum += s_ss[w * KW + q][ml];
            v *= 1.0f / sqrtf(sum / (float)k.K + a.x_eps);
        }
        rows_finish<E>(a, k, m, n, v, p);
    }
}

// Rows that share a pass, x through LDS.  k_rows_w16m fetches every 16 B of x into the lanes that multiply it, 16 scattered runs of 64 B per instruction, for every 16 or 32 features
// again: from 8 rows on that, and no longer the weights, is what the time goes to ([28672, 4096]: 37 us with 1 row, 41 / 52 / 58 / 88 with 8 / 16 / 32 / 64; profile and counts agree, the
// matrix cores idle).  Here a workgroup of WV (eight) waves takes 16 NN features and all of K in chunks of 32 WV U columns: the chunk's rows come in as whole lines, once per workgroup
// (registers, then one of two LDS buffers; rows padded by 16 B, conflict-free both ways), each wave multiplies every WV-th 32-column step by weights that it streams two chunks ahead.
// Loads go by descriptors whose bounds drop what lies behind a row, a matrix or K (zeros), so no load has a branch around it.  Two workgroups of eight waves share a CU (launch bounds: 128 registers),
// one loads while the other finishes.  Sixteen features per wave and step re-read x most (NN = 1), four blocks least: NN follows from how many workgroups are left (rows_lds_pick).
// [28672, 4096] with 8 / 16 / 32 / 64 rows: 39 / 40 / 42 / 64 us = 6.0 / 5.9 / 5.6 / 3.7 TB/s.  Experts have fewer bytes per workgroup, and workgroups of four waves (WV) fill the gaps that
// others leave better: 60 active ones of [2816, 2048] with 3 rows each 131 (k_rows_w16m) -> 110 (eight waves) -> 103 us (6.7 TB/s), of [2048, 1408] 90 -> 58 -> 53 us.
template <class E, int NT, int NN, int U, int WV = 8>
__global__ void __launch_bounds__(64 * WV, 4) k_rows_lds(const RowsArgs a) {
    constexpr int C = 32 * WV * U, LD = C + 8, ST = 20;            // columns of x per chunk; u16 per LDS row; floats per line of the reduction image
    constexpr int PR = C / 8, RP = 64 * WV / PR, XJ = 16 * NT / RP;  // 16-byte pieces per row of a chunk; rows that all threads fetch at once; pieces per thread
    constexpr size_t X_BYTES = (size_t)2 * 16 * NT * LD * 2, RED_BYTES = (size_t)WV * NN * NT * 16 * ST * 4;
    static_assert(64 * WV % PR == 0 && 16 * NT % RP == 0, "whole rows per round of loads");
    __shared__ __attribute__((aligned(16))) char s_mem[X_BYTES > RED_BYTES ? X_BYTES : RED_BYTES];
    u16 *s_x = (u16 *)s_mem;
    float *s_red = (float *)s_mem;
    if constexpr (__is_same(E, ElemBF16))
        if (rows_ride<ElemBF16, 64 * WV>(a, s_red)) return;
    int bx = blockIdx.x, by = blockIdx.y;
    if (a.flat_tiles < 0) {  // a list, workgroup after workgroup
        for (by = 0;; ++by) {
            const int t = (a.mats[by].N + 16 * NN - 1) / (16 * NN);
            if (bx < t) break;
            bx -= t;
        }
    } else if (a.flat_tiles > 0) {  // the shared expert (it has all rows, and the longest workgroups), then the others
        const int first = a.shared.w ? (a.shared.N + 16 * NN - 1) / (16 * NN) : 0;
        if (bx < first) by = a.flat_batches;
        else by = (bx - first) / a.flat_tiles, bx = (bx - first) % a.flat_tiles;
    }
    RowsWork k;
    if (!rows_select(a, k, by, a.flat_tiles > 0 ? a.flat_batches : (int)gridDim.y - 1)) return;
    if (bx * NN * 16 >= k.N) return;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), c = lane & 15, kq = lane >> 4;
    const int t16 = bx * NN, groups = (k.K + 63) >> 6, steps = 2 * groups, K8 = (k.K + 7) & ~7, iters = (steps + WV * U - 1) / (WV * U);
    const int w_tiles = min(((k.N + 31) >> 5) - (t16 >> 1), (NN + 1) / 2);  // 32-row tiles of this workgroup: a matrix ends with a whole tile
    const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc(const_cast<char *>(k.w + (size_t)(t16 >> 1) * groups * 4096), 0, w_tiles * groups * 4096, 0x00020000);
    const unsigned wlane = (kq >> 1) * 1024 + ((kq & 1) * 32 + c) * 16 + (t16 & 1) * 256;
    const int xc = threadIdx.x % PR * 8, xr0 = threadIdx.x / PR;  // this thread's columns and rows of a chunk
    for (int i0 = blockIdx.z * 16 * NT; i0 < k.count; i0 += gridDim.z * 16 * NT) {
        const u16 *x0 = (const u16 *)k.x + (k.rows ? 0 : (size_t)(k.row0 + i0) * k.ldx) + k.xoff;
        const __amdgpu_buffer_rsrc_t xs = __builtin_amdgcn_make_buffer_rsrc(const_cast<u16 *>(x0), 0, 0x7FFFFFF0, 0x00020000);
        constexpr unsigned NOWHERE = 0x80000000u;  // behind every descriptor's end
        unsigned xo[XJ];
#pragma unroll
        for (int j = 0; j < XJ; ++j) {
            const int r = xr0 + RP * j;
            const bool in = i0 + r < k.count;
            const int xr = k.rows ? k.rows[in ? i0 + r : i0] : r;
            xo[j] = in ? (unsigned)(xr * k.ldx + xc) * 2u : NOWHERE;
        }
        auto load_x = [&](int it, mf_u32x4(&xv)[XJ]) {
            const unsigned at = xc + it * C < K8 ? (unsigned)(it * C * 2) : NOWHERE;
#pragma unroll
            for (int j = 0; j < XJ; ++j) xv[j] = __builtin_amdgcn_raw_buffer_load_b128(xs, (int)(xo[j] | at) < 0 ? NOWHERE : xo[j] + at, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        };
        auto store_x = [&](int buf, const mf_u32x4(&xv)[XJ]) {
#pragma unroll
            for (int j = 0; j < XJ; ++j) *(mf_u32x4 *)(s_x + (buf * 16 * NT + xr0 + RP * j) * LD + xc) = xv[j];
        };
        auto load_w = [&](int it, mf_u32x4(&wv)[U][NN]) {
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int s = (it * U + u) * WV + wave;
#pragma unroll
                for (int n = 0; n < NN; ++n)  // non-temporal: a weight is read once, except an expert's with more than 16 NT rows
                    wv[u][n] = __builtin_amdgcn_raw_buffer_load_b128(wr, s < steps ? wlane + (unsigned)((n >> 1) * groups * 4096 + s * 2048 + (n & 1) * 256) : NOWHERE, 0, 2);
            }
            __builtin_amdgcn_sched_barrier(0);
        };
        mf_f32x4 acc[NN][NT];
#pragma unroll
        for (int n = 0; n < NN; ++n)
#pragma unroll
            for (int t = 0; t < NT; ++t) acc[n][t] = (mf_f32x4){0.0f, 0.0f, 0.0f, 0.0f};
        auto multiply = [&](int buf, const mf_u32x4(&wv)[U][NN]) {
#pragma unroll
            for (int u = 0; u < U; ++u) {
                mf_u32x4 xv[NT];
#pragma unroll
                for (int t = 0; t < NT; ++t) xv[t] = *(const mf_u32x4 *)(s_x + (buf * 16 * NT + 16 * t + c) * LD + (WV * u + wave) * 32 + 8 * kq);
#pragma unroll
                for (int n = 0; n < NN; ++n)
#pragma unroll
                    for (int t = 0; t < NT; ++t) acc[n][t] = rows_mfma<E>(wv[u][n], xv[t], acc[n][t]);
            }
        };
        // (x before w: waiting for the next chunk's x must not wait for the weights behind it.  The loads stay in this order, and the last two chunks, or one of an odd number, load nothing; of an odd number the round before asks for a chunk past the end, which the
        // descriptors drop.  With loads that the scheduler moved, or a
        // round left halfway by a break, the compiler waited for every load in flight in every other chunk.  us, 8 / 32 rows, that / this: [6144, 4096] 13.1 / 12.4, 16.7 / 15.9; [5120, 3072] 10.9 / 10.0,
        // 13.9 / 13.2; [4096, 14336] 23.5 / 23.0, 33.5 / 31.4; [10752, 4096] 19.5 / 18.7, 23.2 / 22.1; [32768, 4096] 43.4 / 43.0, 47.2 / 45.8; [28672, 4096] 40.3 / 40.3, 42.9 / 42.7)
        mf_u32x4 w[2][U][NN], xv[XJ];
        load_x(0, xv);
        load_w(0, w[0]);
        store_x(0, xv);
        load_x(1, xv);
        load_w(1, w[1]);
        __syncthreads();
        int it = 0;
        for (; it + 2 < iters; it += 2) {
#pragma unroll
            for (int d = 0; d < 2; ++d) {
                multiply(d, w[d]);
                store_x(d ^ 1, xv);
                load_x(it + d + 2, xv);
                load_w(it + d + 2, w[d]);
                __syncthreads();
            }
        }
        multiply(0, w[0]);
        if (it + 1 < iters) {
            store_x(1, xv);
            __syncthreads();
            multiply(1, w[1]);
        }
        __syncthreads();
        // lane (kq, c) holds features 4 kq .. + 3 of row c
#pragma unroll
        for (int n = 0; n < NN; ++n)
#pragma unroll
            for (int t = 0; t < NT; ++t) *(mf_f32x4 *)(s_red + (((wave * NN + n) * NT + t) * 16 + c) * ST + 4 * kq) = acc[n][t];
        __syncthreads();
        const bool paired = rows_paired(a.epi);
        for (int id = threadIdx.x; id < NN * NT * 256; id += 64 * WV) {
            const int nl = id & 15, ml = (id >> 4) % (16 * NT), nn = id / (256 * NT), n = (t16 + nn) * 16 + nl, m = i0 + ml;
            if (n >= k.N || m >= k.count || (paired && (nl & 1))) continue;
            const float *r = s_red + ((nn * NT + (ml >> 4)) * 16 + (ml & 15)) * ST + nl;
            float v = 0.0f, p = 0.0f;
#pragma unroll
            for (int q = 0; q < WV; ++q) v += r[q * NN * NT * 16 * ST];
            if (paired)
#pragma unroll
                for (int q = 0; q < WV; ++q) p += r[q * NN * NT * 16 * ST + 1];
            rows_finish<E>(a, k, m, n, v, p);
        }
        __syncthreads();
    }
}

// fp32: one output per thread, 16 features x 16 rows per workgroup, both operands through LDS
__global__ void __launch_bounds__(256) k_rows_f32(const RowsArgs a) {
    __shared__ float s_w[16][65], s_x[16][65], s_v[16][17];
    if (rows_ride<ElemF32, 256>(a, s_v[0])) return;
    RowsWork k;
    if (!rows_select(a, k, blockIdx.y, (int)gridDim.y - 1)) return;
    const int i0 = blockIdx.z * 16, n0 = blockIdx.x * 16;
    if (i0 >= k.count || n0 >= k.N) return;
    const int tn = threadIdx.x & 15, tm = threadIdx.x >> 4;
    const int Kp = (k.K + 63) & ~63;
    float acc = 0.0f;
    for (int k0 = 0; k0 < Kp; k0 += 64) {
        for (int id = threadIdx.x; id < 1024; id += 256) {
            const int r = id >> 6, c = id & 63;
            s_w[r][c] = n0 + r < k.N ? ((const float *)k.w)[(size_t)(n0 + r) * Kp + k0 + c] : 0.0f;
            int i = i0 + r;
            i = i < k.count ? i : k.count - 1;
            const int xr = k.rows ? k.rows[i] : k.row0 + i;
            s_x[r][c] = k0 + c < k.K ? ((const float *)k.x)[(size_t)xr * k.ldx + k.xoff + k0 + c] : 0.0f;
        }
        __syncthreads();
#pragma unroll 16
        for (int c = 0; c < 64; ++c) acc = fmaf(s_w[tn][c], s_x[tm][c], acc);
        __syncthreads();
    }
    s_v[tm][tn] = acc;
    __syncthreads();
    const int n = n0 + tn, m = i0 + tm;
    if (n < k.N && m < k.count) rows_finish<ElemF32>(a, k, m, n, acc, s_v[tm][tn < 15 ? tn + 1 : 15]);
}

template <class E, int NT, int NN, int U, int WV = 8>
int rows_lds_go(RowsArgs a, int n_max, int batches, hipStream_t st) {
    auto tiles = [](int n) { return (unsigned)((n + 16 * NN - 1) / (16 * NN)); };
    rows_slice(a, tiles(n_max), batches);
    dim3 grid(tiles(n_max), (unsigned)(batches + rows_riders(a) * a.ride_slices), (unsigned)((a.M + 16 * NT - 1) / (16 * NT)));
    if (a.active) {  // one workgroup per tile of every expert, and it goes through all the expert's rows: most experts have few
        a.flat_batches = a.shared.w ? batches - 1 : batches, a.flat_tiles = (int)tiles(a.m.N);
        grid = dim3(a.flat_batches * a.flat_tiles + (a.shared.w ? tiles(a.shared.N) : 0));
    } else if (a.n_mats) {
        a.flat_tiles = -1, grid.x = 0, grid.y = 1;
        for (int i = 0; i < a.n_mats; ++i) grid.x += tiles(a.mats[i].N);
    }
    hipLaunchKernelGGL((k_rows_lds<E, NT, NN, U, WV>), grid, dim3(64 * WV), 0, st, a);
    PIE_LAUNCH_CHECK();
    return PIE_OK;
}

// Experts: blocks of 16 rows, or of 32 where many rows would make a workgroup go through its weights twice -- the shared expert's, which has all rows of the pass (beside so many other experts
// that it does not matter, 16 stay), or the experts' own.  From two rounds of workgroups on (four a CU) chunks of half the length.  us, 16 / 32 rows in long / 32 in short chunks:
//   64 experts, 6 a row, shared beside   [2816, 2048] 17 rows 92.4 / 91.3 / 91.0, 32 rows 110.8 / 109.0 / 109.3, 64 rows 126.6 / 121.0 / 121.8   [2048, 1408] 32 rows 57.2 / 60.0 / 56.2, 64 rows 68.3 / 66.6 / 63.4
//   8 experts, 2 a row   shared [7168, 2048] 17 rows 48.4 / 44.7 / 45.1, 64 rows 83.3 / 53.7 / 52.6   none 32 rows 38.2 / 41.9 / 41.6, 48 rows 50.0 / 42.8 / 42.4   shared [2048, 3584] 17 rows 34.6 / 28.6 / 25.5
//   16 experts, 2 a row, shared [2048, 2816] beside [2048, 1408]   17 rows 26.7 / 21.8 / 22.7, 64 rows 42.5 / 30.4 / 36.6      128 experts, 8 a row, shared [1536, 2048]   20 rows 86.1 / 88.3 / 87.9
static bool rows_lds_two(const RowsArgs &a, int batches) { return a.M > 16 && ((a.shared.w && batches <= 65) || a.mean_rows >= 12); }

// How many features a workgroup of k_rows_lds takes; blocks: 16-feature blocks of the whole launch.  As few as leave at most one workgroup per CU (a few more workgroups than that and most
// CUs wait for those with two), and beyond 1024 blocks two, four where 17 to 32 rows make x the larger part.  us with NN = 1 / 2 / 4:
//   8 rows   [4608, 2048] 10.1 / 8.2 / 10.2   [9216, 3072] 16.5 / 16.5 / 14.2   [11264, 2048] 14.0 / 13.1 / 11.4   [12320, 4096] 24.3 / 21.1 / 18.9   [18944, 4096] 31.3 / 29.9 / 34.7   [28672, 4096] 42.7 / 39.6 / 39.6
//   20 rows  [4608, 2048] 11.0 / 9.1 / 11.7   [9216, 3072] 19.3 / 18.6 / 16.1   [11264, 2048] 15.9 / 15.0 / 12.9   [18944, 4096] 37.0 / 33.5 / 37.1   [24576, 4096] 44.5 / 35.5 / 39.3   [28672, 4096] 51.0 / 43.9 / 40.7
// More than 32 rows of x per CU take the room of the fourth block.
template <class E>
int rows_lds_pick(const RowsArgs &a, int n_max, long blocks, int batches, hipStream_t st) {
    if (a.active) {
        if (!rows_lds_two(a, batches)) return rows_lds_go<E, 1, 2, 2, 4>(a, n_max, batches, st);
        const long wgs = (long)(batches - (a.shared.w != nullptr)) * ((a.m.N + 31) / 32) + (a.shared.w ? (a.shared.N + 31) / 32 : 0);
        return wgs < 2048 ? rows_lds_go<E, 2, 2, 2, 4>(a, n_max, batches, st) : rows_lds_go<E, 2, 2, 1, 4>(a, n_max, batches, st);
    }
    const int nn = blocks <= 256 ? 1 : blocks <= 512 ? 2 : blocks <= 1024 ? 4 : a.M <= 16 || blocks <= 1600 ? 2 : 4;
    if (a.M <= 16) return nn == 1 ? rows_lds_go<E, 1, 1, 4>(a, n_max, batches, st) : nn == 2 ? rows_lds_go<E, 1, 2, 2>(a, n_max, batches, st) : rows_lds_go<E, 1, 4, 1>(a, n_max, batches, st);
    if (a.M <= 32) return nn == 1 ? rows_lds_go<E, 2, 1, 2>(a, n_max, batches, st) : nn == 2 ? rows_lds_go<E, 2, 2, 2>(a, n_max, batches, st) : rows_lds_go<E, 2, 4, 1>(a, n_max, batches, st);
    return blocks < 320 ? rows_lds_go<E, 4, 1, 1>(a, n_max, batches, st) : rows_lds_go<E, 4, 2, 1>(a, n_max, batches, st);
}

template <class E, int NT, int NN>
int rows_go(RowsArgs a, int n_max, int k_max, int batches, hipStream_t st) {
    const int steps = 2 * ((k_max + 63) / 64), tiles = (n_max + 16 * NN - 1) / (16 * NN);
    const int z = (a.M + 16 * NT - 1) / (16 * NT);  // (grouped: most experts have few rows, their later z leave at once)
    // waves along K: enough steps for each, and enough workgroups for the chip
    int kw = steps >= 32 ? 8 : steps >= 16 ? 4 : steps >= 8 ? 2 : 1;
    while (kw < 8 && steps >= 2 * kw && (size_t)((tiles + 8 / kw - 1) / (8 / kw)) * batches * z < 256) kw *= 2;
    rows_slice(a, (unsigned)((tiles + 8 / kw - 1) / (8 / kw)), batches);
    const dim3 grid((unsigned)((tiles + 8 / kw - 1) / (8 / kw)), (unsigned)(batches + rows_riders(a) * a.ride_slices), (unsigned)z);
    auto go = [&](auto k8, auto k4, auto k2, auto k1) { hipLaunchKernelGGL((kw == 8 ? k8 : kw == 4 ? k4 : kw == 2 ? k2 : k1), grid, dim3(512), 0, st, a); };
    if constexpr (__is_same(E, ElemBF16)) {
        if (a.x_norm) go(&k_rows_w16m<E, 1, 8, 1, false, true>, &k_rows_w16m<E, 1, 4, 1, false, true>, &k_rows_w16m<E, 1, 2, 1, false, true>, &k_rows_w16m<E, 1, 1, 1, false, true>);
        else if (a.merge.splits > 0) go(&k_rows_w16m<E, 1, 8, 1, true>, &k_rows_w16m<E, 1, 4, 1, true>, &k_rows_w16m<E, 1, 2, 1, true>, &k_rows_w16m<E, 1, 1, 1, true>);
    }
    if (!a.x_norm && a.merge.splits <= 0) go(&k_rows_w16m<E, NT, 8, NN>, &k_rows_w16m<E, NT, 4, NN>, &k_rows_w16m<E, NT, 2, NN>, &k_rows_w16m<E, NT, 1, NN>);
    PIE_LAUNCH_CHECK();
    return PIE_OK;
}

__global__ void __launch_bounds__(256) k_pack_f32(const u16 *w, int N, int K, int Kp, float *out) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= (size_t)N * Kp) return;
    const int n = (int)(i / Kp), c = (int)(i % Kp);
    out[i] = c < K ? BF16::to_f32(w[(size_t)n * K + c]) : 0.0f;
}

}  // namespace

static bool rows_narrow(const RowsArgs &a, int n_max, int batches) { return (long)batches * n_max <= 16 * 64 && !a.merge.splits; }  // so few workgroups that they should not all read all rows
// k_rows_lds counts the bytes behind its first row of x in 31 bits: all of x where a list picks rows from it, 64 rows otherwise; of the widest operand that the launch has
static bool rows_lds_reaches(const RowsArgs &a) {
    const size_t rows = a.rows ? (size_t)a.x_rows : a.gather ? (size_t)a.M : 64;
    int ldx = a.n_mats ? 0 : a.shared.w ? std::max(a.m.ldx, a.shared.ldx) : a.m.ldx;
    for (int i = 0; i < a.n_mats; ++i) ldx = std::max(ldx, a.mats[i].ldx);
    return rows * (size_t)ldx * 2 < (1u << 31);
}
static long rows_blocks(const RowsArgs &a, int batches) {  // of 16 features, over the whole launch
    long blocks = a.n_mats ? 0 : (long)batches * ((a.m.N + 15) / 16);
    for (int i = 0; i < a.n_mats; ++i) blocks += (a.mats[i].N + 15) / 16;
    return blocks;
}
// x through LDS costs a start and an end per workgroup, the operands straight into the lanes cost x again per 16 features: the latter is the faster up to so many rows, fewer the longer the
// rows (its eight waves walk K in rounds of 2048, a part of one costs a whole one) and the better the chip is filled by k_rows_lds.  us, k_rows_w16m / k_rows_lds:
//   up to 256 blocks   [2048, 2048] 5 rows 5.2 / 6.7, 16 rows 6.4 / 7.3, 32 rows 8.3 / 8.2   [3072, 3072] 8 rows 8.0 / 8.0, 12 rows 8.6 / 8.3   [4096, 4096] 8 rows 8.8 / 9.9, 16 rows 10.4 / 10.4
//                      [2048, 1024] 8 rows 5.1 / 5.8, 16 rows 5.9 / 5.9   [2048, 6144] 5 rows 10.0 / 10.5, 10 rows 11.4 / 11.1
//   up to 512          [8192, 2048] 5 rows 8.3 / 9.7, 12 rows 9.1 / 9.6, 16 rows 10.1 / 9.8   [6144, 1536] 6 rows 7.5 / 7.7, 8 rows 7.9 / 7.8   [4608, 4096] 5 rows 12.1 / 11.2
//   up to 1024         [9216, 3072] 5 rows 16.1 / 14.1   [11264, 2048] 8 rows 11.7 / 11.4   [12320, 4096] 5 rows 21.2 / 19.0   [16384, 2048] 5 rows 13.8 / 14.5, 12 rows 15.4 / 14.6
//   beyond             [16896, 2048] 8 rows 16.0 / 17.9, 12 rows 17.5 / 18.3, 16 rows 19.4 / 18.4   [18944, 4096] 5 rows 27.8 / 29.7, 10 rows 31.3 / 30.3   [24576, 2048] 5 rows 19.5 / 21.2, 10 rows 20.5 / 20.1
//                      [28672, 4096] 5 rows 38.9 / 39.4, 8 rows 41.3 / 39.6   [32768, 2048] 5 rows 24.6 / 25.0, 8 rows 25.6 / 24.9
static bool rows_direct_faster(int M, int K, long blocks) {
    const long rounds = (K + 2047) / 2048, rows = blocks <= 256 ? 26 : blocks <= 512 ? 10 : blocks <= 1024 ? 0 : blocks <= 1280 ? 13 : blocks <= 1600 ? 10 : 0;  // (at K = 2048)
    return M * rounds * rounds * 2048 < rows * K;
}
static bool rows_lds_serves(const RowsArgs &a, int n_max, int k_max, int batches) {
    if (a.M <= 4 || k_max < 1024 || rows_narrow(a, n_max, batches) || a.x_norm || a.merge.splits > 0 || !rows_lds_reaches(a)) return false;
    return a.active || !rows_direct_faster(a.M, k_max, rows_blocks(a, batches));
}
template <class E>
static int rows_launch(const RowsArgs &a, int n_max, int k_max, int batches, hipStream_t st) {
    if (rows_lds_serves(a, n_max, k_max, batches)) return rows_lds_pick<E>(a, n_max, rows_blocks(a, batches), batches, st);
    if (a.M <= 16 || a.active || rows_narrow(a, n_max, batches)) return rows_go<E, 1, 1>(a, n_max, k_max, batches, st);
    int n_all = batches == 1 ? n_max : 0;
    for (int i = 0; i < a.n_mats; ++i) n_all += a.mats[i].N;
    const bool wide = n_all >= 32 * 140;  // two feature blocks per wave where half as many workgroups still fill most of the chip
    if (a.M <= 32) return wide ? rows_go<E, 2, 2>(a, n_max, k_max, batches, st) : rows_go<E, 2, 1>(a, n_max, k_max, batches, st);
    if constexpr (__is_same(E, ElemBF16)) return wide ? rows_go<E, 4, 2>(a, n_max, k_max, batches, st) : rows_go<E, 4, 1>(a, n_max, k_max, batches, st);
    else return pie::fail(PIE_E_SHAPE, "few-row 16-bit Linear: at most 32 rows");
}

size_t rows_weight_bytes(int dtype, int N, int K) {
    return dtype == PIE_F32 ? (size_t)N * ((K + 63) & ~63) * 4 : w16m_size(N, K);
}

int rows_gemm_launch(int dtype, const RowsArgs &a, int batches, hipStream_t st) {
    if (a.M <= 0 || batches <= 0) return PIE_OK;
    PIE_REQUIRE(a.n_mats || (a.m.N > 0 && a.m.K > 0), PIE_E_SHAPE, "row-wise Linear: empty matrix");
    PIE_REQUIRE(batches < 65535 && (!rows_riders(a) || !(a.shared.w || a.active)), PIE_E_SHAPE, "row-wise Linear: too many batches");
    PIE_REQUIRE(a.n_mats == 0 || (a.n_mats == batches && a.n_mats <= ROWS_LIST && !rows_riders(a) && !a.shared.w && !a.active && !a.rows && a.merge.splits <= 0 && !a.x_norm), PIE_E_ARG,
                "row-wise Linear: a list of matrices is a launch of its own");
    int n_max = a.shared.w && a.shared.N > a.m.N ? a.shared.N : a.m.N, k_max = a.shared.w && a.shared.K > a.m.K ? a.shared.K : a.m.K;
    for (int i = 0; i < a.n_mats; ++i) {
        const RowsMat &m = a.mats[i];
        PIE_REQUIRE(m.N > 0 && m.K > 0 && m.ldx % 8 == 0 && pie_aligned(m.x, 16) && pie_aligned(m.w, 16), PIE_E_ALIGN, "row-wise Linear: 16-byte alignment required");
        n_max = i ? std::max(n_max, m.N) : m.N, k_max = i ? std::max(k_max, m.K) : m.K;
    }
    PIE_REQUIRE(!a.x_norm || (dtype == PIE_BF16 && a.M <= 16 && batches == 1 && !a.active && !a.shared.w && !a.rows && a.merge.splits <= 0), PIE_E_SHAPE, "row-wise Linear: too many rows to norm on the way in");
    if (dtype == PIE_F32) {
        RowsArgs f = a;
        rows_slice(f, (unsigned)((n_max + 15) / 16), batches);
        const dim3 grid((unsigned)((n_max + 15) / 16), (unsigned)(batches + rows_riders(a) * f.ride_slices), (unsigned)((a.M + 15) / 16));
        hipLaunchKernelGGL(k_rows_f32, grid, dim3(256), 0, st, f);
        PIE_LAUNCH_CHECK();
        return PIE_OK;
    }
    PIE_REQUIRE(a.merge.splits <= 64 && (a.merge.splits <= 0 || (a.merge.M == a.M && a.M <= MERGE_ROWS && a.merge.ldr <= MERGE_LDR && a.merge.ldr % 8 == 0 && !a.active && !a.rows)), PIE_E_SHAPE,
                "row-wise Linear: too many rows or columns to merge key splits on the way in");
    PIE_REQUIRE(a.m.ldx % 8 == 0 && a.x_batch % 8 == 0 && pie_aligned(a.m.x, 16) && pie_aligned(a.m.w, 16), PIE_E_ALIGN, "row-wise Linear: 16-byte alignment required");
    return rows_launch<ElemBF16>(a, n_max, k_max, batches, st);
}

int rows_w16_launch(int dtype, const void *w16m, const void *x, int M, int N, int K, void *y, const void *bias, bool swiglu, hipStream_t st) {
    PIE_REQUIRE(M >= 1 && M <= ROWS_W16_MAX && N > 0 && K > 0 && K % 64 == 0, PIE_E_SHAPE, "few-row 16-bit Linear: 1 to 32 rows, in_features % 64 == 0");
    PIE_REQUIRE(dtype == PIE_BF16 || dtype == PIE_F16, PIE_E_ARG, "few-row 16-bit Linear: dtype must be PIE_BF16 or PIE_F16");
    PIE_REQUIRE(pie_aligned(x, 16) && pie_aligned(w16m, 16), PIE_E_ALIGN, "few-row 16-bit Linear: 16-byte alignment required");
    PIE_REQUIRE(!swiglu || N % 2 == 0, PIE_E_SHAPE, "few-row 16-bit Linear: the fused activation pairs columns");
    RowsArgs a = {};
    a.m = {(const char *)w16m, N, K, x, K, y, swiglu ? N / 2 : N};
    a.M = M, a.epi = swiglu ? ROWS_SWIGLU : ROWS_LINEAR, a.bias = (const u16 *)bias;
    return dtype == PIE_F16 ? rows_launch<ElemF16>(a, N, K, 1, st) : rows_launch<ElemBF16>(a, N, K, 1, st);
}

extern "C" {

size_t pie_stack_weight_bytes(int dtype, int N, int K) {
    return N > 0 && K > 0 && (dtype == PIE_BF16 || dtype == PIE_F32) ? rows_weight_bytes(dtype, N, K) : 0;
}

int pie_stack_linear_kernel(int M, int N, int K, int ldx, int x_rows) {
    PIE_REQUIRE(M > 0 && N > 0 && K > 0 && ldx >= K && x_rows >= -1, -1, "pie_stack_linear_kernel: bad sizes");
    RowsArgs a = {};
    const int any = 0;
    a.m.N = N, a.m.K = K, a.m.ldx = ldx, a.M = M, a.rows = x_rows > 0 ? &any : nullptr, a.x_rows = x_rows;
    if (x_rows < 0) a.mats[0] = a.m, a.n_mats = 1, a.m = {};
    return rows_lds_serves(a, N, K, 1);
}

int pie_stack_pack_weight(const void *w, int N, int K, int dtype, void *packed, void *stream) {
    PIE_REQUIRE(w && packed, PIE_E_ARG, "pie_stack_pack_weight: null pointer");
    PIE_REQUIRE(N > 0 && K > 0, PIE_E_SHAPE, "pie_stack_pack_weight: empty matrix");
    if (dtype == PIE_BF16) return pie_repack_w16m(w, N, K, PIE_BF16, packed, stream);
    PIE_REQUIRE(dtype == PIE_F32, PIE_E_ARG, "pie_stack_pack_weight: dtype must be PIE_BF16 or PIE_F32");
    const int Kp = (K + 63) & ~63;
    hipLaunchKernelGGL(k_pack_f32, dim3((unsigned)(((size_t)N * Kp + 255) / 256)), dim3(256), 0, (hipStream_t)stream, (const u16 *)w, N, K, Kp, (float *)packed);
    PIE_LAUNCH_CHECK();
    return PIE_OK;
}

}  // extern "C"
