// prefill.hip -- batched prompt processing: Model.__call__(inputs[1, L], cache) for L > 1
// (models/llama/language.py:199-210 with the causal mask of models/base.py:18-53), SURVEY.md 8 row f1.
//
// At L > 1 the reference's nn.QuantizedLinear reaches MLX's matrix kernels (qmm), which dequantise the int4 block to T
// and feed a T x T -> fp32 MMA; the vector kernels (qmv, exact fp32 affine math) serve only the few-row case.  This file
// follows that split: prompts of prefill_min_rows() tokens or more run here, shorter ones as iterated decode steps.
//
// MI355X design, per weight format (no library GEMM anywhere: the hipBLASLt path of rounds 1-4 was removed in round 5):
//   * int4 g=64 modules multiply their 4-bit W4M tiles directly (w4m_gemm.hip: k_w4r_gemm up to 256 rows, k_w4l2_gemm beyond);
//   * dense modules, and int8 / group-32 modules, multiply a 16-bit copy in W16M tiles (w16_gemm.hpp: k_w16l_gemm, the weights
//     straight into MFMA fragment registers, x through LDS-DMA) -- dense ones tiled from their W16S units, quantised ones from
//     k_dequant_w4s / k_dequant_w8s (the mx.dequantize arithmetic: T(fp32(s*q) + b)); 288 GB of HBM keep the copies resident;
//   * hand-written HIP for everything around it: RMSNorm rows, RoPE + cache append from the packed q|k|v rows, causal
//     attention (MFMA flash kernel), the split merge, SwiGLU on the interleaved gate/up rows, residual adds.
// The chunk is bounded (PIE_KNOB_PREFILL_CHUNK, default 4096 rows: ~0.6 GB of activation scratch on the 8B model).
#include <cstdlib>
#include <map>
#include <mutex>

#include "decoder.hpp"
#include "prefill_attn.hpp"
#include "stack_types.hpp"  // rows_w16_launch

size_t w16m_size(int N, int K);  // bytes of a matrix as W16M and as W4M tiles
size_t w4m_bytes(int N, int K);

// ---------------------------------------------------------------- kernels
// W4S -> T row-major [N, K]; one thread per code word (8 weights, 16 B out).  Same arithmetic as k_dequantize_w4g64.
template <class T, bool G32 = false>  // G32: W4S32 units (two {scale | bias} words per lane: code piece j is its own 32-wide group)
__global__ void k_dequant_w4s(const u32 *packed, int N, int K, int ns, u16 *out) {
    const size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int wpr = K >> 3;  // words per row
    if (idx >= (size_t)N * wpr) return;
    const int r = (int)(idx / wpr), wk = (int)(idx % wpr);
    const int g = wk >> 3, lane = (r & 1) * 32 + (g & 31), j = (wk & 7) >> 2, t = wk & 3;
    const u32 *unit = packed + ((size_t)(r >> 1) * ns + (g >> 5)) * ((G32 ? W4S32_UNIT_BYTES : W4S_UNIT_BYTES) / 4);
    const u32 word = unit[j * 256 + lane * 4 + t], sb = G32 ? unit[512 + 2 * lane + j] : unit[512 + lane];
    const float s = lo_f32<T>(sb), b = hi_f32<T>(sb);
    u32 o[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {  // codes (2i, 2i+1) sit in the low / high half at nibble i (the W4S nibble order)
        const float lo = __fadd_rn(__fmul_rn(s, (float)((word >> (4 * i)) & 0xFu)), b);
        const float hi = __fadd_rn(__fmul_rn(s, (float)((word >> (16 + 4 * i)) & 0xFu)), b);
        o[i] = pack2<T>(lo, hi);
    }
    *reinterpret_cast<uint4 *>(out + (size_t)r * K + (size_t)wk * 8) = make_uint4(o[0], o[1], o[2], o[3]);
}

// W2S -> T row-major [N, K]; one thread per code word (16 weights, 32 B out).
template <class T>
__global__ void k_dequant_w2s(const u32 *packed, int N, int K, int ns, u16 *out) {
    const size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int wpr = K >> 4;  // words per row
    if (idx >= (size_t)N * wpr) return;
    const int r = (int)(idx / wpr), wk = (int)(idx % wpr);
    const int g = wk >> 2, lane = (r & 1) * 32 + (g & 31), t = wk & 3;
    const u32 *unit = packed + ((size_t)(r >> 1) * ns + (g >> 5)) * (W2S_UNIT_BYTES / 4);
    const u32 word = unit[lane * 4 + t], sb = unit[256 + lane];
    const float s = lo_f32<T>(sb), b = hi_f32<T>(sb);
    u32 o[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {  // codes (2j, 2j+1) of the word sit at bits 2j of the low / high half (the W2S order)
        const float lo = __fadd_rn(__fmul_rn(s, (float)((word >> (2 * j)) & 0x3u)), b);
        const float hi = __fadd_rn(__fmul_rn(s, (float)((word >> (16 + 2 * j)) & 0x3u)), b);
        o[j] = pack2<T>(lo, hi);
    }
    uint4 *dst = reinterpret_cast<uint4 *>(out + (size_t)r * K + (size_t)wk * 16);
    dst[0] = make_uint4(o[0], o[1], o[2], o[3]), dst[1] = make_uint4(o[4], o[5], o[6], o[7]);
}

// W6S -> T row-major [N, K]; one thread per low-plane code word (8 weights, 16 B out): q = low nibble + 16 x the high plane's two bits.
template <class T>
__global__ void k_dequant_w6s(const u32 *packed, int N, int K, int ns, u16 *out) {
    const size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int wpr = K >> 3;
    if (idx >= (size_t)N * wpr) return;
    const int r = (int)(idx / wpr), wk = (int)(idx % wpr);
    const int g = wk >> 3, lane = (r & 1) * 32 + (g & 31), w4 = wk & 7, j = w4 >> 2, t = w4 & 3;
    const u32 *unit = packed + ((size_t)(r >> 1) * ns + (g >> 5)) * (W6S_UNIT_BYTES / 4);
    const u32 word = unit[j * 256 + lane * 4 + t], sb = unit[768 + lane];
    const u32 hiw = unit[512 + lane * 4 + (w4 >> 1)] >> (8 * (w4 & 1));  // codes 8 w4 .. + 7 = pairs 4 (w4 & 1) .. + 3 of high word w4 >> 1
    const float s = lo_f32<T>(sb), b = hi_f32<T>(sb);
    u32 o[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const u32 qa = ((word >> (4 * i)) & 0xFu) | (((hiw >> (2 * i)) & 0x3u) << 4), qb = ((word >> (16 + 4 * i)) & 0xFu) | (((hiw >> (16 + 2 * i)) & 0x3u) << 4);
        o[i] = pack2<T>(__fadd_rn(__fmul_rn(s, (float)qa), b), __fadd_rn(__fmul_rn(s, (float)qb), b));
    }
    *reinterpret_cast<uint4 *>(out + (size_t)r * K + (size_t)wk * 8) = make_uint4(o[0], o[1], o[2], o[3]);
}

// W8S -> T row-major [N, K]; one thread per code word (4 weights, 8 B out).
template <class T, bool G32 = false>  // G32: W8S32 units (code pieces 0-1 / 2-3 are two 32-wide groups)
__global__ void k_dequant_w8s(const u32 *packed, int N, int K, int ns, u16 *out) {
    const size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int wpr = K >> 2;
    if (idx >= (size_t)N * wpr) return;
    const int r = (int)(idx / wpr), wk = (int)(idx % wpr);
    const int g = wk >> 4, lane = (r & 1) * 32 + (g & 31), j = (wk & 15) >> 2, t = wk & 3;
    const u32 *unit = packed + ((size_t)(r >> 1) * ns + (g >> 5)) * ((G32 ? W8S32_UNIT_BYTES : W8S_UNIT_BYTES) / 4);
    const u32 word = unit[j * 256 + lane * 4 + t], sb = G32 ? unit[1024 + 2 * lane + (j >> 1)] : unit[1024 + lane];
    const float s = lo_f32<T>(sb), b = hi_f32<T>(sb);
    // stored byte order (c0, c2, c1, c3)
    const float q0 = __fadd_rn(__fmul_rn(s, (float)(word & 0xFFu)), b), q2 = __fadd_rn(__fmul_rn(s, (float)((word >> 8) & 0xFFu)), b);
    const float q1 = __fadd_rn(__fmul_rn(s, (float)((word >> 16) & 0xFFu)), b), q3 = __fadd_rn(__fmul_rn(s, (float)(word >> 24)), b);
    *reinterpret_cast<uint2 *>(out + (size_t)r * K + (size_t)wk * 4) = make_uint2(pack2<T>(q0, q1), pack2<T>(q2, q3));
}

// The head of a pass, one workgroup per row: h = embed_tokens(ids) (language.py:176; or the caller's embeddings), the first layer's input_layernorm, and (cos, sin) of the row's rotary
// angles -- the angle of pair ii at position p is the same for all heads and all layers, and sincosf on arguments up to ~1e5 rad (argument reduction) was most of
// k_rope_append_rows' 8 us per layer.  Three launches of nothing but latency took 14.3 us (traced) in a step of 8 rows, this one 5.8.
// Its chain is id, code, scale, norm; the angles are computed while the row is on its way.
struct PassRowsArgs {
    const int *ids;       // nullptr: embeds [M, H]
    const u16 *embeds;
    const void *table;    // [V, H] of T (FMT 0), or packed codes, scales and biases
    const u16 *scales, *biases;
    int V, H, group_shift;  // (group of 1 << group_shift columns)
    const float *freqs;
    const DecState *state;  // row m at state->pos + m, or
    const int *ctx_len;     // at ctx_len[m] - 1
    int half;
    float *cs;
    const u16 *norm_w;    // nullptr: no norm
    float eps;
    u16 *x, *xn;
    int rows, *total;  // workgroup `rows`, where there is one: the sum of ctx_len that are above 0 (k_attn_step, whose workgroups each summed them: two layers of 4096 rows, 32 / 8 heads of 128, 2653 us, 889 now)
};
template <class T, int FMT>  // 0: rows of T, 4 / 8: bits per code
__global__ void __launch_bounds__(256) k_pass_rows(const PassRowsArgs a) {
    __shared__ float red[4];
    const int m = blockIdx.x, H = a.H;
    if (m == a.rows) {
        __shared__ int sums[4];
        int sum = 0;
        for (int r = threadIdx.x; r < a.rows; r += 256) sum += max(a.ctx_len[r], 0);
#pragma unroll
        for (int i = 1; i < 64; i <<= 1) sum += __shfl_xor(sum, i);
        if ((threadIdx.x & 63) == 0) sums[threadIdx.x >> 6] = sum;
        __syncthreads();
        if (threadIdx.x == 0) *a.total = (sums[0] + sums[1]) + (sums[2] + sums[3]);
        return;
    }
    size_t id = m;
    if (a.ids) {
        const int i = a.ids[m];
        id = i < 0 ? 0 : i >= a.V ? a.V - 1 : i;
    }
    const u16 *rows = (a.ids ? (const u16 *)a.table : a.embeds) + id * H, *scale = a.scales + (id * H >> a.group_shift), *bias = a.biases + (id * H >> a.group_shift);
    const u32 *codes = (const u32 *)a.table + id * (H * FMT / 32);
    auto octet = [&](int i) {  // columns i .. i + 7
        if (FMT == 0) return *reinterpret_cast<const uint4 *>(rows + i);
        const float s = T::to_f32(scale[i >> a.group_shift]), b = T::to_f32(bias[i >> a.group_shift]);
        if (FMT == 4) return dequant_word_u4<T>(codes[i >> 3], s, b);
        u32 o[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {  // separate multiply and add roundings, as in k_embedding_w4g64
            const u32 w = codes[(i >> 2) + (k >> 1)] >> (16 * (k & 1));
            o[k] = pack2<T>(__fadd_rn(__fmul_rn(s, (float)(w & 0xFFu)), b), __fadd_rn(__fmul_rn(s, (float)((w >> 8) & 0xFFu)), b));
        }
        return make_uint4(o[0], o[1], o[2], o[3]);
    };
    u16 *xr = a.x + (size_t)m * H, *yr = a.xn + (size_t)m * H;
    constexpr int KEPT = 4;  // octets that a thread keeps for the norm: H <= 8192; it reads the rest again
    uint4 hv[KEPT];
    float ssq = 0.0f;
    auto square = [&](const uint4 &q) {
        const u32 v[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float lo = lo_f32<T>(v[j]), hi = hi_f32<T>(v[j]);
            ssq = fmaf(lo, lo, ssq), ssq = fmaf(hi, hi, ssq);
        }
    };
#pragma unroll
    for (int p = 0; p < KEPT; ++p) {
        const int i = (threadIdx.x + p * 256) * 8;
        if (i < H) hv[p] = octet(i);
    }
    __builtin_amdgcn_sched_barrier(0);  // the angles while the row is on its way
    if ((int)threadIdx.x >= 256 - a.half) {
        const int ii = threadIdx.x - (256 - a.half);
        int pos = a.ctx_len ? a.ctx_len[m] - 1 : a.state->pos + m;
        pos = pos < 0 ? 0 : pos;
        float sn, c;
        sincosf((float)pos * (1.0f / a.freqs[ii]), &sn, &c);
        *reinterpret_cast<float2 *>(a.cs + ((size_t)m * a.half + ii) * 2) = make_float2(c, sn);
    }
#pragma unroll
    for (int p = 0; p < KEPT; ++p) {
        const int i = (threadIdx.x + p * 256) * 8;
        if (i < H) *reinterpret_cast<uint4 *>(xr + i) = hv[p], square(hv[p]);
    }
    for (int i = (threadIdx.x + KEPT * 256) * 8; i < H; i += 256 * 8) {
        const uint4 q = octet(i);
        *reinterpret_cast<uint4 *>(xr + i) = q, square(q);
    }
    if (!a.norm_w) return;
    ssq = wave_sum(ssq);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = ssq;
    __syncthreads();
    const float inv = 1.0f / sqrtf((red[0] + red[1] + red[2] + red[3]) / (float)H + a.eps);
    auto norm = [&](const uint4 &q, int i) {  // k_rms_norm's arithmetic
        const uint4 g = *reinterpret_cast<const uint4 *>(a.norm_w + i);
        const u32 vv[4] = {q.x, q.y, q.z, q.w}, gg[4] = {g.x, g.y, g.z, g.w};
        u32 o[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) o[j] = pack2<T>(round_T<T>(lo_f32<T>(vv[j]) * inv) * lo_f32<T>(gg[j]), round_T<T>(hi_f32<T>(vv[j]) * inv) * hi_f32<T>(gg[j]));
        *reinterpret_cast<uint4 *>(yr + i) = make_uint4(o[0], o[1], o[2], o[3]);
    };
#pragma unroll
    for (int p = 0; p < KEPT; ++p) {
        const int i = (threadIdx.x + p * 256) * 8;
        if (i < H) norm(hv[p], i);
    }
    for (int i = (threadIdx.x + KEPT * 256) * 8; i < H; i += 256 * 8) norm(octet(i), i);
}

// A K-split many-row GEMM (w4m_gemm.hip) leaves S fp32 partial slabs [S][M][N]; its consumer can form the Linear's output itself --
// the slabs summed in slab order, then the one rounding to T: exactly k_w4l_reduce's arithmetic -- which saves that launch and the
// round trip of y through memory (prompts of 33..~700 rows split K; a launch is ~5 us of a 150-300 us layer there).
struct W4lSlabs {
    const float *part = nullptr;
    int S = 0;
    size_t MN = 0;
};
// RoPE (llama/utils.py:42-50, offset = cache.offset) + cache append (reusable.py:134-137) for M rows of the packed
// q|k|v projection: packed columns (2i, 2i+1) of a q/k head are its dims (i, i + D/2); v columns are natural.
// A thread takes eight packed columns (four pairs) at a time: 16 bytes in, twice 8 (or once 16) out; as many workgroups per row (blockIdx.y) as leave a thread one round where rows are few.
// (A pair per thread, stores of two bytes and two divisions by the head size took, traced, at 4096 rows of Llama-3-8B 31.4 us, now
// 19.1 = 5.3 TB/s; 509 rows 10.6 -> 5.7; 37 rows of slabs 5.7 -> 4.5.)
// SLAB / I8: the two optional input / output forms as compile-time switches -- carried as run-time branches they cost the plain
// 4096-row launch 7.6 us (34.4 vs 26.8 us per layer)
struct RopeRowsArgs {
    const u16 *qkv;                       // [M, n_cols], or
    const float *part;                    // (SLAB) the fp32 slabs of a K-split GEMM (W4lSlabs)
    int S, n_cols;
    size_t MN;
    const DecState *state;                // row m continues the decoder's one sequence at state->pos + m, or
    const int *ctx_len;                   // (multi-sequence step) row m is its own sequence at position ctx_len[m] - 1 with its own block table row
    const unsigned long long *kv_table;   // the layers' K and V buffers or slab bases, or
    u16 *slab;                            // this layer's slab
    int layer, n_layers, n_heads, n_kv_heads, hd_shift, traditional;  // heads of 1 << hd_shift: 64 or 128
    u16 *q_out;
    const int *block_table, *row_seq;     // row m belongs to sequence row_seq[m] (several prompts in one pass), else to sequence m
    int bt_stride, n_pages;
    const float *rope_cs;                 // k_pass_rows
    u16 *kc, *vc;                         // nullable: the rotated K and the V rows, also to contiguous [n_kv_heads, rows, HD] (what the attention of a varlen pass reads)
    size_t i8_page_bytes;                 // (I8, with slab) int8 pages with per-head fp16 scales (paged_i8.hip): the rotated K / the V element x, already rounded to T, is stored as
};                                        // clamp(rint(x / s), -127, 127) with the scale of (its page, its kv-head)
template <class T, bool SLAB = false, bool I8 = false>
__global__ void __launch_bounds__(256) k_rope_append_rows(const RopeRowsArgs a) {
    const int m = blockIdx.x, pos = a.ctx_len ? a.ctx_len[m] - 1 : a.state->pos + m, HD = 1 << a.hd_shift, half = HD >> 1;
    if (pos < 0) return;  // idle slot of the batch
    int cap = a.ctx_len ? 64 : a.state->cap, kvrow = pos;
    const int q_cols = a.n_heads * HD, k_cols = a.n_kv_heads * HD, n_rows = gridDim.x;
    u16 *kdst = a.slab ? a.slab : reinterpret_cast<u16 *>(a.kv_table[a.layer]);
    u16 *vdst = a.slab ? a.slab + (size_t)a.n_kv_heads * 64 * HD : reinterpret_cast<u16 *>(a.kv_table[a.n_layers + a.layer]);
    char *page8 = nullptr;  // int8 pages: this row's page
    if (a.block_table) {  // paged KV: the row goes to slot pos % 64 of page block_table[pos / 64]
        const int *bt = a.block_table + (size_t)(a.row_seq ? a.row_seq[m] : m) * a.bt_stride;
        const unsigned pg = min((unsigned)bt[pos >> 6], (unsigned)a.n_pages - 1u);
        const size_t pg_off = (size_t)pg * 2 * 64 * a.n_kv_heads * HD;
        kdst += pg_off, vdst += pg_off, cap = 64, kvrow = pos & 63;
        if (I8 && a.i8_page_bytes && a.slab) page8 = reinterpret_cast<char *>(a.slab) + (size_t)pg * a.i8_page_bytes;
    }
    const size_t blk8 = (size_t)a.n_kv_heads * 64 * HD;
    auto q8 = [](float x, float sc) {
        float q = rintf(x / sc);
        q = q < -127.0f ? -127.0f : (q > 127.0f ? 127.0f : q);
        return (signed char)(q == q ? (int)q : 0);
    };
    auto f16f = [](u16 h) { return (float)__builtin_bit_cast(_Float16, h); };
    for (int R = (blockIdx.y * blockDim.x + threadIdx.x) * 8; R < a.n_cols; R += gridDim.y * blockDim.x * 8) {
        u32 pr[4];
        if constexpr (SLAB) {
            const size_t i[2] = {(size_t)m * a.n_cols + R, (size_t)m * a.n_cols + R + 4};
            float4 f[2];
            slab_sum<float4, 2>(a.part, a.S, a.MN, i, f);
            pr[0] = pack2<T>(f[0].x, f[0].y), pr[1] = pack2<T>(f[0].z, f[0].w), pr[2] = pack2<T>(f[1].x, f[1].y), pr[3] = pack2<T>(f[1].z, f[1].w);
        } else {
            const uint4 v = *reinterpret_cast<const uint4 *>(a.qkv + (size_t)m * a.n_cols + R);
            pr[0] = v.x, pr[1] = v.y, pr[2] = v.z, pr[3] = v.w;
        }
        const bool is_q = R < q_cols, is_k = !is_q && R < q_cols + k_cols;
        const int rr = is_q ? R : is_k ? R - q_cols : R - q_cols - k_cols, head = rr >> a.hd_shift, col = rr & (HD - 1);  // (eight columns lie in one head)
        if (is_q || is_k) {
            const int ii = col >> 1;
            const float4 c0 = *reinterpret_cast<const float4 *>(a.rope_cs + ((size_t)m * half + ii) * 2), c1 = *reinterpret_cast<const float4 *>(a.rope_cs + ((size_t)m * half + ii) * 2 + 4);
            const float cs[4] = {c0.x, c0.z, c1.x, c1.z}, sn[4] = {c0.y, c0.w, c1.y, c1.w};
            u16 o0[4], o1[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float ra = lo_f32<T>(pr[j]), rb = hi_f32<T>(pr[j]);
                o0[j] = T::from_f32(__fsub_rn(__fmul_rn(ra, cs[j]), __fmul_rn(rb, sn[j]))), o1[j] = T::from_f32(__fadd_rn(__fmul_rn(ra, sn[j]), __fmul_rn(rb, cs[j])));
            }
            auto put = [&](u16 *dst) {
                if (a.traditional)
                    *reinterpret_cast<uint4 *>(dst + 2 * ii) =
                        make_uint4(o0[0] | (u32)o1[0] << 16, o0[1] | (u32)o1[1] << 16, o0[2] | (u32)o1[2] << 16, o0[3] | (u32)o1[3] << 16);
                else {
                    *reinterpret_cast<uint2 *>(dst + ii) = make_uint2(o0[0] | (u32)o0[1] << 16, o0[2] | (u32)o0[3] << 16);
                    *reinterpret_cast<uint2 *>(dst + ii + half) = make_uint2(o1[0] | (u32)o1[1] << 16, o1[2] | (u32)o1[3] << 16);
                }
            };
            if (is_q) put(a.q_out + ((size_t)m * a.n_heads + head) * HD);
            else if (I8 && page8) {
                const float sk = f16f(reinterpret_cast<const u16 *>(page8 + 2 * blk8)[head]);
                signed char *kb = reinterpret_cast<signed char *>(page8) + ((size_t)head * 64 + kvrow) * HD;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    kb[a.traditional ? 2 * (ii + j) : ii + j] = q8(T::to_f32(o0[j]), sk);
                    kb[a.traditional ? 2 * (ii + j) + 1 : ii + j + half] = q8(T::to_f32(o1[j]), sk);
                }
            } else put(kdst + ((size_t)head * cap + kvrow) * HD);
            if (a.kc && is_k) put(a.kc + ((size_t)head * n_rows + m) * HD);
        } else {
            const uint4 v = make_uint4(pr[0], pr[1], pr[2], pr[3]);
            if (I8 && page8) {
                const float sv = f16f(reinterpret_cast<const u16 *>(page8 + 2 * blk8)[a.n_kv_heads + head]);
                signed char *vb = reinterpret_cast<signed char *>(page8) + blk8 + ((size_t)head * 64 + kvrow) * HD + col;
#pragma unroll
                for (int j = 0; j < 4; ++j) vb[2 * j] = q8(lo_f32<T>(pr[j]), sv), vb[2 * j + 1] = q8(hi_f32<T>(pr[j]), sv);
            } else *reinterpret_cast<uint4 *>(vdst + ((size_t)head * cap + kvrow) * HD + col) = v;
            if (a.vc) *reinterpret_cast<uint4 *>(a.vc + ((size_t)head * n_rows + m) * HD + col) = v;
        }
    }
}
// nn.silu(gate) * up (language.py:127) on interleaved columns (2i, 2i+1) = (gate_i, up_i); 4 outputs per thread.
template <class T>
__global__ void k_swiglu_rows(const u16 *gu, size_t n_out, u16 *act) {
    const size_t i = ((size_t)blockIdx.x * blockDim.x + threadIdx.x) * 4;
    if (i >= n_out) return;  // n_out is a multiple of 4 (inter % 64 == 0)
    const uint4 v = *reinterpret_cast<const uint4 *>(gu + 2 * i);
    const u32 w[4] = {v.x, v.y, v.z, v.w};
    u16 o[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const float g = lo_f32<T>(w[k]), u = hi_f32<T>(w[k]);
        o[k] = T::from_f32(round_T<T>(g / (1.0f + expf(-g))) * u);
    }
    *reinterpret_cast<uint2 *>(act + i) = make_uint2((u32)o[0] | ((u32)o[1] << 16), (u32)o[2] | ((u32)o[3] << 16));
}

// y[m, :] = T(y[m, :] + b) for the Linear biases (y already T-rounded by the GEMM); 8 columns per thread, N % 8 == 0.
template <class T>
__global__ void k_bias_rows(u16 *y, const u16 *b, size_t n8, int N8) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n8) return;
    const uint4 v = reinterpret_cast<const uint4 *>(y)[i], bb = reinterpret_cast<const uint4 *>(b)[i % N8];
    const u32 a[4] = {v.x, v.y, v.z, v.w}, c[4] = {bb.x, bb.y, bb.z, bb.w};
    u32 o[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) o[k] = pack2<T>(lo_f32<T>(a[k]) + lo_f32<T>(c[k]), hi_f32<T>(a[k]) + hi_f32<T>(c[k]));
    reinterpret_cast<uint4 *>(y)[i] = make_uint4(o[0], o[1], o[2], o[3]);
}

// h = x + r (language.py:151,153) fused with the RMSNorm that follows it (language.py:137-141): x <- T(x + r) in place,
// xn <- w * T(h * rsqrt(mean(h^2) + eps)).  One workgroup per row, eight columns per thread (H / 8 threads, H <= 8192): the row stays in registers.
//
// A step's few rows wait for memory, not for bandwidth: x, the norm's weights, the bias and SLABS slabs are all asked for before the first of them is used.  (256 threads that took
// their octets one after the other, the slabs four at a time and the weights behind the barrier waited four to six times.)  Llama-3-8B int4, four layers: a step of 8 rows 5165 -> 5010 us for 16 steps, of 32 rows
// 7368 -> 7257; bf16, 8 rows 8539 -> 8312; 509 and 4096 rows level.
template <class T, int SLABS>  // 0: r holds the Linear's output; else its fp32 slabs (W4lSlabs), SLABS of them in flight
__global__ void __launch_bounds__(1024) k_add_rms_norm_rows(u16 *x, const u16 *r, const u16 *w, float eps, int H, u16 *xn, const u16 *bias, const float *part, int S, size_t MN) {
    __shared__ float red[16];
    const int i = threadIdx.x * 8;
    const size_t at = (size_t)blockIdx.x * H + i;
    u32 hv[4] = {0, 0, 0, 0};
    uint4 g = make_uint4(0, 0, 0, 0);
    float ssq = 0.0f;
    if (i < H) {
        const uint4 a = *reinterpret_cast<const uint4 *>(x + at);
        g = *reinterpret_cast<const uint4 *>(w + i);
        uint4 b;
        if constexpr (SLABS > 0) {  // r = T(T(sum of the slabs) + bias)
            uint4 bb = make_uint4(0, 0, 0, 0);
            if (bias) bb = *reinterpret_cast<const uint4 *>(bias + i);
            const size_t o[2] = {at, at + 4};
            float4 f[2];
            slab_sum<float4, 2, SLABS>(part, S, MN, o, f);
            float v[8] = {f[0].x, f[0].y, f[0].z, f[0].w, f[1].x, f[1].y, f[1].z, f[1].w};
            if (bias) {
                const u32 bw[4] = {bb.x, bb.y, bb.z, bb.w};
#pragma unroll
                for (int j = 0; j < 4; ++j) v[2 * j] = round_T<T>(v[2 * j]) + lo_f32<T>(bw[j]), v[2 * j + 1] = round_T<T>(v[2 * j + 1]) + hi_f32<T>(bw[j]);
            }
            b = make_uint4(pack2<T>(v[0], v[1]), pack2<T>(v[2], v[3]), pack2<T>(v[4], v[5]), pack2<T>(v[6], v[7]));
        } else b = *reinterpret_cast<const uint4 *>(r + at);
        const u32 av[4] = {a.x, a.y, a.z, a.w}, bv[4] = {b.x, b.y, b.z, b.w};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            hv[j] = pack2<T>(lo_f32<T>(av[j]) + lo_f32<T>(bv[j]), hi_f32<T>(av[j]) + hi_f32<T>(bv[j]));
            const float lo = lo_f32<T>(hv[j]), hi = hi_f32<T>(hv[j]);
            ssq = fmaf(lo, lo, ssq), ssq = fmaf(hi, hi, ssq);
        }
        *reinterpret_cast<uint4 *>(x + at) = make_uint4(hv[0], hv[1], hv[2], hv[3]);
    }
    ssq = wave_sum(ssq);
    const int waves = blockDim.x >> 6;
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = ssq;
    __syncthreads();
    float sum = red[0];
    for (int k = 1; k < waves; ++k) sum += red[k];
    if (i >= H) return;
    const float inv = 1.0f / sqrtf(sum / (float)H + eps);
    const u32 gg[4] = {g.x, g.y, g.z, g.w};
    u32 o[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) o[j] = pack2<T>(round_T<T>(lo_f32<T>(hv[j]) * inv) * lo_f32<T>(gg[j]), round_T<T>(hi_f32<T>(hv[j]) * inv) * hi_f32<T>(gg[j]));
    *reinterpret_cast<uint4 *>(xn + at) = make_uint4(o[0], o[1], o[2], o[3]);
}

template <class T>
static int add_rms_norm_rows(u16 *x, const u16 *r, const void *w, float eps, int M, int H, int dtype, u16 *xn, hipStream_t st,
                             const void *bias = nullptr, const W4lSlabs *sl = nullptr) {
    const bool slabs = sl && sl->S > 1;  // (linear_rows only hands out slabs for H <= 8192)
    if (!slabs && H > 8192) {  // wider than the register-resident row: the two separate kernels
        const int rc = pie_add(x, r, (size_t)M * H, dtype, x, st);
        return rc ? rc : pie_rms_norm(x, w, eps, M, H, dtype, xn, st);
    }
    const dim3 block((unsigned)((H / 8 + 63) & ~63));
    if (!slabs) hipLaunchKernelGGL((k_add_rms_norm_rows<T, 0>), dim3(M), block, 0, st, x, r, (const u16 *)w, eps, H, xn, (const u16 *)nullptr, (const float *)nullptr, 0, (size_t)0);
    else if (sl->S <= 4) hipLaunchKernelGGL((k_add_rms_norm_rows<T, 3>), dim3(M), block, 0, st, x, r, (const u16 *)w, eps, H, xn, (const u16 *)bias, sl->part, sl->S, sl->MN);
    else hipLaunchKernelGGL((k_add_rms_norm_rows<T, 7>), dim3(M), block, 0, st, x, r, (const u16 *)w, eps, H, xn, (const u16 *)bias, sl->part, sl->S, sl->MN);
    PIE_LAUNCH_CHECK();
    return PIE_OK;
}

__global__ void k_add_pos(DecState *s, int delta) { s->pos += delta; }

// ---------------------------------------------------------------- scratch
struct PrefillScratch {
    int rows = 0;           // chunk capacity (rows)
    size_t w_elems = 0;     // capacity of the dequantised-weight buffer (elements)
    u16 *wT = nullptr, *wM = nullptr, *x = nullptr, *xn = nullptr, *qkv = nullptr, *q = nullptr, *attn = nullptr, *gu = nullptr, *act = nullptr, *r = nullptr;
    float *rope_cs = nullptr;
    int *arrived = nullptr;   // k_attn_step's counters, [rows, n_kv_heads], and behind them
    int *total = nullptr;     // the sum of a batch step's lengths
    u16 *kc = nullptr, *vc = nullptr;  // [n_kv_heads, rows, head_dim]: this pass's K / V rows, contiguous (several prompts in one pass)
    float *part_acc = nullptr, *part_ml = nullptr;  // sums of rows whose decode attention is split: sized by what takes them, not by the rows of a prompt
    size_t parts = 0;                               // their capacity in (row, split)s
    // Resident T copies of the layer matrices, keyed by the packed-weight pointer: the per-chunk dequantisation moves
    // 4.6 B per parameter (7 ms of a 10.8 ms 128-token prefill on the 8B model) for 2 B per parameter of HBM; kept when
    // that is a small share of the free memory (PIE_KNOB_PREFILL_RESIDENT overrides), built on first use.
    std::map<const void *, u16 *> resident;
    // W4M (W8M) tile copies (w4m_gemm.hip) of int4 (int8) matrices: 0.5625 (1.0625) B per weight each
    struct Tiles { void *p; size_t bytes; bool wide; };  // wide: some scale is too large for k_w4a_gemm (w4m_wide_scales)
    std::map<const void *, Tiles> resident_w4m;
    LogitStat *tail_stats = nullptr;  // fused few-sequence step: the lm_head GEMV's tail partials, one per wave and row; other rows' tiles (RowStat) where the tail takes two launches
    size_t tail_entries = 0;           // its capacity in entries
    // Captured multi-sequence step (pie_decoder_step_batch with PIE_STEP_GRAPH): valid while the caller's buffers (key) and every
    // device allocation baked into the launches (alloc_gen) stay what they were at capture time.
    unsigned alloc_gen = 0;
    hipGraphExec_t batch_graph = nullptr;
    std::vector<uintptr_t> batch_key, warm_key;
    unsigned batch_gen = 0, warm_gen = 0;
    bool batch_form = false;  // batch_fused() of the captured step
    void *w4l_ws = nullptr;   // fp32 partial tiles of the K-split prompt GEMM (w4m_gemm.hip)
    size_t w4l_ws_bytes = 0;
    float *attn_part = nullptr;  // sums of prompt attention split along the keys (reserve_attn_part)
    int last_shares = 0;         // pie_decoder_prompt_shares
    int resident_mode = -1;   // -1: budget not fixed yet
    size_t resident_left = 0; // bytes still available for resident copies
};

static_assert(sizeof(RowStat) == sizeof(LogitStat), "one buffer for both");
static int tail_stats_reserve(PrefillScratch *s, size_t entries) {
    if (s->tail_entries >= entries) return PIE_OK;
    if (s->tail_stats) (void)hipFree(s->tail_stats);
    s->tail_stats = nullptr, s->tail_entries = 0;
    PIE_HIP_TRY(hipMalloc((void **)&s->tail_stats, sizeof(LogitStat) * entries));
    s->tail_entries = entries, ++s->alloc_gen;
    return PIE_OK;
}

static void scratch_release(PrefillScratch *s) {  // the chunk buffers; resident weight copies survive a re-size
    void *ptrs[] = {s->wT, s->wM, s->x, s->xn, s->qkv, s->q, s->attn, s->gu, s->act, s->r, s->arrived, s->rope_cs, s->kc, s->vc};
    for (void *p : ptrs)
        if (p) (void)hipFree(p);
    auto keep = std::move(s->resident);
    auto keep_m = std::move(s->resident_w4m);
    LogitStat *keep_ts = s->tail_stats;
    const size_t keep_tr = s->tail_entries;
    const unsigned gen = s->alloc_gen + 1;  // the chunk buffers move: captured launches are stale
    if (s->batch_graph) (void)hipGraphExecDestroy(s->batch_graph);
    const int mode = s->resident_mode;
    const size_t left = s->resident_left;
    void *keep_ws = s->w4l_ws;
    const size_t keep_wsb = s->w4l_ws_bytes;
    float *keep_part = s->attn_part, *keep_acc = s->part_acc, *keep_ml = s->part_ml;
    const size_t keep_parts = s->parts;
    *s = PrefillScratch();
    s->w4l_ws = keep_ws, s->w4l_ws_bytes = keep_wsb, s->attn_part = keep_part, s->part_acc = keep_acc, s->part_ml = keep_ml, s->parts = keep_parts;
    s->resident = std::move(keep), s->resident_w4m = std::move(keep_m), s->resident_mode = mode, s->resident_left = left;
    s->tail_stats = keep_ts, s->tail_entries = keep_tr, s->alloc_gen = gen;
}

void prefill_free(pie_decoder *d) {
    if (!d->prefill) return;
    scratch_release(d->prefill);
    for (auto &kv : d->prefill->resident) (void)hipFree(kv.second);
    for (auto &kv : d->prefill->resident_w4m) (void)hipFree(kv.second.p);
    if (d->prefill->tail_stats) (void)hipFree(d->prefill->tail_stats);
    if (d->prefill->w4l_ws) (void)hipFree(d->prefill->w4l_ws);
    if (d->prefill->attn_part) (void)hipFree(d->prefill->attn_part);
    if (d->prefill->part_acc) (void)hipFree(d->prefill->part_acc);
    if (d->prefill->part_ml) (void)hipFree(d->prefill->part_ml);
    if (d->prefill->batch_graph) (void)hipGraphExecDestroy(d->prefill->batch_graph);
    delete d->prefill;
    d->prefill = nullptr;
}

// The embedding, the final norm and the head are others from here on, perhaps behind the same pointers: the old and the new head's copies and the captured
// step go, the layers' copies stay
void prefill_globals_changed(pie_decoder *d, const void *new_head) {
    PrefillScratch *s = d->prefill;
    if (!s) return;
    ++s->alloc_gen;
    for (const void *head : {(const void *)d->glob.lm_head, new_head}) {
        const int N = d->cfg.vocab, K = d->cfg.hidden;
        if (auto it = s->resident.find(head); it != s->resident.end()) (void)hipFree(it->second), s->resident.erase(it), s->resident_left += w16m_size(N, K);
        if (auto it = s->resident_w4m.find(head); it != s->resident_w4m.end()) (void)hipFree(it->second.p), s->resident_left += it->second.bytes, s->resident_w4m.erase(it);
    }
}

int prefill_min_rows() {  // read per call (not cached): tests and tools switch regimes inside one process
    const int k = pie_knob(PIE_KNOB_PREFILL_MIN);  // prompts shorter than this run as iterated decode steps (MLX's qmv regime)
    const int n = k >= 0 ? k : 6;  // MLX's own qmv limit is 6..32 rows by device and shape; 5 ms batched vs 1.35 ms per iterated row
    return n < 2 ? 2 : n;
}

static int prefill_chunk_rows() {
    const int k = pie_knob(PIE_KNOB_PREFILL_CHUNK);  // measured on the 8B model, 4096-token prompt: 512 -> 119 ms, 1024 -> 83, 2048 -> 67, 4096 -> 65
    const int n = k >= 0 ? k : 4096;
    return n < 16 ? 16 : (n > 8192 ? 8192 : n);
}

// parts: rows whose decode attention is split, times the splits.  Every buffer only grows: prompts have many rows and no such parts, a batch's step few rows and many, and a serving loop
// takes them in turn (sized by the call at hand each took the buffers from the other, all of them anew twice a prompt, and the captured step with them).
static int scratch_reserve(pie_decoder *d, int rows, size_t w_elems, size_t parts) {
    if (!d->prefill) d->prefill = new PrefillScratch();
    PrefillScratch *s = d->prefill;
    const pie_decoder_config &c = d->cfg;
    const size_t QD = (size_t)c.n_heads * c.head_dim, NQKV = QD + 2 * (size_t)c.n_kv_heads * c.head_dim;
    if (rows > s->rows) {
        const size_t we = s->w_elems > w_elems ? s->w_elems : w_elems;
        scratch_release(s);
        const size_t R = (size_t)rows;
#define PF_ALLOC(ptr, bytes) PIE_HIP_TRY(hipMalloc((void **)&(ptr), (bytes)))
        PF_ALLOC(s->x, 2 * R * c.hidden);
        PF_ALLOC(s->xn, 2 * R * c.hidden);
        PF_ALLOC(s->r, 2 * R * c.hidden);
        PF_ALLOC(s->qkv, 2 * R * NQKV);
        PF_ALLOC(s->q, 2 * R * QD);
        PF_ALLOC(s->attn, 2 * R * QD);
        PF_ALLOC(s->gu, 2 * R * 2 * c.inter);
        PF_ALLOC(s->act, 2 * R * c.inter);
        PF_ALLOC(s->arrived, 4 * (R * c.n_kv_heads + 1));
        s->total = s->arrived + R * c.n_kv_heads;
        PIE_HIP_TRY(hipMemset(s->arrived, 0, 4 * (R * c.n_kv_heads + 1)));
        PIE_HIP_TRY(hipStreamSynchronize(nullptr));  // (a pass on a stream that does not wait for the null stream)
        PF_ALLOC(s->rope_cs, 4 * R * c.head_dim);
        PF_ALLOC(s->kc, 2 * R * c.n_kv_heads * c.head_dim);
        PF_ALLOC(s->vc, 2 * R * c.n_kv_heads * c.head_dim);
        PF_ALLOC(s->wT, 2 * we);
        PF_ALLOC(s->wM, 2 * we);
        s->rows = rows, s->w_elems = we;
    }
    if (w_elems > s->w_elems) {
        if (s->wT) (void)hipFree(s->wT);
        if (s->wM) (void)hipFree(s->wM);
        s->wT = nullptr, s->wM = nullptr;
        PF_ALLOC(s->wT, 2 * w_elems);
        PF_ALLOC(s->wM, 2 * w_elems);
        s->w_elems = w_elems, ++s->alloc_gen;
    }
    if (parts > s->parts) {
        if (s->part_acc) (void)hipFree(s->part_acc);
        if (s->part_ml) (void)hipFree(s->part_ml);
        s->part_acc = s->part_ml = nullptr, s->parts = 0, ++s->alloc_gen;
        PF_ALLOC(s->part_acc, 4 * parts * c.n_heads * c.head_dim);
        PF_ALLOC(s->part_ml, 4 * parts * c.n_heads * 2);
        s->parts = parts;
    }
#undef PF_ALLOC
    return PIE_OK;
}

// Room for the sums of prompt attention split along the keys: the most that any split takes (34 MB at 32 / 8 heads of 128), once, with the first prompt's buffers -- no captured launch
// holds it, and a serving loop's longer and longer prefixes must neither allocate nor invalidate the captured batch step.  No room: prompts are not split.
static void reserve_attn_part(pie_decoder *d) {
    const pie_decoder_config &c = d->cfg;
    if (d->prefill->attn_part || 512 / c.n_kv_heads < 2) return;
    if (hipMalloc((void **)&d->prefill->attn_part, prefill_attn_part_bytes(c.n_heads, c.n_kv_heads, c.head_dim)) != hipSuccess) (void)hipGetLastError(), d->prefill->attn_part = nullptr;
}
// How a prompt's attention is launched: split along the keys where that pays (before: keys cached in front of the first row)
static void split_attn(pie_decoder *d, PrefillAttnArgs &a, int before, bool told = true) {  // told: pie_decoder_prompt_shares hears of it
    const int splits = d->prefill->attn_part ? prefill_attn_splits(a.M, before, a.Hq, a.Hkv, d->cfg.head_dim) : 1;
    a.before = before;
    if (told) d->prefill->last_shares = splits;
    if (splits > 1) a.splits = splits, a.part = d->prefill->attn_part;
}

// rows of a pass; few of them (fewer than four workgroups a CU otherwise): a thread's columns in one round
template <class T>
static int rope_append_rows(const pie_decoder *d, const W4lSlabs &sl, int M, int layer, RopeRowsArgs a, hipStream_t st) {
    const pie_decoder_config &c = d->cfg;
    a.qkv = d->prefill->qkv, a.part = sl.part, a.S = sl.S, a.MN = sl.MN, a.n_cols = (c.n_heads + 2 * c.n_kv_heads) * c.head_dim;
    a.layer = layer, a.n_layers = c.n_layers, a.n_heads = c.n_heads, a.n_kv_heads = c.n_kv_heads, a.hd_shift = c.head_dim == 128 ? 7 : 6, a.traditional = c.rope_traditional;
    if (!a.slab) a.n_pages = d->n_pages;
    a.q_out = d->prefill->q, a.rope_cs = d->prefill->rope_cs;
    const bool i8 = a.i8_page_bytes != 0;
    auto k = sl.S > 1 ? i8 ? &k_rope_append_rows<T, true, true> : &k_rope_append_rows<T, true, false> : i8 ? &k_rope_append_rows<T, false, true> : &k_rope_append_rows<T, false, false>;
    hipLaunchKernelGGL(k, dim3(M, M < 1024 ? (a.n_cols + 2047) / 2048 : 1), dim3(256), 0, st, a);
    PIE_LAUNCH_CHECK();
    return PIE_OK;
}

// ---------------------------------------------------------------- the batched forward

// Byte budget for resident T copies of layer matrices, fixed at the first batched prefill: half of the free device memory
// (PIE_KNOB_PREFILL_RESIDENT: 0 disables, <GiB> sets it).  Matrices are admitted in first-use order while the budget lasts
// (8B model: all 15 GB; 70B: ~7/8 of its 140 GB); the rest keep going through the scratch every chunk.
static size_t resident_budget(const pie_decoder *d) {
    PrefillScratch *s = d->prefill;
    if (s->resident_mode < 0) {
        size_t free_b = 0, total_b = 0;
        const int k = pie_knob(PIE_KNOB_PREFILL_RESIDENT);
        if (k >= 0) s->resident_left = (size_t)k << 30;
        else s->resident_left = hipMemGetInfo(&free_b, &total_b) == hipSuccess ? free_b / 2 : 0;
        s->resident_mode = 1;
    }
    return s->resident_left;
}

// Bytes of the 16-bit copies that an int8 model may still make: its prompts beyond 32 rows multiply those, steps and short prompts only prefer the codes' tiles, which take what is left of the budget.
// (First come first served, a model of more copies than budget that stepped first expanded most of its matrices anew in every chunk of its prompts.)
static size_t w16_to_come(const pie_decoder *d) {
    const pie_decoder_config &c = d->cfg;
    const int QD = c.n_heads * c.head_dim, NQKV = QD + 2 * c.n_kv_heads * c.head_dim;
    size_t bytes = 0;
    auto add = [&](const void *packed, int N, int K) {
        if (d->mat_fmt(packed) == PIE_W_INT8_G64 && !d->prefill->resident.count(packed)) bytes += w16m_size(N, K);
    };
    for (const pie_layer_weights &w : d->layers) add(w.wqkv, NQKV, c.hidden), add(w.wo, c.hidden, QD), add(w.wgateup, 2 * c.inter, c.hidden), add(w.wdown, c.hidden, c.inter);
    add(d->glob.lm_head, c.vocab, c.hidden);
    return bytes;
}

// w16_gemm.hpp / w4m_gemm.hip: the 16-bit many-row MFMA GEMM on W16M tiles (weights in MFMA A-fragment order)
int w16m_from_rows_launch(const void *w, int N, int K, void *w16m, hipStream_t st);
int w16m_from_w16s_launch(const void *w16s, int N, int K, void *w16m, hipStream_t st);
size_t w16l_workspace_bytes(int M, int N, int K);
int w16l_gemm_launch(int dtype, const void *w16m, const void *x, int ldx, int M, int N, int K, void *y, void *workspace, hipStream_t st, const void *bias,
                     void *swiglu_act, bool *fused, int ldy);

// The 16-bit operand of a many-row product, as W16M tiles: dense modules straight from their W16S units, int8 / group-32 modules
// dequantised (mx.dequantize's arithmetic: the qmm regime multiplies T copies) into the row-major staging buffer and tiled from there.
template <class T>
static int expand_weights(pie_decoder *d, const void *packed, int N, int K, void *w16m, u16 *staging, hipStream_t st) {
    const int wf = d->mat_fmt(packed);  // per-module quantisation: a checkpoint may mix formats (models/utils.py:99-109)
    if (wf == PIE_W_DENSE) return w16m_from_w16s_launch(packed, N, K, w16m, st);
    if (wf == PIE_W_INT8_G64 || wf == PIE_W_INT8_G32) {
        const size_t w8 = (size_t)N * (K >> 2);
        if (wf == PIE_W_INT8_G32) hipLaunchKernelGGL((k_dequant_w8s<T, true>), dim3((unsigned)((w8 + 255) / 256)), dim3(256), 0, st, (const u32 *)packed, N, K, w4s_slices(K), staging);
        else hipLaunchKernelGGL((k_dequant_w8s<T, false>), dim3((unsigned)((w8 + 255) / 256)), dim3(256), 0, st, (const u32 *)packed, N, K, w4s_slices(K), staging);
        PIE_LAUNCH_CHECK();
        return w16m_from_rows_launch(staging, N, K, w16m, st);
    }
    if (wf == PIE_W_INT2_G64) {
        const size_t w2 = (size_t)N * (K >> 4);
        hipLaunchKernelGGL((k_dequant_w2s<T>), dim3((unsigned)((w2 + 255) / 256)), dim3(256), 0, st, (const u32 *)packed, N, K, w4s_slices(K), staging);
        PIE_LAUNCH_CHECK();
        return w16m_from_rows_launch(staging, N, K, w16m, st);
    }
    if (wf == PIE_W_INT6_G64) {
        const size_t w6 = (size_t)N * (K >> 3);
        hipLaunchKernelGGL((k_dequant_w6s<T>), dim3((unsigned)((w6 + 255) / 256)), dim3(256), 0, st, (const u32 *)packed, N, K, w4s_slices(K), staging);
        PIE_LAUNCH_CHECK();
        return w16m_from_rows_launch(staging, N, K, w16m, st);
    }
    const size_t words = (size_t)N * (K >> 3);
    if (wf == PIE_W_INT4_G32) hipLaunchKernelGGL((k_dequant_w4s<T, true>), dim3((unsigned)((words + 255) / 256)), dim3(256), 0, st, (const u32 *)packed, N, K, w4s_slices(K), staging);
    else hipLaunchKernelGGL((k_dequant_w4s<T, false>), dim3((unsigned)((words + 255) / 256)), dim3(256), 0, st, (const u32 *)packed, N, K, w4s_slices(K), staging);
    PIE_LAUNCH_CHECK();
    return w16m_from_rows_launch(staging, N, K, w16m, st);
}

// y[M, N] = x[M, K] . W^T for one streaming-layout matrix.  keep: a resident copy may be made (layer matrices, the head of batch steps); the
// lm_head of a logits-on-every-position call uses one that is there, and goes through the scratch otherwise.
// w4m_gemm.hip: the few-row int4 GEMM on W4M tiles
int w4m_repack_launch(const void *w4s, int N, int K, void *w4m, hipStream_t st);
struct W4mRope {  // q|k|v epilogue arguments (defined identically in w4m_gemm.hip)
    const float *rope_cs;
    const DecState *state;
    const int *ctx_len;
    const unsigned long long *kv_table;
    u16 *slab;
    const int *block_table;
    int bt_stride, n_pages, layer, n_layers, n_heads, n_kv_heads, HD, traditional;
    u16 *q_out;
    const u16 *bias;
    size_t i8_page_bytes;  // != 0 (with slab): int8 pages with per-head scales (paged_i8.hip)
};
int w4m_gemm_launch(int dtype, const void *w4m, const void *x, int M, int N, int K, void *y, hipStream_t st, int swiglu, const void *bias, const W4mRope *rope);
int w4l_gemm_launch(int dtype, const void *w4m, const void *x, int M, int N, int K, void *y, void *workspace, hipStream_t st, void *swiglu_act, bool *fused,
                    int *slabs);  // many rows (MFMA-bound)
size_t w4l_workspace_bytes(int M, int N, int K);
// 6 .. 256 rows: the weight-streaming form (w4r_gemm.hpp); epi 0 store (+ bias), 1 SwiGLU (+ bias), 2 RoPE + append
bool w4r_serves(int M, int N, int K);
int w4r_splits(int M, int N, int K);
size_t w4r_workspace_bytes(int M, int N, int K);
bool w4m_wide_scales(const void *w4m);
bool w4a_serves(int M, int N, int K, int bits = 4, bool step = false);
int w4a_splits(int M, int N, int K, int bits);
size_t w4a_workspace_bytes(int M, int N, int K, int bits);
size_t w8m_bytes(int N, int K);
int w8m_repack_launch(const void *w8s, int N, int K, void *w8m, hipStream_t st);
int w4a_gemm_launch(int dtype, const void *w4m, const void *x, int M, int N, int K, void *y, void *workspace, hipStream_t st, int epi, const void *bias,
                    const W4mRope *rope, int *slabs, bool *bias_done, int bits);
int w4r_gemm_launch(int dtype, const void *w4m, const void *x, int M, int N, int K, void *y, void *workspace, hipStream_t st, int epi, const void *bias,
                    const W4mRope *rope, int *slabs, bool *bias_done, bool wide_scales);

// int4 checkpoints: prompts beyond small_rows() rows run the hand-written many-row W4 MFMA GEMM on the same W4M tiles -- no 16-bit
// copy of the weights (shapes the tile kernels do not take, N not a multiple of 32, go through the T copy and k_w16l_gemm).
static bool w4l_enabled() { return true; }
// Rows up to which an int4 Linear runs on the W4M kernel instead of the T copy + k_w16l_gemm (PIE_KNOB_SMALL_M: 0 disables, max 32).
static int small_rows() {
    const int k = pie_knob(PIE_KNOB_SMALL_M);
    const int v = k >= 0 ? k : 32;
    return v < 0 ? 0 : (v > 32 ? 32 : v);
}

template <class T>
static int bias_rows(u16 *y, const void *bias, int M, int N, hipStream_t st) {
    const size_t n8 = (size_t)M * N / 8;
    hipLaunchKernelGGL(k_bias_rows<T>, dim3((unsigned)((n8 + 255) / 256)), dim3(256), 0, st, y, (const u16 *)bias, n8, N / 8);
    PIE_LAUNCH_CHECK();
    return PIE_OK;
}

template <class T>
static int linear_rows(pie_decoder *d, const void *packed, int N, int K, const u16 *x, int M, u16 *y, hipStream_t st, bool keep = true,
                       const void *bias = nullptr, bool keep_w4m = false, u16 *act = nullptr, bool *used_act = nullptr, W4mRope *rope = nullptr,
                       W4lSlabs *slabs = nullptr, int pass_rows = 0, bool step = false) {
    // step: M sequences' next rows (w4a_serves).  pass_rows (0: M): rows of the pass that these M belong to: they decide between MLX's regimes, M between the kernels of one
    // slabs: the caller's consumer takes the fp32 slabs of a K-split many-row GEMM (and the bias) instead of y; slabs->S > 1 tells whether it must
    // rope / used_act: for the packed q|k|v matrix the few-row kernel can rotate q / k and append k / v itself
    // act / used_act: for the packed gate|up matrix the few-row kernel can apply the SwiGLU itself and write act [M, N / 2]
    PrefillScratch *s = d->prefill;
    if (used_act) *used_act = false;
    if (slabs) *slabs = W4lSlabs();
    if (pie_knob(PIE_KNOB_W4L_SLABS) == 0) slabs = nullptr;  // always reduce in the GEMM's own launch (the bit-equality test)
    // 8B prompt of 64 / 128 / 256 / 512 / 700 tokens, slabs summed by the consumers vs reduce launches: 3.70 / 4.56 / 6.13 / 9.56 / 14.26 ms
    // vs 3.96 / 4.82 / 6.20 / 9.75 / 14.38.  (With ONE workgroup per row the RoPE consumer could not keep enough slab loads in flight
    // below ~200 rows -- 4.21 ms at 64 tokens -- so few rows get several there, one per 2048 columns (rope_append_rows); the add + RMSNorm
    // consumers, whose reduction is the row's, have one and ask for more slabs at a time.)
    const bool is_int4 = d->mat_fmt(packed) == PIE_W_INT4_G64, qmv = (pass_rows ? pass_rows : M) <= GEMV_ROWS_MAX;
    if ((d->mat_fmt(packed) == PIE_W_INT4_G32 || d->mat_fmt(packed) == PIE_W_INT8_G32 || d->mat_fmt(packed) == PIE_W_INT2_G64 || d->mat_fmt(packed) == PIE_W_INT6_G64) && qmv && K <= 32768 && N % 2 == 0) {  // group-32 / two-bit codes, qmv regime: the streaming GEMV, one pass per row
        GemvArgs a = {};
        a.fmt = d->mat_fmt(packed) == PIE_W_INT2_G64 ? FMT_W2S : d->mat_fmt(packed) == PIE_W_INT6_G64 ? FMT_W6S : d->mat_fmt(packed) == PIE_W_INT8_G32 ? FMT_W8S32 : FMT_W4S32, a.w = (const char *)packed, a.K = K, a.N = N, a.x = x, a.y = y, a.lin_bias = (const u16 *)bias;
        return w4s_gemv_launch(d->cfg.dtype, PRO_NONE, EPI_STORE, a, M, st);
    }
    // resident W4M (W8M) tile copy of an int4 (int8) matrix (0.5625 B, 1.0625 B per weight, built on first use within the residency budget); nullptr: no room
    const bool is_int8 = d->mat_fmt(packed) == PIE_W_INT8_G64;
    const size_t tile_bytes = is_int8 ? w8m_bytes(N, K) : w4m_bytes(N, K);
    bool wide = false;  // of the tiles that w4m_tiles found
    auto w4m_tiles = [&](void **out) -> int {
        *out = nullptr;
        auto it = s->resident_w4m.find(packed);
        if (it != s->resident_w4m.end()) {
            *out = it->second.p, wide = it->second.wide;
            return PIE_OK;
        }
        void *wm = nullptr;
        if (resident_budget(d) >= tile_bytes + (is_int8 ? w16_to_come(d) : 0) && hipMalloc(&wm, tile_bytes) == hipSuccess) {
            const int rc = is_int8 ? w8m_repack_launch(packed, N, K, wm, st) : w4m_repack_launch(packed, N, K, wm, st);
            wide = !is_int8 && w4m_wide_scales(wm);
            s->resident_w4m[packed] = {wm, tile_bytes, wide}, s->resident_left -= tile_bytes, ++s->alloc_gen;
            *out = wm;
            return rc;
        }
        (void)hipGetLastError();
        return PIE_OK;
    };
    auto w4l_reserve = [&](size_t wb) -> int {  // fp32 slabs of a K-split product
        if (wb > s->w4l_ws_bytes) {
            if (s->w4l_ws) (void)hipFree(s->w4l_ws);
            s->w4l_ws = nullptr, s->w4l_ws_bytes = 0;
            PIE_HIP_TRY(hipMalloc(&s->w4l_ws, wb));
            s->w4l_ws_bytes = wb, ++s->alloc_gen;
        }
        return PIE_OK;
    };
    // A product of W4M tiles: affine: k_w4a_gemm, else k_w4r_gemm.  q|k|v, o_proj and down split K over workgroups and hand fp32 slabs to their consumers (RoPE + append, add + RMSNorm); gate|up
    // carries the SwiGLU in its epilogue.
    auto tiles_gemm = [&](void *wm, bool affine) -> int {
        const int bits = is_int8 ? 8 : 4;
        auto go = [&](void *to, void *ws, int epi, const void *b, const W4mRope *r, int *n_slabs, bool *done) {
            return affine ? w4a_gemm_launch(d->cfg.dtype, wm, x, M, N, K, to, ws, st, epi, b, r, n_slabs, done, bits) : w4r_gemm_launch(d->cfg.dtype, wm, x, M, N, K, to, ws, st, epi, b, r, n_slabs, done, wide);
        };
        if (act && used_act) {  // gate|up: SwiGLU (and the Linear's bias) in the epilogue
            *used_act = true;
            return go(act, nullptr, 1, bias, nullptr, nullptr, nullptr);
        }
        // q|k|v wide enough to fill the chip without a K split: RoPE + append in the epilogue.  Not from k_w4a_gemm for a step over T pages: its attention's launch can rotate as
        // well (int8, 24 layers of hidden 1024, 2 / 6 / 32 rows, us a step: 803 / 930 / 1138 rotated here, 755 / 811 / 1050 there; int4, 16 layers
        // of Llama-3-70B, 3 / 8 rows, 2222 / 2316 and 2098 / 2182).
        const bool rotates = rope && used_act && !(affine && rope->slab && !rope->i8_page_bytes);
        if (rotates && (affine ? w4a_splits(M, N, K, bits) : w4r_splits(M, N, K)) == 1) {
            *used_act = true;
            rope->bias = (const u16 *)bias;
            return go(nullptr, nullptr, 2, nullptr, rope, nullptr, nullptr);
        }
        int rc = w4l_reserve(affine ? slabs ? w4a_workspace_bytes(M, N, K, bits) : 0 : w4r_workspace_bytes(M, N, K));
        if (rc) return rc;
        int n_slabs = 0;
        bool bias_done = false;
        rc = go(y, s->w4l_ws, 0, bias, nullptr, slabs ? &n_slabs : nullptr, &bias_done);
        if (!rc && n_slabs > 1) {  // y was NOT written: the consumer sums the slabs, rounds and adds the bias
            slabs->part = (const float *)s->w4l_ws, slabs->S = n_slabs, slabs->MN = (size_t)M * N;
            return PIE_OK;
        }
        if (rc || !bias || bias_done) return rc;
        return bias_rows<T>(y, bias, M, N, st);
    };
    // Three to 16 rows (8 of a prompt and a narrow matrix): the scales on the sums.  One and two go to the GEMV below, as a step's do (batch_fused), also the one that a longer pass leaves to its last layer.
    if (is_int4 && w4a_serves(M, N, K, 4, step) && M > GEMV_FUSED_ROWS) {
        void *wm = nullptr;
        const int rc = w4m_tiles(&wm);
        if (rc) return rc;
        if (wm && !wide) return tiles_gemm(wm, true);
    }
    // Int8 codes, up to 32 rows: the same form (no scale is too large for it: a code has no offset)
    if (is_int8 && (keep || keep_w4m) && w4a_serves(M, N, K, 8)) {
        void *wm = nullptr;
        const int rc = w4m_tiles(&wm);
        if (rc) return rc;
        if (wm) return tiles_gemm(wm, true);
    }
    // Below 6 rows MLX multiplies row by row (qmv: exact fp32 per row, mx.quantized_matmul as reached from nn.QuantizedLinear): the
    // streaming GEMV with the rows' images side by side -- one pass over the weights, each row with the batch-1 arithmetic.  One or two rows of any pass are cheapest there: four
    // layers, 37 rows behind 900, us, the last layer's row in k_w4r_gemm / k_w4a_gemm / here: Llama-3-8B 386 / 386 / 371, Llama-3.2-3B 298 / 304 / 294 (16 rows 262 / 273 / 265: down has nobody to sum
    // its splits, which costs the first a launch of its own and the second the splits).
    const bool last_rows = !qmv && M <= GEMV_FUSED_ROWS && w4r_serves(M, N, K);
    if (is_int4 && (qmv || last_rows) && K % 64 == 0 && N % 2 == 0 && gemv_rows_lds_bytes(K, 1) <= 160u * 1024u) {
        PIE_REQUIRE(!last_rows || pie_aligned(bias, 16), PIE_E_ALIGN, "a prompt's last rows: a Linear's bias needs 16-byte alignment");
        return w4s_gemv_rows_launch(d->cfg.dtype, packed, N, K, x, M, y, (const u16 *)bias, st);
    }
    // Up to 256 rows (a chat turn behind a cached prefix, a prompt chunk, a multi-sequence step): the weight-streaming MFMA GEMM, every CU
    // streaming its slab of W4M tiles once (w4r_gemm.hpp).
    if (is_int4 && w4r_serves(M, N, K)) {
        void *wm = nullptr;
        const int rc = w4m_tiles(&wm);
        if (rc) return rc;
        if (wm) return tiles_gemm(wm, false);
    }
    // Up to 32 rows of a shape k_w4r_gemm does not take (K < 256) -- or all of them with knob PIE_KNOB_W4R = 0, the tests' comparator: round 2's
    // first few-row kernel, one workgroup per 32-column strip
    if ((keep || keep_w4m) && is_int4 && M <= small_rows() && N % 32 == 0 && K % 64 == 0) {
        void *wm = nullptr;
        int rc = w4m_tiles(&wm);
        if (rc) return rc;
        if (wm) {
            if (rope && used_act) {
                *used_act = true;
                rope->bias = (const u16 *)bias;
                return w4m_gemm_launch(d->cfg.dtype, wm, x, M, N, K, nullptr, st, 2, nullptr, rope);
            }
            if (act && used_act) {
                *used_act = true;
                return w4m_gemm_launch(d->cfg.dtype, wm, x, M, N, K, act, st, 1, bias, nullptr);
            }
            rc = w4m_gemm_launch(d->cfg.dtype, wm, x, M, N, K, y, st, 0, nullptr, nullptr);
            if (rc || !bias) return rc;
            return bias_rows<T>(y, bias, M, N, st);
        }
    }
    if (is_int4 && N % 32 == 0 && K % 64 == 0 && w4l_enabled()) {  // beyond 256 rows: the many-row tile kernels
        void *wm = nullptr;
        int rc = w4m_tiles(&wm);
        if (rc) return rc;
        if (wm) {
            if ((rc = w4l_reserve(w4l_workspace_bytes(M, N, K)))) return rc;  // fp32 partial tiles of a K-split shape (medium prompts)
            bool fused = false;  // gate|up without a Linear bias: the SwiGLU rides in the GEMM's epilogue where the shape allows
            int n_slabs = 0;
            rc = w4l_gemm_launch(d->cfg.dtype, wm, x, M, N, K, y, s->w4l_ws, st, (act && used_act && !bias) ? act : nullptr, &fused, slabs ? &n_slabs : nullptr);
            if (fused) *used_act = true;
            if (!rc && n_slabs > 1) {  // y was NOT written: the consumer sums the slabs, rounds and adds the bias
                slabs->part = (const float *)s->w4l_ws, slabs->S = n_slabs, slabs->MN = (size_t)M * N;
                return PIE_OK;
            }
            if (rc || !bias) return rc;
            return bias_rows<T>(y, bias, M, N, st);
        }
    }
    // Everything else -- dense modules, int8 beyond 32 rows, group-32 modules beyond the GEMV's rows -- multiplies a 16-bit copy of the matrix in W16M
    // tiles with the hand-written MFMA GEMM (w16_gemm.hpp); resident copies are built on first use within the budget.
    PIE_REQUIRE(K % 64 == 0, PIE_E_SHAPE, "prefill: a many-row Linear needs in_features % 64 == 0 (pie_set_knob(PIE_KNOB_PREFILL_MIN, 1000000) processes prompts as iterated decode steps)");
    u16 *wM = s->wM;
    bool ready = false;
    auto it = s->resident.find(packed);
    if (it != s->resident.end()) wM = it->second, ready = true;
    else if (keep && resident_budget(d) >= w16m_size(N, K)) {
        const size_t bytes = w16m_size(N, K);
        if (hipMalloc((void **)&wM, bytes) == hipSuccess) s->resident[packed] = wM, s->resident_left -= bytes, ++s->alloc_gen;
        else (void)hipGetLastError(), wM = s->wM, s->resident_left = 0;  // out of memory: scratch from here on
    }
    int rc = PIE_OK;
    if (!ready && (rc = expand_weights<T>(d, packed, N, K, wM, s->wT, st))) return rc;
    // A few sequences' step, a few prompt rows: the streaming form, one launch without slabs or a reduce behind it, up to the rows where k_w16l_gemm's tiles are full enough.  8B layer
    // with 8 rows, k_w16l_gemm (+ reduce) / streaming, us: q|k|v, o_proj and down 58 + 14 / 43, gate|up 55 / 39; with 32 rows 58 + 14 / 57, 55 / 42.
    if (M <= ROWS_W16_MAX) {
        const bool sg = act && used_act;
        if (sg) *used_act = true;
        return rows_w16_launch(d->cfg.dtype, wM, x, M, N, K, sg ? act : y, bias, sg, st);
    }
    if ((rc = w4l_reserve(w16l_workspace_bytes(M, N, K)))) return rc;  // fp32 slabs of a K-split shape (few rows, narrow matrices)
    bool fused = false;  // gate|up: bias and SwiGLU in the GEMM's epilogue where the shape does not split K
    rc = w16l_gemm_launch(d->cfg.dtype, wM, x, 0, M, N, K, y, s->w4l_ws, st, bias, (act && used_act) ? act : nullptr, &fused, 0);
    if (fused) *used_act = true;
    return rc;
}

// x, xn and rope_cs of a pass's M rows.  ctx_len: row m is at position ctx_len[m] - 1 (nullptr: at the decoder's own + m); norm: the first layer's (nullptr: xn is not wanted); total: the
// lengths' sum is, for a step
static int pass_rows(pie_decoder *d, const int32_t *ids, const void *embeds, int M, const int32_t *ctx_len, const void *norm, hipStream_t st, bool total = false) {
    const pie_decoder_config &c = d->cfg;
    PrefillScratch *s = d->prefill;
    const bool dense = !ids || d->mat_fmt(d->glob.embed_codes) == PIE_W_DENSE;
    const int form = dense ? 0 : embed_bits(d), bits = form == PIE_EMBED_W4G32 ? 4 : form == PIE_EMBED_W8G32 ? 8 : form;
    PIE_REQUIRE(c.hidden % (dense ? 8 : 64) == 0, PIE_E_SHAPE, "embedding: hidden must be a multiple of 64 (dense tables: of 8)");
    PIE_REQUIRE(ids ? !dense || pie_aligned(d->glob.embed_codes, 16) : pie_aligned(embeds, 16), PIE_E_ALIGN, "embedding: 16-byte alignment required");
    PIE_REQUIRE(pie_aligned(norm, 16), PIE_E_ALIGN, "pie_rms_norm: 16-byte alignment required");
    PassRowsArgs a = {};
    a.ids = ids, a.embeds = (const u16 *)embeds, a.table = d->glob.embed_codes, a.scales = (const u16 *)d->glob.embed_scales, a.biases = (const u16 *)d->glob.embed_biases;
    a.V = c.vocab, a.H = c.hidden, a.group_shift = form == PIE_EMBED_W4G32 || form == PIE_EMBED_W8G32 ? 5 : 6;
    a.freqs = d->glob.rope_freqs, a.state = d->state, a.ctx_len = ctx_len, a.half = c.head_dim / 2, a.cs = s->rope_cs, a.norm_w = (const u16 *)norm, a.eps = c.rms_eps, a.x = s->x, a.xn = s->xn, a.rows = M, a.total = s->total;
    const dim3 grid(total ? M + 1 : M);
#define PASS_ROWS(T_)                                                                                                  \
    if (bits == 0) hipLaunchKernelGGL((k_pass_rows<T_, 0>), grid, dim3(256), 0, st, a);      \
    else if (bits == 4) hipLaunchKernelGGL((k_pass_rows<T_, 4>), grid, dim3(256), 0, st, a); \
    else hipLaunchKernelGGL((k_pass_rows<T_, 8>), grid, dim3(256), 0, st, a)
    if (c.dtype == PIE_BF16) {
        PASS_ROWS(BF16);
    } else {
        PASS_ROWS(F16);
    }
#undef PASS_ROWS
    PIE_LAUNCH_CHECK();
    return PIE_OK;
}

template <class T>
static int prefill_t(pie_decoder *d, const int32_t *ids, const void *embeds, int L, void *logits_all, int &moved, hipStream_t st) {  // moved: by how much the device's position has
    const pie_decoder_config &c = d->cfg;
    const int H = c.hidden, D = c.head_dim, QD = c.n_heads * D, KVD = c.n_kv_heads * D, NQKV = QD + 2 * KVD, I = c.inter;
    const int chunk = prefill_chunk_rows() < L ? prefill_chunk_rows() : L;
    size_t w_elems = w16m_size(2 * I, H) / 2;  // the 16-bit copies are W16M tiles (rows padded to 32, columns to 64)
    if (w16m_size(NQKV, H) / 2 > w_elems) w_elems = w16m_size(NQKV, H) / 2;
    if (w16m_size(H, I) / 2 > w_elems) w_elems = w16m_size(H, I) / 2;
    if (logits_all && w16m_size(c.vocab, H) / 2 > w_elems) w_elems = w16m_size(c.vocab, H) / 2;
    const bool mfma_attn = pie_knob(PIE_KNOB_PREFILL_ATTN_VALU) != 1;  // 1 forces the row-per-launch-slice VALU kernel (tests compare the two)
    int rc = scratch_reserve(d, chunk, w_elems, mfma_attn ? 0 : (size_t)chunk * d->splits);
    if (rc) return rc;
    PrefillScratch *s = d->prefill;
    if (mfma_attn) reserve_attn_part(d);
    for (int c0 = 0; c0 < L; c0 += chunk) {
        const int M = L - c0 < chunk ? L - c0 : chunk;
        const bool last = c0 + M >= L;
        int R = M;  // rows that go on
        const void *rows = embeds ? (const u16 *)embeds + (size_t)c0 * H : nullptr;  // (models/intern/language.py:155-158: h = inputs_embeds)
        if ((rc = pass_rows(d, embeds ? nullptr : ids + c0, rows, M, nullptr, d->layers[0].attn_norm, st))) return rc;
        for (int li = 0; li < c.n_layers; ++li) {
            const pie_layer_weights &w = d->layers[li];
            // Attention.__call__ (language.py:75-108) on input_layernorm(x): layer 0's is pass_rows', the later ones are fused with the previous block's residual add
            W4mRope re = {s->rope_cs, d->state, nullptr, d->kv_table, nullptr, d->block_table, 0, d->n_pages, li, c.n_layers, c.n_heads, c.n_kv_heads, D,
                          c.rope_traditional, s->q, nullptr, 0};
            bool roped = false;
            W4lSlabs sq, so, sd;  // K-split products handed over as fp32 slabs (q|k|v only without a bias: RoPE takes T(x W^T + b))
            if ((rc = linear_rows<T>(d, w.wqkv, NQKV, H, s->xn, M, s->qkv, st, true, w.bqkv, false, nullptr, &roped, &re, w.bqkv ? nullptr : &sq)))
                return rc;
            if (!roped) {
                RopeRowsArgs ra = {};
                ra.state = d->state, ra.kv_table = d->kv_table, ra.block_table = d->block_table;
                if ((rc = rope_append_rows<T>(d, sq, M, li, ra, st))) return rc;
            }
            // Past the last layer's cache append only the prompt's last row is looked at: of the last chunk that row goes on alone, of an earlier one none (language.py:205-209 multiplies
            // every position by lm_head; logits_all asks for that).  Llama-3-8B widths, four layers, us: int4, 4096 tokens 7082 -> 5631, dense, 509 tokens 1236 -> 1085, int4, 37 tokens behind
            // 900 cached ones 418 -> 401: the last layer then costs its q|k|v and one row's weights.  (Of 32 layers that is a 32nd.)
            if (li + 1 == c.n_layers && !logits_all) {
                if (!last) break;
                hipLaunchKernelGGL(k_add_pos, dim3(1), dim3(1), 0, st, d->state, M - 1);
                PIE_LAUNCH_CHECK();
                moved += M - 1, R = 1;
            }
            u16 *x = s->x + (size_t)(M - R) * H, *q = s->q + (size_t)(M - R) * QD, *attn = s->attn + (size_t)(M - R) * QD;
            if (mfma_attn) {  // causal flash attention on the MFMA units (prefill_attn.hpp)
                PrefillAttnArgs pa = {};
                pa.q = q, pa.kv_table = d->kv_table, pa.layer = li, pa.n_layers = c.n_layers, pa.state = d->state;
                pa.block_table = d->block_table, pa.n_pages = d->n_pages;
                pa.M = R, pa.Hq = c.n_heads, pa.Hkv = c.n_kv_heads, pa.scale = 1.0f / sqrtf((float)D), pa.out = attn;
                split_attn(d, pa, d->pos_hint + c0 + M - R, li == 0);
                if ((rc = prefill_attn_launch_t<T>(pa, D, st))) return rc;
            } else {  // PIE_KNOB_PREFILL_ATTN_VALU = 1: the VALU decode kernel, one query row per blockIdx.z (cross-check for the tests)
                AttnArgs a = {};
                a.q = q, a.kv_table = d->kv_table, a.layer = li, a.n_layers = c.n_layers, a.state = d->state;
                a.block_table = d->block_table, a.n_pages = d->n_pages, a.bt_stride = 0;  // every row reads the one sequence's table
                a.Hq = c.n_heads, a.Hkv = c.n_kv_heads, a.splits = d->splits, a.rows = R, a.scale = 1.0f / sqrtf((float)D);
                a.part_acc = s->part_acc, a.part_ml = s->part_ml, a.out = attn;
                if ((rc = attn_decode_launch(c.dtype, D, a, true, st))) return rc;
            }
            if ((rc = linear_rows<T>(d, w.wo, H, QD, attn, R, s->r, st, true, w.bo, false, nullptr, nullptr, nullptr,
                                     H <= 8192 ? &so : nullptr, M)))
                return rc;
            // h = x + r (language.py:151) + post_attention_layernorm(h) for MLP.__call__ (language.py:126-127)
            if ((rc = add_rms_norm_rows<T>(x, s->r, w.mlp_norm, c.rms_eps, R, H, c.dtype, s->xn, st, so.S > 1 ? w.bo : nullptr, &so)))
                return rc;
            bool fused_act = false;
            if ((rc = linear_rows<T>(d, w.wgateup, 2 * I, H, s->xn, R, s->gu, st, true, w.bgateup, false, s->act, &fused_act, nullptr, nullptr, M))) return rc;
            if (!fused_act) {
                const size_t n_act = (size_t)R * I;
                hipLaunchKernelGGL(k_swiglu_rows<T>, dim3((unsigned)((n_act / 4 + 255) / 256)), dim3(256), 0, st, s->gu, n_act, s->act);
                PIE_LAUNCH_CHECK();
            }
            const bool fused_next = li + 1 < c.n_layers;
            if ((rc = linear_rows<T>(d, w.wdown, H, I, s->act, R, s->r, st, true, w.bdown, false, nullptr, nullptr, nullptr,
                                     fused_next && H <= 8192 ? &sd : nullptr, M)))
                return rc;
            // out = h + r (language.py:153), fused with the next block's input_layernorm when there is one; the prompt's last row goes where the head looks for it
            if (fused_next)
                rc = add_rms_norm_rows<T>(x, s->r, d->layers[li + 1].attn_norm, c.rms_eps, R, H, c.dtype, s->xn, st, sd.S > 1 ? w.bdown : nullptr, &sd);
            else rc = pie_add(x, s->r, (size_t)R * H, c.dtype, logits_all ? x : d->h, st);
            if (rc) return rc;
        }
        if (logits_all) {  // lm_head on every position, like the reference (language.py:205-209)
            if ((rc = pie_rms_norm(s->x, d->glob.final_norm, c.rms_eps, M, H, c.dtype, s->xn, st))) return rc;
            if ((rc = linear_rows<T>(d, d->glob.lm_head, c.vocab, H, s->xn, M, (u16 *)logits_all + (size_t)c0 * c.vocab, st, false))) return rc;
        }
        if (last && logits_all)  // the last position continues through the decode step's lm_head + tail below
            PIE_HIP_TRY(hipMemcpyAsync(d->h, s->x + (size_t)(M - 1) * H, 2 * (size_t)H, hipMemcpyDeviceToDevice, st));
        if (last && !logits_all) break;  // (the position has moved)
        hipLaunchKernelGGL(k_add_pos, dim3(1), dim3(1), 0, st, d->state, last ? M - 1 : M);
        PIE_LAUNCH_CHECK();
        moved += last ? M - 1 : M;
    }
    // logits[:, -1, :] -> logprobs -> greedy token; the tail advances the device-side offset past the last prompt token
    if ((rc = enqueue_kernel(d, PIE_K_LMHEAD, 0, nullptr, d->logits, st))) return rc;
    return enqueue_kernel(d, PIE_K_TAIL, 0, nullptr, d->logits, st);
}

extern "C" int pie_decoder_prompt_shares(const pie_decoder *d) { return d && d->prefill ? d->prefill->last_shares : 0; }

// mx.fast.scaled_dot_product_attention(q, k, v, scale, mask=causal) for L > 1 (models/base.py:37-53,111-113), op level.
extern "C" int pie_sdpa_prefill(const void *q, const void *k, const void *v, int Hq, int Hkv, int L, int offset, int cap, int D, float scale,
                                int dtype, void *out, void *stream) {
    PIE_REQUIRE(q && k && v && out, PIE_E_ARG, "pie_sdpa_prefill: null pointer");
    PIE_REQUIRE(L >= 1 && offset >= 0 && offset + L <= cap, PIE_E_SHAPE, "pie_sdpa_prefill: need offset + L <= cap");
    PIE_REQUIRE(D == 64 || D == 128, PIE_E_SHAPE, "pie_sdpa_prefill: head_dim must be 64 or 128");
    PIE_REQUIRE(Hkv > 0 && Hq % Hkv == 0 && Hq / Hkv <= 8, PIE_E_SHAPE, "pie_sdpa_prefill: n_heads / n_kv_heads must be between 1 and 8");
    PIE_REQUIRE(pie_aligned(q, 16) && pie_aligned(k, 16) && pie_aligned(v, 16) && pie_aligned(out, 8), PIE_E_ALIGN, "pie_sdpa_prefill: misaligned pointer");
    PrefillAttnArgs a = {};
    a.q = (const u16 *)q, a.k = (const u16 *)k, a.v = (const u16 *)v, a.offset = a.before = offset, a.cap = cap;
    a.M = L, a.Hq = Hq, a.Hkv = Hkv, a.scale = scale, a.out = (u16 *)out;
    if (dtype == PIE_BF16) return prefill_attn_launch_t<BF16>(a, D, (hipStream_t)stream);
    if (dtype == PIE_F16) return prefill_attn_launch_t<F16>(a, D, (hipStream_t)stream);
    return pie::fail(PIE_E_ARG, "pie_sdpa_prefill: dtype must be PIE_BF16 or PIE_F16");
}


// attention splits of a batch of B decode rows over block tables of max_blocks pages
static int batch_attn_splits(const pie_decoder *d, int B, int max_blocks, bool step) {  // step: for k_attn_step (T pages)
    const pie_decoder_config &c = d->cfg;
    if (step) {
        // Room for pieces, as many as the kernel may want of a row: how many it cuts depends on the lengths (step_split).  More than rows of like lengths need, for a row that is longer.
        const int n = B * c.n_kv_heads, most = max_blocks < ATTN_MAX_SPLITS ? max_blocks : ATTN_MAX_SPLITS, pieces = 512 / n > 4 ? 512 / n : 4;
        return pieces < most ? pieces : most;
    }
    // attention splits: enough workgroups for two per CU across the batch, never more than pages per sequence
    int splits = ((d->kv_i8 ? 1024 : 512) + B * c.n_kv_heads - 1) / (B * c.n_kv_heads);  // (the int8-page kernel runs 4-wave workgroups: twice as many)
    splits = splits > ATTN_MAX_SPLITS ? ATTN_MAX_SPLITS : (splits > max_blocks ? max_blocks : splits);
    splits = splits < 1 ? 1 : splits;
    // short sequences (tables of at most 8 pages) in a batch of 64+ (sequence, kv-head) workgroups: one split, and no combine launch
    // (threshold 128 -> 64, i.e. from 8 sequences of the 8B model: 8 / 12 sequences 2.46 / 2.57 -> 2.40 / 2.46 ms at ~170 positions,
    // 2.59 / 2.78 -> 2.57 / 2.61 at ~420; at 48 the 6-sequence step lost 1 % at ~420 positions)
    if (max_blocks <= 8 && B * c.n_kv_heads >= (d->kv_i8 ? 512 : 64)) splits = 1;  // (the int8-page kernel's workgroups are half as wide)
    // a handful of short sequences: one split as well -- the split kernel + its combine launch cost 10.6 us per layer against 5.5 for the
    // batch-1 step's attention, and a few hundred positions are a handful of row blocks per wave
    if (B <= GEMV_ROWS_MAX && max_blocks <= 4 && !d->kv_i8) splits = 1;
    return splits;
}

// Whether every matrix of an int4 step has its W4M tiles, or room for them, and k_w4a_gemm takes it.
static bool step_tiles(const pie_decoder *d, int B) {
    const pie_decoder_config &c = d->cfg;
    const int QD = c.n_heads * c.head_dim, NQKV = QD + 2 * c.n_kv_heads * c.head_dim;
    size_t more = 0;
    auto has = [&](const void *packed, int N, int K) {
        if (!w4a_serves(B, N, K, 4, true)) return false;
        const auto it = d->prefill->resident_w4m.find(packed);
        if (it != d->prefill->resident_w4m.end()) return !it->second.wide;
        more += w4m_bytes(N, K);
        return true;
    };
    for (const pie_layer_weights &w : d->layers)
        if (!has(w.wqkv, NQKV, c.hidden) || !has(w.wo, c.hidden, QD) || !has(w.wgateup, 2 * c.inter, c.hidden) || !has(w.wdown, c.hidden, c.inter)) return false;
    return has(d->glob.lm_head, c.vocab, c.hidden) && more <= resident_budget(d);
}

// Up to 2 sequences on an int4 checkpoint (5 without W4M tiles): the batch-1 launch sequence, once, with every GEMV multiplying all rows per weight
// unit (k_w4s_gemv_rows: RMSNorm prologues; RoPE + page append, residual, SwiGLU and logits epilogues, per row) -- 6 launches per
// layer instead of 7, each row in MLX's row-by-row fp32 regime.  Biases, int8 pages and hidden sizes beyond 8192 take the
// general path, and from 3 rows on every step whose matrices k_w4a_gemm takes: the GEMV's work grows with its rows (Llama-3-8B, four layers, 16 steps at 200 positions, 2 / 3 / 4 / 5 rows
// 3812 / 4515 / 5283 / 6332 us; the general path, 2 / 3 / 4 / 5 / 6 / 8 rows 3617 / 3672 / 3715 / 3770 / 3785 / 3897; Llama-3.2-3B, 2 rows 3172, general 2926.  Two rows, too, would gain by the general path since its
// products are 16 x 16; the line was drawn before).
static bool batch_fused(const pie_decoder *d, int B) {
    if (B > GEMV_ROWS_MAX || !d->uniform_int4() || d->kv_i8 || d->cfg.hidden > 8192 || w4s_gemv_waves(d->cfg.vocab, d->cfg.hidden) > TAIL_MAX_STATS) return false;
    for (const pie_layer_weights &w : d->layers)
        if (w.bqkv || w.bo || w.bgateup || w.bdown) return false;
    return B <= GEMV_FUSED_ROWS || !step_tiles(d, B);
}
// fused: the form of the layers that follow, replayed ones too (step_batch keeps it with the graph): with norm and lengths' sum they take another pass's rows
static int batch_rows(pie_decoder *d, const int32_t *tokens, const int32_t *ctx_len, int B, bool fused, hipStream_t st) {
    return pass_rows(d, tokens, nullptr, B, ctx_len, fused ? nullptr : d->layers[0].attn_norm, st, !fused);
}

// ---------------------------------------------------------------- one decode step for B sequences (continuous batching)
// The weights stream once for all B rows (few-row int4 GEMM for B <= 32, the T copy + k_w16l_gemm beyond); each row is its own
// sequence: RoPE at its own position, K/V appended to its own page, attention over its own block table (k_attn_step,
// one sequence per blockIdx.z), lm_head + tail on every row.  What the reference's Scheduler / BatchDetails / PagedAttention
// skeleton (src/pie_core/include/engine/batch_details.hpp:10-88, scheduler.hpp) describes for decode-state sequences.
template <class T>
static int decode_batch_t(pie_decoder *d, const int32_t *tokens, const int32_t *ctx_len, const void *const *slabs, int n_pages,
                          const int32_t *block_tables, int max_blocks, int B, u16 *logits, float *logprobs, int32_t *next_tokens, int32_t *lens, bool fused_rows, hipStream_t st) {
    const pie_decoder_config &c = d->cfg;
    const int H = c.hidden, D = c.head_dim, QD = c.n_heads * D, KVD = c.n_kv_heads * D, NQKV = QD + 2 * KVD, I = c.inter;
    size_t w_elems = w16m_size(2 * I, H) / 2;  // the 16-bit copies are W16M tiles (rows padded to 32, columns to 64)
    if (w16m_size(NQKV, H) / 2 > w_elems) w_elems = w16m_size(NQKV, H) / 2;
    if (w16m_size(H, I) / 2 > w_elems) w_elems = w16m_size(H, I) / 2;
    if (w16m_size(c.vocab, H) / 2 > w_elems) w_elems = w16m_size(c.vocab, H) / 2;
    // (the layers' products say whether they rotated and appended themselves, and with it which kernel attends)
    const int splits = batch_attn_splits(d, B, max_blocks, false), step_splits = fused_rows ? splits : batch_attn_splits(d, B, max_blocks, true);
    int rc = scratch_reserve(d, B, w_elems, (size_t)B * (step_splits > splits ? step_splits : splits));
    if (rc) return rc;
    PrefillScratch *s = d->prefill;
    if (tokens && (rc = batch_rows(d, tokens, ctx_len, B, fused_rows, st))) return rc;  // (nullptr: they are there already)
    const int lm_waves = w4s_gemv_waves(c.vocab, H);
    const bool tiles = !fused_rows && logits_in_tiles(B, c.vocab);
    if ((fused_rows || tiles) && (rc = tail_stats_reserve(s, (size_t)(tiles ? LOGITS_TILES : lm_waves) * (size_t)B))) return rc;
    if (fused_rows) {
        for (int li = 0; li < c.n_layers; ++li) {
            const pie_layer_weights &w = d->layers[li];
            GemvRowsArgs g = {};
            g.w = (const char *)w.wqkv, g.K = H, g.N = NQKV, g.M = B, g.x = s->x, g.norm_w = (const u16 *)w.attn_norm, g.eps = c.rms_eps;
            g.rope_cs = s->rope_cs, g.ctx_len = ctx_len, g.block_table = block_tables, g.slab = (u16 *)slabs[li], g.q_out = s->q;
            g.bt_stride = max_blocks, g.n_pages = n_pages, g.n_heads = c.n_heads, g.n_kv_heads = c.n_kv_heads, g.head_dim = D, g.rope_traditional = c.rope_traditional;
            if ((rc = w4s_gemv_rows_fused_launch(c.dtype, PRO_RMSNORM, EPI_ROPE_KV, g, st))) return rc;
            AttnArgs a = {};
            a.q = s->q, a.slab = (const u16 *)slabs[li], a.block_table = block_tables, a.ctx_len = ctx_len, a.bt_stride = max_blocks, a.n_pages = n_pages;
            a.rows = B, a.Hq = c.n_heads, a.Hkv = c.n_kv_heads, a.splits = splits, a.scale = 1.0f / sqrtf((float)D);
            a.nt_kv = (size_t)B * max_blocks * 64 >= 2048;
            a.part_acc = s->part_acc, a.part_ml = s->part_ml, a.out = s->attn;
            if ((rc = attn_decode_launch(c.dtype, D, a, true, st))) return rc;
            g = GemvRowsArgs();
            g.w = (const char *)w.wo, g.K = QD, g.N = H, g.M = B, g.x = s->attn, g.resid = s->x;
            if ((rc = w4s_gemv_rows_fused_launch(c.dtype, PRO_NONE, EPI_RESIDUAL, g, st))) return rc;
            g = GemvRowsArgs();
            g.w = (const char *)w.wgateup, g.K = H, g.N = 2 * I, g.M = B, g.x = s->x, g.norm_w = (const u16 *)w.mlp_norm, g.eps = c.rms_eps, g.y = s->act;
            if ((rc = w4s_gemv_rows_fused_launch(c.dtype, PRO_RMSNORM, EPI_SWIGLU, g, st))) return rc;
            g = GemvRowsArgs();
            g.w = (const char *)w.wdown, g.K = I, g.N = H, g.M = B, g.x = s->act, g.resid = s->x;
            if ((rc = w4s_gemv_rows_fused_launch(c.dtype, PRO_NONE, EPI_RESIDUAL, g, st))) return rc;
        }
        GemvRowsArgs g = {};
        g.w = (const char *)d->glob.lm_head, g.K = H, g.N = c.vocab, g.M = B, g.x = s->x, g.norm_w = (const u16 *)d->glob.final_norm, g.eps = c.rms_eps;
        g.y = logits, g.stats = s->tail_stats;
        if ((rc = w4s_gemv_rows_fused_launch(c.dtype, PRO_RMSNORM, EPI_LOGITS, g, st))) return rc;
        const dim3 fg(TAIL_FINISH_BLOCKS, B);
        if (c.dtype == PIE_BF16)
            hipLaunchKernelGGL(k_logits_finish<BF16>, fg, dim3(256), 0, st, logits, c.vocab, s->tail_stats, lm_waves, logprobs, next_tokens, (DecState *)nullptr, (int *)nullptr, 0, (const unsigned *)nullptr, lens);
        else
            hipLaunchKernelGGL(k_logits_finish<F16>, fg, dim3(256), 0, st, logits, c.vocab, s->tail_stats, lm_waves, logprobs, next_tokens, (DecState *)nullptr, (int *)nullptr, 0, (const unsigned *)nullptr, lens);
        PIE_LAUNCH_CHECK();
        return PIE_OK;
    }
    for (int li = 0; li < c.n_layers; ++li) {
        const pie_layer_weights &w = d->layers[li];
        const size_t i8pb = d->kv_i8 ? pie_page_i8_bytes(c.n_kv_heads, D) : 0;  // int8 pages: the append (epilogue or row kernel) quantises
        W4mRope re = {s->rope_cs, nullptr, ctx_len, nullptr, (u16 *)slabs[li], block_tables, max_blocks, n_pages, li, c.n_layers, c.n_heads, c.n_kv_heads,
                      D, c.rope_traditional, s->q, nullptr, i8pb};
        bool roped = false;
        W4lSlabs sq;  // q|k|v as the fp32 slabs of a K-split product (no Linear bias: RoPE takes T(x W^T + b))
        if ((rc = linear_rows<T>(d, w.wqkv, NQKV, H, s->xn, B, s->qkv, st, true, w.bqkv, false, nullptr, &roped, &re, w.bqkv ? nullptr : &sq, 0, true)))
            return rc;
        const bool rope_in_attn = !roped && !d->kv_i8;  // T pages: inside the attention launch (k_attn_step)
        if (!roped && d->kv_i8) {
            RopeRowsArgs ra = {};
            ra.ctx_len = ctx_len, ra.slab = (u16 *)slabs[li], ra.block_table = block_tables, ra.bt_stride = max_blocks, ra.n_pages = n_pages, ra.i8_page_bytes = i8pb;
            if ((rc = rope_append_rows<T>(d, sq, B, li, ra, st))) return rc;
        }
        AttnRopeArgs a = {};
        a.q = s->q, a.slab = (const u16 *)slabs[li], a.block_table = block_tables, a.ctx_len = ctx_len, a.bt_stride = max_blocks, a.n_pages = n_pages;
        a.rows = B, a.Hq = c.n_heads, a.Hkv = c.n_kv_heads, a.splits = rope_in_attn ? step_splits : splits, a.scale = 1.0f / sqrtf((float)D);
        a.nt_kv = (size_t)B * max_blocks * 64 >= 2048;
        a.part_acc = s->part_acc, a.part_ml = s->part_ml, a.out = s->attn;
        a.qkv = s->qkv, a.part = sq.part, a.S = sq.S, a.MN = sq.MN, a.n_cols = NQKV, a.rope_cs = s->rope_cs, a.traditional = c.rope_traditional, a.pages = (u16 *)slabs[li], a.arrived = s->arrived, a.total = s->total;
        rc = d->kv_i8 ? paged_attn_i8_launch(c.dtype, D, a, st) : rope_in_attn ? attn_rope_decode_launch(c.dtype, D, a, st) : attn_decode_launch(c.dtype, D, a, true, st);
        if (rc) return rc;
        W4lSlabs so, sd;  // o_proj / down handed over as K-split fp32 slabs where the shape qualifies
        if ((rc = linear_rows<T>(d, w.wo, H, QD, s->attn, B, s->r, st, true, w.bo, false, nullptr, nullptr, nullptr,
                                 H <= 8192 ? &so : nullptr, 0, true)))
            return rc;
        if ((rc = add_rms_norm_rows<T>(s->x, s->r, w.mlp_norm, c.rms_eps, B, H, c.dtype, s->xn, st, so.S > 1 ? w.bo : nullptr, &so)))
            return rc;
        bool fused_act = false;
        if ((rc = linear_rows<T>(d, w.wgateup, 2 * I, H, s->xn, B, s->gu, st, true, w.bgateup, false, s->act, &fused_act, nullptr, nullptr, 0, true))) return rc;
        if (!fused_act) {
            const size_t n_act = (size_t)B * I;
            hipLaunchKernelGGL(k_swiglu_rows<T>, dim3((unsigned)((n_act / 4 + 255) / 256)), dim3(256), 0, st, s->gu, n_act, s->act);
            PIE_LAUNCH_CHECK();
        }
        if ((rc = linear_rows<T>(d, w.wdown, H, I, s->act, B, s->r, st, true, w.bdown, false, nullptr, nullptr, nullptr,
                                 H <= 8192 ? &sd : nullptr, 0, true)))
            return rc;
        const void *next_norm = li + 1 < c.n_layers ? d->layers[li + 1].attn_norm : d->glob.final_norm;  // final norm: language.py:187
        if ((rc = add_rms_norm_rows<T>(s->x, s->r, next_norm, c.rms_eps, B, H, c.dtype, s->xn, st, sd.S > 1 ? w.bdown : nullptr, &sd)))
            return rc;
    }
    // the head's 16-bit tiles stay, like the layers' (int4: its W4M tiles do): laid out anew for every step they cost more than the product (268 MB: 115 us beside 42)
    const bool keep_head = d->mat_fmt(d->glob.lm_head) != PIE_W_INT4_G64;
    if ((rc = linear_rows<T>(d, d->glob.lm_head, c.vocab, H, s->xn, B, logits, st, keep_head, nullptr, true, nullptr, nullptr, nullptr, nullptr, 0, true))) return rc;
    return logits_tail_rows_launch(c.dtype, logits, c.vocab, B, tiles ? (RowStat *)s->tail_stats : nullptr, logprobs, next_tokens, st, lens);
}


// ---------------------------------------------------------------- several fresh prompts in one pass
__global__ void k_gather_rows(const uint4 *x, int H8, uint4 *y, const uint4 *a, int A8, uint4 *b, const int *rows) {  // y[s] = x[rows[s]], b[s] = a[rows[s]]; H8, A8: 16-byte pieces per row
    const size_t row = rows[blockIdx.x], at = blockIdx.x;
    for (int i = threadIdx.x; i < H8 + A8; i += blockDim.x)
        if (i < H8) y[at * H8 + i] = x[row * H8 + i];
        else b[at * A8 + i - H8] = a[row * A8 + i - H8];
}

// The rows of S prompts concatenated ([N] ids): one pass of GEMMs over all N rows, RoPE at each row's own position, K / V into
// each prompt's own pages AND a contiguous copy the attention of this pass reads (causal inside each prompt = the segment
// kernel with seg_hi[r] = r + 1), lm_head + tail on every prompt's last row.  Fresh prompts only (nothing cached before them).
// n_decode > 0 (a mixed batch, batch_details.hpp:10-88's prefill- and decode-state sequences in one BatchDetails): rows
// [0, n_decode) are decode-state sequences -- row r is sequence r (row_seq[r] == r, block-table row r) at position
// row_ctx[r] - 1 with a trivial segment [r, r + 1) -- whose attention then runs over their pages (the multi-sequence step's
// paged kernel) and replaces the segment kernel's rows; the prompt rows follow.  One pass over the weights for both kinds.
template <class T>
static int prefill_varlen_t(pie_decoder *d, const int32_t *ids, const int32_t *row_ctx, const int32_t *row_seq, const int32_t *seg_lo,
                            const int32_t *seg_hi, const int32_t *last_rows, int N, int S, int n_decode, const void *const *slabs, int n_pages,
                            const int32_t *block_tables, int max_blocks, u16 *logits, float *logprobs, int32_t *next_tokens, hipStream_t st,
                            int n_chunks = 0, const int32_t *chunks = nullptr) {
    const pie_decoder_config &c = d->cfg;
    const int H = c.hidden, D = c.head_dim, QD = c.n_heads * D, KVD = c.n_kv_heads * D, NQKV = QD + 2 * KVD, I = c.inter;
    size_t w_elems = w16m_size(2 * I, H) / 2;  // the 16-bit copies are W16M tiles (rows padded to 32, columns to 64)
    if (w16m_size(NQKV, H) / 2 > w_elems) w_elems = w16m_size(NQKV, H) / 2;
    if (w16m_size(H, I) / 2 > w_elems) w_elems = w16m_size(H, I) / 2;
    if (w16m_size(c.vocab, H) / 2 > w_elems) w_elems = w16m_size(c.vocab, H) / 2;
    const int dsplits = n_decode > 0 ? batch_attn_splits(d, n_decode, max_blocks, false) : 1;
    int rc = scratch_reserve(d, N > S ? N : S, w_elems, (size_t)n_decode * dsplits);
    if (rc) return rc;
    PrefillScratch *s = d->prefill;
    const bool tiles = logits_in_tiles(S, c.vocab);
    if (tiles && (rc = tail_stats_reserve(s, (size_t)LOGITS_TILES * S))) return rc;
    if (n_chunks > 0) reserve_attn_part(d);
    if ((rc = pass_rows(d, ids, nullptr, N, row_ctx, d->layers[0].attn_norm, st))) return rc;
    for (int li = 0; li < c.n_layers; ++li) {
        const pie_layer_weights &w = d->layers[li];
        W4lSlabs sq;  // q|k|v as the fp32 slabs of a K-split product (no Linear bias: RoPE takes T(x W^T + b))
        if ((rc = linear_rows<T>(d, w.wqkv, NQKV, H, s->xn, N, s->qkv, st, true, w.bqkv, false, nullptr, nullptr, nullptr, w.bqkv ? nullptr : &sq)))
            return rc;
        RopeRowsArgs ra = {};
        ra.ctx_len = row_ctx, ra.slab = (u16 *)slabs[li], ra.block_table = block_tables, ra.bt_stride = max_blocks, ra.n_pages = n_pages, ra.row_seq = row_seq, ra.kc = s->kc, ra.vc = s->vc;
        ra.i8_page_bytes = d->kv_i8 ? pie_page_i8_bytes(c.n_kv_heads, D) : (size_t)0;  // int8 pages: quantised on the way in; this pass's own attention reads the T copies
        if ((rc = rope_append_rows<T>(d, sq, N, li, ra, st))) return rc;
        PrefillAttnArgs pa = {};
        pa.q = s->q, pa.k = s->kc, pa.v = s->vc, pa.offset = 0, pa.cap = N, pa.seg_lo = seg_lo, pa.seg_hi = seg_hi;
        pa.M = N, pa.Hq = c.n_heads, pa.Hkv = c.n_kv_heads, pa.scale = 1.0f / sqrtf((float)D), pa.out = s->attn;
        if ((rc = segment_attn_gqa_launch_t<T>(pa, D, st))) return rc;
        if (n_decode > 0) {  // the decode-state rows attend to their pages (which hold the row just appended)
            AttnArgs a = {};
            a.q = s->q, a.slab = (const u16 *)slabs[li], a.block_table = block_tables, a.ctx_len = row_ctx, a.bt_stride = max_blocks, a.n_pages = n_pages;
            a.rows = n_decode, a.Hq = c.n_heads, a.Hkv = c.n_kv_heads, a.splits = dsplits, a.scale = pa.scale;
            a.nt_kv = (size_t)n_decode * max_blocks * 64 >= 2048;
            a.part_acc = s->part_acc, a.part_ml = s->part_ml, a.out = s->attn;
            if ((rc = d->kv_i8 ? paged_attn_i8_launch(c.dtype, D, a, st) : attn_decode_launch(c.dtype, D, a, true, st))) return rc;
        }
        for (int ci = 0; ci < n_chunks; ++ci) {  // prompts continuing a cached prefix: causal attention over their pages from the cached length
            const int32_t *ch = chunks + 4 * ci;
            PrefillAttnArgs ca = {};
            ca.q = s->q + (size_t)ch[0] * QD, ca.out = s->attn + (size_t)ch[0] * QD;
            ca.k = (const u16 *)slabs[li], ca.v = (const u16 *)slabs[li] + (size_t)c.n_kv_heads * PIE_PAGE_TOKENS * D;
            ca.offset = ch[2], ca.cap = PIE_PAGE_TOKENS, ca.block_table = block_tables + (size_t)ch[3] * max_blocks, ca.n_pages = n_pages;
            ca.M = ch[1], ca.Hq = c.n_heads, ca.Hkv = c.n_kv_heads, ca.scale = pa.scale;
            split_attn(d, ca, ch[2]);
            if ((rc = prefill_attn_launch_t<T>(ca, D, st))) return rc;
        }
        u16 *x = s->x, *attn = s->attn, *xn = s->xn;
        int R = N;  // rows that go on: past the last layer's cache append, those the head looks at
        if (li + 1 == c.n_layers) {
            R = S, x = s->xn, attn = s->q, xn = s->x;  // (the normalised rows and the queries are used up)
            hipLaunchKernelGGL(k_gather_rows, dim3(S), dim3(256), 0, st, (const uint4 *)s->x, H / 8, (uint4 *)x, (const uint4 *)s->attn, QD / 8, (uint4 *)attn, last_rows);
            PIE_LAUNCH_CHECK();
        }
        W4lSlabs so, sd;  // K-split products handed to their consumers as fp32 slabs (as in the single-prompt path)
        if ((rc = linear_rows<T>(d, w.wo, H, QD, attn, R, s->r, st, true, w.bo, false, nullptr, nullptr, nullptr,
                                 H <= 8192 ? &so : nullptr, N)))
            return rc;
        if ((rc = add_rms_norm_rows<T>(x, s->r, w.mlp_norm, c.rms_eps, R, H, c.dtype, xn, st, so.S > 1 ? w.bo : nullptr, &so)))
            return rc;
        bool fused_act = false;
        if ((rc = linear_rows<T>(d, w.wgateup, 2 * I, H, xn, R, s->gu, st, true, w.bgateup, false, s->act, &fused_act, nullptr, nullptr, N))) return rc;
        if (!fused_act) {
            const size_t n_act = (size_t)R * I;
            hipLaunchKernelGGL(k_swiglu_rows<T>, dim3((unsigned)((n_act / 4 + 255) / 256)), dim3(256), 0, st, s->gu, n_act, s->act);
            PIE_LAUNCH_CHECK();
        }
        if ((rc = linear_rows<T>(d, w.wdown, H, I, s->act, R, s->r, st, true, w.bdown, false, nullptr, nullptr, nullptr,
                                 H <= 8192 ? &sd : nullptr, N)))
            return rc;
        const void *next_norm = li + 1 < c.n_layers ? d->layers[li + 1].attn_norm : d->glob.final_norm;
        if ((rc = add_rms_norm_rows<T>(x, s->r, next_norm, c.rms_eps, R, H, c.dtype, xn, st, sd.S > 1 ? w.bdown : nullptr, &sd)))
            return rc;
    }
    // the normalised last row of every prompt -> lm_head -> tail
    const bool keep_head = d->mat_fmt(d->glob.lm_head) != PIE_W_INT4_G64;  // (as in a step)
    if ((rc = linear_rows<T>(d, d->glob.lm_head, c.vocab, H, s->x, S, logits, st, keep_head, nullptr, true))) return rc;
    return logits_tail_rows_launch(c.dtype, logits, c.vocab, S, tiles ? (RowStat *)s->tail_stats : nullptr, logprobs, next_tokens, st);
}

static size_t active_page_bytes(const pie_decoder *d);
static int varlen_batch(pie_decoder *d, const int32_t *ids, const int32_t *row_context_lens, const int32_t *row_seq, const int32_t *seg_lo,
                        const int32_t *seg_hi, const int32_t *last_rows, int N, int S, int n_decode, const void *const *slabs, size_t n_pages, size_t slab_bytes,
                        const int32_t *block_tables, int max_blocks, void *logits, float *logprobs, int32_t *next_tokens, void *stream, int n_chunks = 0,
                        const int32_t *chunks = nullptr) {
    PIE_REQUIRE(d && ids && row_context_lens && row_seq && seg_lo && seg_hi && last_rows && slabs && block_tables && logits && logprobs && next_tokens,
                PIE_E_ARG, "pie_decoder_prefill_batch / _step_mixed: null pointer");
    PIE_REQUIRE(n_chunks >= 0 && (n_chunks == 0 || chunks), PIE_E_ARG, "pie_decoder_step_mixed: chunks without their descriptor array");
    PIE_REQUIRE(n_chunks == 0 || !d->kv_i8, PIE_E_STATE, "pie_decoder_step_mixed: a prompt continuing a cached prefix reads T pages (int8 pages: fresh prompts and decode rows only)");
    for (int ci = 0; ci < n_chunks; ++ci) {
        const int32_t *ch = chunks + 4 * ci;
        PIE_REQUIRE(ch[0] >= n_decode && ch[1] >= 1 && ch[0] + ch[1] <= N && ch[2] >= 1 && ch[3] >= 0 && ch[3] < S &&
                        (ch[2] + ch[1] + PIE_PAGE_TOKENS - 1) / PIE_PAGE_TOKENS <= max_blocks,
                    PIE_E_SHAPE, "pie_decoder_step_mixed: a chunk is {first row >= n_decode, rows >= 1, cached positions >= 1, sequence < S} inside the batch and its block table");
    }
    PIE_REQUIRE(d->glob_set, PIE_E_STATE, "pie_decoder_prefill_batch / _step_mixed: set_globals must be called first");
    for (char s : d->layer_set) PIE_REQUIRE(s, PIE_E_STATE, "pie_decoder_prefill_batch / _step_mixed: a layer has no weights (pie_decoder_set_layer)");
    PIE_REQUIRE(S >= 1 && N >= S && N <= 65535 && max_blocks > 0 && n_pages > 0 && n_pages < 0x7FFFFFFFu, PIE_E_SHAPE, "pie_decoder_prefill_batch / _step_mixed: bad batch shape");
    PIE_REQUIRE(slab_bytes >= n_pages * active_page_bytes(d), PIE_E_SHAPE,
                "pie_decoder_prefill_batch / _step_mixed: the slabs are smaller than n_pages pages of the active page format (an int8 pool needs PIE_OPT_KV_I8, a T pool must not have it)");
    PIE_REQUIRE(d->cfg.hidden % 8 == 0 && d->cfg.hidden <= 8192, PIE_E_SHAPE, "pie_decoder_prefill_batch / _step_mixed: hidden must be a multiple of 8, at most 8192");
    const int rep = d->cfg.n_heads / d->cfg.n_kv_heads;
    PIE_REQUIRE(rep >= 1 && rep <= 8, PIE_E_SHAPE, "pie_decoder_prefill_batch / _step_mixed: n_heads / n_kv_heads must be between 1 and 8");
    for (int i = 0; i < d->cfg.n_layers; ++i) PIE_REQUIRE(slabs[i] && pie_aligned(slabs[i], 16), PIE_E_ALIGN, "pie_decoder_prefill_batch / _step_mixed: null or misaligned slab");
    hipStream_t st = (hipStream_t)stream;
    return d->cfg.dtype == PIE_BF16 ? prefill_varlen_t<BF16>(d, ids, row_context_lens, row_seq, seg_lo, seg_hi, last_rows, N, S, n_decode, slabs, (int)n_pages,
                                                             block_tables, max_blocks, (u16 *)logits, logprobs, next_tokens, st, n_chunks, chunks)
                                    : prefill_varlen_t<F16>(d, ids, row_context_lens, row_seq, seg_lo, seg_hi, last_rows, N, S, n_decode, slabs, (int)n_pages,
                                                            block_tables, max_blocks, (u16 *)logits, logprobs, next_tokens, st, n_chunks, chunks);
}

extern "C" int pie_decoder_prefill_batch(pie_decoder *d, const int32_t *ids, const int32_t *row_context_lens, const int32_t *row_seq,
                                         const int32_t *seg_lo, const int32_t *seg_hi, const int32_t *last_rows, int N, int S,
                                         const void *const *slabs, size_t n_pages, size_t slab_bytes, const int32_t *block_tables, int max_blocks, void *logits,
                                         float *logprobs, int32_t *next_tokens, void *stream) {
    return varlen_batch(d, ids, row_context_lens, row_seq, seg_lo, seg_hi, last_rows, N, S, 0, slabs, n_pages, slab_bytes, block_tables,
                        max_blocks, logits, logprobs, next_tokens, stream);
}

extern "C" int pie_decoder_step_mixed(pie_decoder *d, const int32_t *ids, const int32_t *row_context_lens, const int32_t *row_seq,
                                      const int32_t *seg_lo, const int32_t *seg_hi, const int32_t *out_rows, int N, int S, int n_decode,
                                      const void *const *slabs, size_t n_pages, size_t slab_bytes, const int32_t *block_tables, int max_blocks, void *logits,
                                      float *logprobs, int32_t *next_tokens, int n_chunks, const int32_t *chunks_host, void *stream) {
    PIE_REQUIRE(n_decode >= 0 && n_decode <= S, PIE_E_SHAPE, "pie_decoder_step_mixed: n_decode must be between 0 and the number of output rows");
    return varlen_batch(d, ids, row_context_lens, row_seq, seg_lo, seg_hi, out_rows, N, S, n_decode, slabs, n_pages, slab_bytes, block_tables,
                        max_blocks, logits, logprobs, next_tokens, stream, n_chunks, chunks_host);
}

static int decode_batch(pie_decoder *d, const int32_t *tokens, const int32_t *ctx_len, const void *const *slabs, int n_pages, const int32_t *block_tables,
                        int max_blocks, int B, void *logits, float *logprobs, int32_t *next_tokens, int32_t *lens, bool fused, hipStream_t st) {
    return d->cfg.dtype == PIE_BF16
               ? decode_batch_t<BF16>(d, tokens, ctx_len, slabs, n_pages, block_tables, max_blocks, B, (u16 *)logits, logprobs, next_tokens, lens, fused, st)
               : decode_batch_t<F16>(d, tokens, ctx_len, slabs, n_pages, block_tables, max_blocks, B, (u16 *)logits, logprobs, next_tokens, lens, fused, st);
}

// bytes one page of the active format takes in a layer's slab: K block + V block of T rows, or the int8 page with its scales
static size_t active_page_bytes(const pie_decoder *d) {
    const pie_decoder_config &c = d->cfg;
    return d->kv_i8 ? pie_page_i8_bytes(c.n_kv_heads, c.head_dim) : (size_t)2 * PIE_PAGE_TOKENS * c.n_kv_heads * c.head_dim * 2;
}

// lens: context_lens where the step moves them on, else nullptr
static int step_batch(pie_decoder *d, const int32_t *tokens, const int32_t *context_lens, int32_t *lens, const void *const *slabs, size_t n_pages, size_t slab_bytes,
                      const int32_t *block_tables, int max_blocks, int B, void *logits, float *logprobs, int32_t *next_tokens, int flags, void *stream) {
    PIE_REQUIRE(d && tokens && context_lens && slabs && block_tables && logits && logprobs && next_tokens, PIE_E_ARG, "pie_decoder_step_batch: null pointer");
    PIE_REQUIRE(d->glob_set, PIE_E_STATE, "pie_decoder_step_batch: set_globals must be called first");
    PIE_REQUIRE(!d->tp(), PIE_E_STATE, "pie_decoder_step_batch: not available on a tensor-parallel shard");
    for (char s : d->layer_set) PIE_REQUIRE(s, PIE_E_STATE, "pie_decoder_step_batch: a layer has no weights (pie_decoder_set_layer)");
    PIE_REQUIRE(B >= 1 && B <= 4096 && max_blocks > 0 && n_pages > 0 && n_pages < 0x7FFFFFFFu, PIE_E_SHAPE, "pie_decoder_step_batch: bad batch shape");
    PIE_REQUIRE(slab_bytes >= n_pages * active_page_bytes(d), PIE_E_SHAPE,
                "pie_decoder_step_batch: the slabs are smaller than n_pages pages of the active page format (an int8 pool needs PIE_OPT_KV_I8, a T pool must not have it)");
    const int rep = d->cfg.n_heads / d->cfg.n_kv_heads;
    PIE_REQUIRE(rep >= 1 && rep <= 8, PIE_E_SHAPE, "pie_decoder_step_batch: n_heads / n_kv_heads must be between 1 and 8");
    for (int i = 0; i < d->cfg.n_layers; ++i) PIE_REQUIRE(slabs[i] && pie_aligned(slabs[i], 16), PIE_E_ALIGN, "pie_decoder_step_batch: null or misaligned slab");
    hipStream_t st = (hipStream_t)stream;
    if (!d->prefill) d->prefill = new PrefillScratch();
    if (!(flags & PIE_STEP_GRAPH)) return decode_batch(d, tokens, context_lens, slabs, (int)n_pages, block_tables, max_blocks, B, logits, logprobs, next_tokens, lens, batch_fused(d, B), st);
    // Graph replay, behind the launch that reads the tokens: those may be another buffer every time (copied to a fixed place first, and the lengths moved on by a launch of their own,
    // a step of 8 sequences took 2 % more).  The launches bake in the caller's buffers and this library's scratch / resident weight copies, so a graph is
    // captured only for a call that repeats the previous call's buffers after that call allocated nothing, and is dropped when
    // either changes.  (First call with new buffers: eager, it may allocate; second: capture; from the third: replay.)
    std::vector<uintptr_t> key = {(uintptr_t)lens, (uintptr_t)context_lens, (uintptr_t)block_tables, (uintptr_t)logits, (uintptr_t)logprobs,
                                  (uintptr_t)next_tokens, (uintptr_t)n_pages, (uintptr_t)max_blocks, (uintptr_t)B, (uintptr_t)d->kv_i8 /* the page format is baked into the launches too */};
    for (int i = 0; i < d->cfg.n_layers; ++i) key.push_back((uintptr_t)slabs[i]);
    PrefillScratch *s = d->prefill;
    if (s->batch_graph && s->batch_key == key && s->batch_gen == s->alloc_gen) {
        if (const int rc = batch_rows(d, tokens, context_lens, B, s->batch_form, st)) return rc;
        PIE_HIP_TRY(hipGraphLaunch(s->batch_graph, st));
        return PIE_OK;
    }
    const bool fused = batch_fused(d, B);
    if (s->warm_key == key && s->warm_gen == s->alloc_gen) {
        if (s->batch_graph) (void)hipGraphExecDestroy(s->batch_graph), s->batch_graph = nullptr;
        hipGraph_t g = nullptr;
        hipStream_t cs = nullptr;
        PIE_HIP_TRY(hipStreamCreateWithFlags(&cs, hipStreamNonBlocking));
        hipError_t e = hipStreamBeginCapture(cs, hipStreamCaptureModeThreadLocal);
        if (e != hipSuccess) {
            (void)hipStreamDestroy(cs);
            return pie::fail(PIE_E_HIP, std::string("hipStreamBeginCapture: ") + hipGetErrorString(e));
        }
        const unsigned gen = s->alloc_gen;
        const int rc = decode_batch(d, nullptr, context_lens, slabs, (int)n_pages, block_tables, max_blocks, B, logits, logprobs, next_tokens, lens, fused, cs);
        e = hipStreamEndCapture(cs, &g);
        (void)hipStreamDestroy(cs);
        if (rc || e != hipSuccess || d->prefill->alloc_gen != gen) {  // something allocated or failed under capture: run this call eagerly instead
            if (g) (void)hipGraphDestroy(g);
            (void)hipGetLastError();
            d->prefill->warm_key.clear();
            return decode_batch(d, tokens, context_lens, slabs, (int)n_pages, block_tables, max_blocks, B, logits, logprobs, next_tokens, lens, fused, st);
        }
        s = d->prefill;
        e = hipGraphInstantiate(&s->batch_graph, g, nullptr, nullptr, 0);
        (void)hipGraphDestroy(g);
        if (e != hipSuccess) return pie::fail(PIE_E_HIP, std::string("hipGraphInstantiate: ") + hipGetErrorString(e));
        s->batch_key = key, s->batch_gen = s->alloc_gen, s->batch_form = fused;
        if (const int rows = batch_rows(d, tokens, context_lens, B, fused, st)) return rows;
        PIE_HIP_TRY(hipGraphLaunch(s->batch_graph, st));
        return PIE_OK;
    }
    const int rc = decode_batch(d, tokens, context_lens, slabs, (int)n_pages, block_tables, max_blocks, B, logits, logprobs, next_tokens, lens, fused, st);
    d->prefill->warm_key = key, d->prefill->warm_gen = d->prefill->alloc_gen;
    return rc;
}
extern "C" int pie_decoder_step_batch(pie_decoder *d, const int32_t *tokens, const int32_t *context_lens, const void *const *slabs, size_t n_pages, size_t slab_bytes,
                                      const int32_t *block_tables, int max_blocks, int B, void *logits, float *logprobs, int32_t *next_tokens,
                                      int flags, void *stream) {
    return step_batch(d, tokens, context_lens, nullptr, slabs, n_pages, slab_bytes, block_tables, max_blocks, B, logits, logprobs, next_tokens, flags, stream);
}
extern "C" int pie_decoder_step_batch_advance(pie_decoder *d, const int32_t *tokens, int32_t *context_lens, const void *const *slabs, size_t n_pages, size_t slab_bytes,
                                              const int32_t *block_tables, int max_blocks, int B, void *logits, float *logprobs, int32_t *next_tokens,
                                              int flags, void *stream) {
    return step_batch(d, tokens, context_lens, context_lens, slabs, n_pages, slab_bytes, block_tables, max_blocks, B, logits, logprobs, next_tokens, flags, stream);
}

int prefill_batched(pie_decoder *d, const int32_t *ids, const void *embeds, int L, void *logits_all, hipStream_t st) {
    const int rep = d->cfg.n_heads / d->cfg.n_kv_heads;
    PIE_REQUIRE(rep >= 1 && rep <= 8, PIE_E_SHAPE, "prefill: n_heads / n_kv_heads must be between 1 and 8");
    int moved = 0;
    const int rc = d->cfg.dtype == PIE_BF16 ? prefill_t<BF16>(d, ids, embeds, L, logits_all, moved, st) : prefill_t<F16>(d, ids, embeds, L, logits_all, moved, st);
    if (rc == PIE_OK) d->pos_hint += L;
    else if (moved) hipLaunchKernelGGL(k_add_pos, dim3(1), dim3(1), 0, st, d->state, -moved);  // a prompt that fails leaves the sequence where it was
    return rc;
}
