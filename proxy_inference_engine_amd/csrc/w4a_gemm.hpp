// w4a_gemm.hpp -- int4 (int8) g=64 x T GEMM for 3 to 16 (1 to 32) rows with the scales and biases applied to the sums: y = sum over groups of s (q . x) + b sum(x), the weights never rounded to T
// (mx.quantized_matmul's row-by-row arithmetic: models/llama/language.py:83,108,127).  (Included by w4m_gemm.hip.)
//
// k_w4r_gemm turns every weight into T in front of its product, 17 vector instructions per eight of them, and its waves wait for each other at every step for the x that they share.  For a
// few rows that is most of its time: gate|up of Llama-3-8B, 66 MB, 19 us for 8 rows; without its products 14, of which 3 are a launch's.  Here
//   * the codes are operands as they stand -- bf16: under the exponent of 128, one v_and_or for two, f16: less 1024 -- and a group's products are multiplied by its scale and joined by bias
//     times the group's sum of x (another product, by ones) in fp32: 2 fused operations per row (of eight) and 32 columns instead of 68;
//   * a wave's K-phase is its own: it stages the x of its groups itself, by LDS-DMA into a ring of its own, and waits for nothing but its loads;
//   * a workgroup takes `halves` half strips of 16 columns, so that 1792 of them are seven for each CU (896 strips: four for 224 CUs); the lanes of the other half of a strip load nothing.
// us, k_w4r_gemm / this, weights from HBM, 8 rows: gate|up [28672, 4096] 19.0 / 16.4-17.6, down [4096, 14336] 11.9 / 11.4, q|k|v [6144, 4096] 7.3 / 6.8, o [4096, 4096] 5.65 / 5.2, head [32768, 4096]
// 20.5 / 19.1; [16384, 3072] 10.9 / 9.8, [3072, 8192] 7.3 / 6.6, [3072, 3072] 5.3 / 4.6.  16 rows: 18.5 / 16.2-17.6, 11.3 / 11.1, 7.0 / 7.4, 5.65 / 6.0, 21.1 / 18.8; 32 rows: 19.1 / 19.8 and
// worse.  Without the products gate|up takes 15 us (5.4 TB/s and a launch): 2 us are not hidden.
// The ring is less deep than written.  The compiler does not count the DMAs, so in front of a weight's use it lets no more loads be in flight, x among them, than (D - 1) steps have of weights: one strip
// of 8 rows 9 and 8 instead of 12, of 16 rows 9 and 8 instead of 16 (two steps, not four), int8 of 32 rows 11 to 9 instead of 21.  Strict, never too weak; but that deeper rings were slower and that
// int4 of 32 rows is better off elsewhere was measured with it.
// Error (2-norm, before the rounding to T) against 64 bits: 9e-7; of weights rounded to bf16 1.7e-3.
#pragma once

constexpr int W4A_ROWS = 16, W8A_ROWS = 32;
constexpr int W8M_TILE_BYTES = 2176;  // W8M (below)
struct W4aArgs {
    const char *w4m;   // W4M (W8M) tiles of the [N, K] matrix
    const u16 *x;      // [M, K]
    int M, N, K;
    int halves;        // half strips (16 columns) per workgroup
    int groups;        // of K (64 columns) per blockIdx.y
    u16 *y;            // STORE: [M, N]; SWIGLU: the activation [M, N / 2]
    float *part;       // SLAB: [gridDim.y][M][N] un-rounded fp32 sums
    const u16 *bias;   // the Linear's bias (nullable; STORE / SWIGLU; ROPE takes W4mRope::bias)
    int epi;
};

// eight codes of a W4M word as T: q + 128 (bf16: a nibble under 128's exponent; the caller takes the 128 out), q itself (f16)
template <class T>
__device__ __forceinline__ uint4 w4a_codes(u32 w) {
    if constexpr (std::is_same<T, F16>::value) return make_uint4(F16::codes2(w & 0x000F000Fu), F16::codes2((w >> 4) & 0x000F000Fu), F16::codes2((w >> 8) & 0x000F000Fu), F16::codes2((w >> 12) & 0x000F000Fu));
    return make_uint4((w & 0x000F000Fu) | 0x43004300u, ((w >> 4) & 0x000F000Fu) | 0x43004300u, ((w >> 8) & 0x000F000Fu) | 0x43004300u, ((w >> 12) & 0x000F000Fu) | 0x43004300u);
}
template <class T>
constexpr float w4a_offset() { return std::is_same<T, F16>::value ? 0.0f : 128.0f; }

// Int8 codes, W8M tiles: as W4M, 32 rows x 64 columns, two pieces of 1 KiB and the 32 {scale, bias} words: lane l = 32 kh + n holds in piece h the codes of row n of k-steps 2 h and 2 h + 1, two words
// each, in the W8S word format (codes 0, 2, 1, 3).  Up to 255 a code is a bf16 and an f16 as it stands.
// Bound by the stream; before, two and more rows multiplied a 16-bit copy, twice the bytes.  us of 16 steps of four layers at 200 positions, 16-bit copy / this: Llama-3-8B 2 rows 6924 / 5080, 4 7209 / 5288,
// 8 7440 / 5474, 16 8042 / 6015, 32 9319 / 6719; Llama-3.2-3B 4 rows 5357 / 3881, 8 5142 / 4033.  Error of a step against 64 bits 0.0095-0.0100 / 0.0089-0.0095.
template <class T>
__device__ __forceinline__ u32 w8a_pair(u32 a, u32 b) {  // two codes as T, b in the high half
    if constexpr (std::is_same<T, F16>::value) return __builtin_bit_cast(u32, __builtin_amdgcn_cvt_pkrtz((float)a, (float)b));
    return __builtin_amdgcn_perm(__builtin_bit_cast(u32, (float)b), __builtin_bit_cast(u32, (float)a), 0x07060302u);
}
template <class T>
__device__ __forceinline__ uint4 w8a_codes(u32 lo, u32 hi) {
    return make_uint4(w8a_pair<T>(lo & 0xFFu, (lo >> 16) & 0xFFu), w8a_pair<T>((lo >> 8) & 0xFFu, lo >> 24), w8a_pair<T>(hi & 0xFFu, (hi >> 16) & 0xFFu), w8a_pair<T>((hi >> 8) & 0xFFu, hi >> 24));
}

template <class T, int MT, int SPW, int D, int BITS = 4>
__global__ void __launch_bounds__(512) k_w4a_gemm(const W4aArgs a, const W4mRope rp) {
    constexpr int PC = BITS / 4, TILE = BITS == 8 ? W8M_TILE_BYTES : W4M_TILE_BYTES;  // code pieces (16 bytes a lane) of a tile; bytes of one
    constexpr int KW = 8, XJ = MT / 8, WL = (PC + 1) * SPW, CHUNK = MT * 128;  // K-phases = waves; DMA instructions (eight rows of a group each), weight loads per step; bytes of x of a step
    constexpr int RL = MT / 2;                                  // accumulators that hold rows < MT
    constexpr int RSTR = 36, BLK = MT * RSTR * 4;               // reduction: one (phase, strip) block, rows of 32 + 4 floats
    constexpr int RED = KW * SPW * BLK, LDS = KW * D * CHUNK > RED ? KW * D * CHUNK : RED;
    constexpr unsigned NOWHERE = 0x80000000u;
    static_assert((D - 1) * (XJ + WL) <= 63 && LDS <= 160 * 1024, "limits");
    __shared__ __attribute__((aligned(1024))) char smem[LDS];
    const int lane = threadIdx.x & 63, p = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n = lane & 31, kh = lane >> 5;
    const int all_groups = a.K >> 6, n_halves = a.N >> 4;
    const int g_lo = blockIdx.y * a.groups + p, g_hi = min(all_groups, ((int)blockIdx.y + 1) * a.groups);  // this wave's groups: g_lo, g_lo + 8, ..
    const int steps = g_hi > g_lo ? (g_hi - g_lo + KW - 1) / KW : 0;
    const int h0 = blockIdx.x * a.halves, h1 = min(h0 + a.halves, n_halves), strip0 = h0 >> 1;
    const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc(const_cast<char *>(a.w4m), 0, (a.N >> 5) * all_groups * TILE, 0x00020000);
    unsigned code_at[SPW], scale_at[SPW], strip_at[SPW];
#pragma unroll
    for (int s = 0; s < SPW; ++s) {
        const int h = 2 * (strip0 + s) + (n >> 4);
        const bool mine = h >= h0 && h < h1;  // (the strips at both ends may be another workgroup's by half)
        code_at[s] = mine ? 16u * lane : NOWHERE, scale_at[s] = mine ? 1024u * PC + 4u * n : NOWHERE;
        strip_at[s] = (unsigned)((strip0 + s) * all_groups + g_lo) * TILE;
    }
    u32 xoffs[XJ];
#pragma unroll
    for (int j = 0; j < XJ; ++j) {
        const int r = 8 * j + (lane >> 3), rr = r < a.M ? r : a.M - 1;  // rows past the end repeat the last one (never stored)
        xoffs[j] = (u32)(((size_t)rr * a.K + (size_t)(((lane & 7) ^ ((r >> 1) & 7)) * 8)) * 2);
    }
    const unsigned lds0 = (unsigned)(size_t)(__attribute__((address_space(3))) void *)smem + (unsigned)(p * D * CHUNK);
    typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
    uint4 cw[D][SPW][PC];
    u32 sb[D][SPW];
    auto issue = [&](int d, int j) {
        const char *src = reinterpret_cast<const char *>(a.x) + (size_t)(g_lo + (j < steps ? j : steps - 1) * KW) * 128;
#pragma unroll
        for (int i = 0; i < XJ; ++i) {
            unsigned keep;
            asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2\n\ts_mov_b32 m0, %0"
                         : "=&s"(keep)
                         : "v"(xoffs[i]), "s"(src), "s"(lds0 + (unsigned)(d * CHUNK + i * 1024))
                         : "memory");
        }
        const unsigned o = (unsigned)j * (KW * TILE), dead = j < steps ? 0u : NOWHERE;
#pragma unroll
        for (int s = 0; s < SPW; ++s) {
#pragma unroll
            for (int q = 0; q < PC; ++q) {
                const u32x4 c = __builtin_amdgcn_raw_buffer_load_b128(wr, (code_at[s] | dead) + 1024u * q, strip_at[s] + o, 2);
                cw[d][s][q] = make_uint4(c.x, c.y, c.z, c.w);
            }
            sb[d][s] = __builtin_amdgcn_raw_buffer_load_b32(wr, scale_at[s] | dead, strip_at[s] + o, 2);
        }
    };
    if (steps > 0)
#pragma unroll
        for (int d = 0; d < D; ++d) issue(d, d);
    int xoff[4];
    const int xrow = n & (MT - 1);
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) xoff[kk] = p * D * CHUNK + xrow * 128 + (((2 * kk + kh) ^ ((xrow >> 1) & 7)) << 4);
    float acc[SPW][RL];
#pragma unroll
    for (int s = 0; s < SPW; ++s)
#pragma unroll
        for (int i = 0; i < RL; ++i) acc[s][i] = 0.0f;
    const u32 one = std::is_same<T, F16>::value ? 0x3C003C00u : 0x3F803F80u;
    const uint4 ones = make_uint4(one, one, one, one);
    const f32x16_t zero = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
    for (int base = 0; base < steps; base += D) {
#pragma unroll
        for (int d = 0; d < D; ++d) {
            if (base + d < steps) {
                W4R_WAIT_VM((D - 1) * (XJ + WL));
                uint4 xq[4];
#pragma unroll
                for (int kk = 0; kk < 4; ++kk) xq[kk] = *reinterpret_cast<const uint4 *>(smem + d * CHUNK + xoff[kk]);
                f32x16_t xs = zero;
#pragma unroll
                for (int kk = 0; kk < 4; ++kk) xs = MfmaT<T>::run(xq[kk], ones, kk ? xs : zero);
#pragma unroll
                for (int s0 = 0; s0 < SPW; s0 += 2) {
                    f32x16_t dot[2];
#pragma unroll
                    for (int kk = 0; kk < 4; ++kk)
#pragma unroll
                        for (int s = s0; s < s0 + 2 && s < SPW; ++s) {
                            uint4 wf;
                            if constexpr (BITS == 8) {
                                const uint4 &c = cw[d][s][kk >> 1];
                                wf = kk & 1 ? w8a_codes<T>(c.z, c.w) : w8a_codes<T>(c.x, c.y);
                            } else {
                                const uint4 &c = cw[d][s][0];
                                wf = w4a_codes<T>(kk == 0 ? c.x : (kk == 1 ? c.y : (kk == 2 ? c.z : c.w)));
                            }
                            dot[s - s0] = MfmaT<T>::run(xq[kk], wf, kk ? dot[s - s0] : zero);
                        }
#pragma unroll
                    for (int s = s0; s < s0 + 2 && s < SPW; ++s) {
                        const float sc = lo_f32<T>(sb[d][s]), bi = BITS == 8 ? hi_f32<T>(sb[d][s]) : fmaf(-w4a_offset<T>(), sc, hi_f32<T>(sb[d][s]));
#pragma unroll
                        for (int i = 0; i < RL; ++i) acc[s][i] = fmaf(bi, xs[i], fmaf(sc, dot[s - s0][i], acc[s][i]));
                    }
                }
            }
            __builtin_amdgcn_sched_barrier(0);
            issue(d, base + d + D);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    W4R_WAIT_VM(0);  // (the DMAs past the end)
    __syncthreads();
    // accumulator i of lane (n, kh): row (i & 3) + 8 (i >> 2) + 4 kh, column n
#pragma unroll
    for (int s = 0; s < SPW; ++s)
#pragma unroll
        for (int i = 0; i < RL; ++i) *reinterpret_cast<float *>(smem + (p * SPW + s) * BLK + (((i & 3) + 8 * (i >> 2) + 4 * kh) * RSTR + n) * 4) = acc[s][i];
    __syncthreads();
    const int EPI = a.epi;
    for (int o = threadIdx.x; o < MT * SPW * 4; o += 512) {  // a row's eight columns
        const int m = o / (4 * SPW), ts = (o >> 2) % SPW, ec = o & 3, col = 32 * (strip0 + ts) + 8 * ec, h = col >> 4;
        if (m >= a.M || h < h0 || h >= h1) continue;
        float v[8] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int ph = 0; ph < KW; ++ph) {
            const float4 *q = reinterpret_cast<const float4 *>(smem + (ph * SPW + ts) * BLK + (m * RSTR + 8 * ec) * 4);
            const float4 lo = q[0], hi = q[1];
            v[0] += lo.x, v[1] += lo.y, v[2] += lo.z, v[3] += lo.w, v[4] += hi.x, v[5] += hi.y, v[6] += hi.z, v[7] += hi.w;
        }
        if (EPI == W4R_SLAB) {
            float *pr = a.part + ((size_t)blockIdx.y * a.M + m) * a.N + col;
            *reinterpret_cast<float4 *>(pr) = make_float4(v[0], v[1], v[2], v[3]);
            *reinterpret_cast<float4 *>(pr + 4) = make_float4(v[4], v[5], v[6], v[7]);
            continue;
        }
        if (EPI == W4R_ROPE) {
#pragma unroll
            for (int e = 0; e < 8; e += 2) w4m_rope_pair<T>(v[e], v[e + 1], m, col + e, rp);
            continue;
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = round_T<T>(v[e]);  // the Linear's rounding to T
        if (a.bias) {
            const uint4 bb = *reinterpret_cast<const uint4 *>(a.bias + col);
            const u32 bw[4] = {bb.x, bb.y, bb.z, bb.w};
#pragma unroll
            for (int e = 0; e < 4; ++e) v[2 * e] = round_T<T>(v[2 * e] + lo_f32<T>(bw[e])), v[2 * e + 1] = round_T<T>(v[2 * e + 1] + hi_f32<T>(bw[e]));
        }
        if (EPI == W4R_SWIGLU) {  // columns (2 i, 2 i + 1) = (gate_i, up_i): act = T(T(silu(g)) * u)
            u16 r[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float g = v[2 * e], u = v[2 * e + 1];
                r[e] = T::from_f32(round_T<T>(g / (1.0f + expf(-g))) * u);
            }
            *reinterpret_cast<uint2 *>(a.y + (size_t)m * (a.N >> 1) + (col >> 1)) = make_uint2((u32)r[0] | ((u32)r[1] << 16), (u32)r[2] | ((u32)r[3] << 16));
        } else
            *reinterpret_cast<uint4 *>(a.y + (size_t)m * a.N + col) = make_uint4(w4m_pack<T>(v[0], v[1]), w4m_pack<T>(v[2], v[3]), w4m_pack<T>(v[4], v[5]), w4m_pack<T>(v[6], v[7]));
    }
}
