// w4a_gemm.hpp -- int4 (int8) g=64 x T GEMM for 3 to 16 (1 to 32) rows with the scales and biases applied to the sums: y = sum over groups of s (q . x) + b sum(x), the weights never rounded to T
// (mx.quantized_matmul's row-by-row arithmetic: models/llama/language.py:83,108,127).  (Included by w4m_gemm.hip.)
//
// k_w4r_gemm turns every weight into T in front of its product, 17 vector instructions per eight of them, and its waves wait for each other at every step for the x that they share.  For a
// few rows that is most of its time.  Here
//   * the codes are operands as they stand -- bf16: under the exponent of 128, one v_and_or for two, f16: less 1024 -- and a group's products are multiplied by its scale and joined by bias
//     times the group's sum of x (another product, by ones) in fp32;
//   * products are 16 x 16 x 32: sixteen rows and sixteen columns, the even or the odd ones of a strip (a v_permlane16_swap of two words makes two such operands of a tile's).  Up to eight
//     rows, rows 8..15 of a product are the same rows against the odd columns (zeros in the others' place), so that no lane of the sums is idle;
//   * a wave's K-phase is its own: it loads the x of its groups straight into the operand's lanes (a group of eight rows is one load) and waits for nothing but its loads, all of them ordinary
//     ones, so that the compiler's waits are exact; the scales of a step's four strips are one load.
// Bound by the stream, a launch (3 us) and the conversion, of which 1.7 us are not hidden.  us, weights from HBM, k_w4r_gemm / the form before (32 x 32 products, x by LDS-DMA, which the compiler's
// waits do not count: rings shallower than written) / this, 8 rows: gate|up [28672, 4096] 18.0 / 17.0 / 14.0, down [4096, 14336] 11.1 / 10.6 / 8.9, q|k|v [6144, 4096] 7.2 / 6.7 / 6.0, o [4096, 4096]
// 5.6 / 5.3 / 4.6, head [32768, 4096] 18.3 / 17.6 / 14.6; [16384, 3072] 9.8 / 9.9 / 8.0, [3072, 8192] 7.2 / 6.7 / 6.0.  16 rows: 17.9 / 18.4 / 15.1, 11.4 / 11.2 / 9.2, 7.3 / 7.6 / 6.2,
// 5.6 / 6.0 / 4.6, 19.8 / 19.5 / 15.6.  32 rows of int4: 18.5 / 19.8 / 21.4, 11.6 / - / 13.0: k_w4r_gemm's.  Without the conversion gate|up takes 12.8 us, without any arithmetic 11.9 to 12.8.
// Two steps in flight per wave are enough (eight waves of 4.6 KB each): three and four cost 1 and 2 us of gate|up's.  The last round issues no loads (loads past a wave's end return nothing but take their
// slots: q|k|v 6.1 / 6.0, o 4.7 / 4.6, int8 down 12.7 / 12.3); both loops need the ring as whole vectors, see there.
// Error (2-norm, before the rounding to T) against 64 bits: 9e-7; of weights rounded to bf16 1.7e-3.
#pragma once

constexpr int W4A_ROWS = 16, W8A_ROWS = 32;
constexpr int W8M_TILE_BYTES = 2176;  // W8M (below)
struct W4aArgs {
    const char *w4m;   // W4M (W8M) tiles of the [N, K] matrix
    const u16 *x;      // [M, K]
    int M, N, K;
    int strips;        // strips (32 columns) per workgroup
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
// Bound by the stream, half the bytes of a 16-bit copy's.  us, the form with 32 x 32 products / this, 8 rows: gate|up 23.3 / 22.1, down 13.3 / 12.3, q|k|v 8.8 / 7.5, o 6.5 / 5.6, head 24.9 / 24.0; 32 rows: 27.0 / 26.8,
// 17.1 / 16.6, 12.1 / 10.2, 8.8 / 7.0, 28.4 / 28.0.
template <class T>
__device__ __forceinline__ u32 w8a_pair(u32 a, u32 b) {  // two codes as T, b in the high half
    if constexpr (std::is_same<T, F16>::value) return __builtin_bit_cast(u32, __builtin_amdgcn_cvt_pkrtz((float)a, (float)b));
    return __builtin_amdgcn_perm(__builtin_bit_cast(u32, (float)b), __builtin_bit_cast(u32, (float)a), 0x07060302u);
}
template <class T>
__device__ __forceinline__ uint4 w8a_codes(u32 lo, u32 hi) {
    return make_uint4(w8a_pair<T>(lo & 0xFFu, (lo >> 16) & 0xFFu), w8a_pair<T>((lo >> 8) & 0xFFu, lo >> 24), w8a_pair<T>(hi & 0xFFu, (hi >> 16) & 0xFFu), w8a_pair<T>((hi >> 8) & 0xFFu, hi >> 24));
}

typedef __attribute__((ext_vector_type(4))) float w4a_f32x4;
template <class T>
__device__ __forceinline__ w4a_f32x4 w4a_mfma(const uint4 &a, const uint4 &b, const w4a_f32x4 &c) {
    if constexpr (std::is_same<T, F16>::value) return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b), c, 0, 0, 0);
    else return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
}
// lanes 16..31 and 48..63 of a for lanes 0..15 and 32..47 of b
__device__ __forceinline__ void w4a_swap16(u32 &a, u32 &b) {
    const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
    a = r[0], b = r[1];
}
__device__ __forceinline__ void w4a_swap32(u32 &a, u32 &b) {  // the upper lanes of a for the lower ones of b
    const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
    a = r[0], b = r[1];
}
// lanes 0..7 of every 16 (LOW: for themselves, else 8..15) to lanes AT .. + 7, the others zero
template <bool LOW, int AT>
__device__ __forceinline__ u32 w4a_eight(u32 v) {
    constexpr int from = LOW ? 0 : 8, ctrl = from == AT ? 0xE4 : 0x128;  // quad_perm 0 1 2 3 / row_ror:8
    return (u32)__builtin_amdgcn_update_dpp(0, (int)v, ctrl, 0xF, AT ? 0xC : 0x3, false);
}
template <bool LOW, int AT>
__device__ __forceinline__ uint4 w4a_eight(const uint4 &v) { return make_uint4(w4a_eight<LOW, AT>(v.x), w4a_eight<LOW, AT>(v.y), w4a_eight<LOW, AT>(v.z), w4a_eight<LOW, AT>(v.w)); }

template <class T, int MT, int SPW, int D, int BITS = 4>
__global__ void __launch_bounds__(512) k_w4a_gemm(const W4aArgs a, const W4mRope rp) {
    constexpr int PC = BITS / 4, TILE = BITS == 8 ? W8M_TILE_BYTES : W4M_TILE_BYTES;  // code pieces (16 bytes a lane) of a tile; bytes of one
    constexpr int KW = 8, RB = (MT + 15) / 16;                  // K-phases = waves; blocks of 16 rows
    constexpr bool PAIR = MT == 8;                              // rows 8..15 of a product: the strip's odd columns
    constexpr int XL = PAIR ? 1 : 2 * RB;                       // loads of x per step, 1 KiB each
    constexpr int AC = PAIR ? 1 : 2 * RB;                       // accumulators of a strip: [block][even, odd columns]
    constexpr int RSTR = 36, BLK = MT * RSTR * 4;               // reduction: one (phase, strip) block, rows of 32 + 4 floats
    constexpr unsigned NOWHERE = 0x80000000u;
    static_assert(SPW <= 4 && D * (XL + 1 + SPW * PC) <= 63, "a strip to 16 lanes of the scales' load; loads in flight");
    __shared__ __attribute__((aligned(16))) char smem[KW * SPW * BLK];
    const int lane = threadIdx.x & 63, p = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int c16 = lane & 15, r16 = lane >> 4;
    const int all_groups = a.K >> 6;
    const int g_lo = blockIdx.y * a.groups + p, g_hi = min(all_groups, ((int)blockIdx.y + 1) * a.groups);  // this wave's groups: g_lo, g_lo + 8, ..
    const int steps = g_hi > g_lo ? (g_hi - g_lo + KW - 1) / KW : 0;
    const int strip0 = blockIdx.x * a.strips, n_strips = min(a.strips, (a.N >> 5) - strip0);
    const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc(const_cast<char *>(a.w4m), 0, (a.N >> 5) * all_groups * TILE, 0x00020000);
    const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(const_cast<u16 *>(a.x), 0, a.M * a.K * 2, 0x00020000);
    // lanes by 16: the even and the odd columns' codes of a k-step's first eight numbers, of its other eight; the scales of strips 0 .. 3, an even and an odd column's
    const unsigned code_at = 16u * (32 * (r16 >> 1) + 2 * c16 + (r16 & 1)), scale_at = r16 < n_strips ? (unsigned)(r16 * all_groups * TILE) + 1024u * PC + 8u * c16 : NOWHERE;
    unsigned strip_at[SPW], gone[SPW];
#pragma unroll
    for (int s = 0; s < SPW; ++s) strip_at[s] = (unsigned)((strip0 + s) * all_groups + g_lo) * TILE, gone[s] = s < n_strips ? 0u : NOWHERE;
    // A product takes 32 columns of x: runs of eight 0, 2, 1, 3 of one half of a group (as the tile's words lie), a run to 16 lanes.  PAIR: the lanes of rows 8..15 load the group's other half
    unsigned x_at[RB];
#pragma unroll
    for (int t = 0; t < RB; ++t) {
        const int r = PAIR ? c16 & 7 : 16 * t + c16;
        x_at[t] = r < a.M ? (unsigned)(r * a.K + 16 * (r16 & 1) + 8 * (r16 >> 1) + (PAIR ? 32 * (c16 >> 3) : 0)) * 2u : NOWHERE;  // (rows past the end are zeros)
    }
    typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
    typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
    u32x4 xv[D][XL], cw[D][SPW][PC];  // (as vectors: split into words they would be copied from round to round, waited for right behind their loads)
    u32x2 sb[D];
    auto issue = [&](int d, int j) {
        const unsigned dead = j < steps ? 0u : NOWHERE, o = (unsigned)j * (KW * TILE), xo = (unsigned)(g_lo + j * KW) * 128u;
#pragma unroll
        for (int t = 0; t < XL; ++t) xv[d][t] = __builtin_amdgcn_raw_buffer_load_b128(xr, (x_at[PAIR ? 0 : t >> 1] | dead) + 64u * (t & 1), xo, 0);
        sb[d] = __builtin_amdgcn_raw_buffer_load_b64(wr, scale_at | dead, strip_at[0] + o, 2);
#pragma unroll
        for (int s = 0; s < SPW; ++s)
#pragma unroll
            for (int q = 0; q < PC; ++q) cw[d][s][q] = __builtin_amdgcn_raw_buffer_load_b128(wr, (code_at | gone[s] | dead) + 1024u * q, strip_at[s] + o, 2);
        __builtin_amdgcn_sched_barrier(0);  // (the loads stay in the order that the compiler's counted waits rely on)
    };
    if (steps > 0)
#pragma unroll
        for (int d = 0; d < D; ++d) issue(d, d);
    const w4a_f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
    w4a_f32x4 acc[SPW][AC];
#pragma unroll
    for (int s = 0; s < SPW; ++s)
#pragma unroll
        for (int i = 0; i < AC; ++i) acc[s][i] = zero;
    const u32 one = std::is_same<T, F16>::value ? 0x3C003C00u : 0x3F803F80u;
    const uint4 ones = make_uint4(one, one, one, one);
    auto words = [](const u32x4 &v) { return make_uint4(v.x, v.y, v.z, v.w); };
    auto compute = [&](int d) {
        uint4 xa[PAIR ? 4 : XL];  // PAIR: the group's halves as rows 0..7, as rows 8..15
        if constexpr (PAIR) xa[0] = w4a_eight<true, 0>(words(xv[d][0])), xa[1] = w4a_eight<false, 0>(words(xv[d][0])), xa[2] = w4a_eight<true, 8>(words(xv[d][0])), xa[3] = w4a_eight<false, 8>(words(xv[d][0]));
        else
#pragma unroll
            for (int t = 0; t < XL; ++t) xa[t] = words(xv[d][t]);
        w4a_f32x4 xs[RB];
#pragma unroll
        for (int t = 0; t < RB; ++t) xs[t] = w4a_mfma<T>(xa[2 * t + 1], ones, w4a_mfma<T>(xa[2 * t], ones, zero));
        if constexpr (PAIR) xs[0] = w4a_mfma<T>(xa[3], ones, w4a_mfma<T>(xa[2], ones, xs[0]));
        u32 sw[4][2];  // every lane's scale word of a strip's even, of its odd column; PAIR: the one of the rows that it sums
        {
            u32 e0 = sb[d].x, e1 = sb[d].x, o0 = sb[d].y, o1 = sb[d].y;
            w4a_swap16(e0, e1), w4a_swap16(o0, o1);  // strips 0 0 2 2, 1 1 3 3
            if constexpr (PAIR) {
                w4a_swap32(e0, o0), w4a_swap32(e1, o1);
                sw[0][0] = e0, sw[2][0] = o0, sw[1][0] = e1, sw[3][0] = o1;
            } else {
                sw[0][0] = sw[2][0] = e0, sw[1][0] = sw[3][0] = e1, sw[0][1] = sw[2][1] = o0, sw[1][1] = sw[3][1] = o1;
#pragma unroll
                for (int s = 0; s < 2; ++s) w4a_swap32(sw[s][0], sw[s + 2][0]), w4a_swap32(sw[s][1], sw[s + 2][1]);
            }
        }
#pragma unroll
        for (int s = 0; s < SPW; ++s) {
            float sc[2], bi[2];
#pragma unroll
            for (int h = 0; h < (PAIR ? 1 : 2); ++h) sc[h] = lo_f32<T>(sw[s][h]), bi[h] = BITS == 8 ? hi_f32<T>(sw[s][h]) : fmaf(-w4a_offset<T>(), sc[h], hi_f32<T>(sw[s][h]));
            uint4 wf[2][2];  // [even, odd columns][half of the group]
            if constexpr (BITS == 8) {
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    uint4 c = words(cw[d][s][h]);
                    w4a_swap16(c.x, c.z), w4a_swap16(c.y, c.w);
                    wf[0][h] = w8a_codes<T>(c.x, c.y), wf[1][h] = w8a_codes<T>(c.z, c.w);
                }
            } else {
                uint4 c = words(cw[d][s][0]);
                w4a_swap16(c.x, c.y), w4a_swap16(c.z, c.w);
                wf[0][0] = w4a_codes<T>(c.x), wf[1][0] = w4a_codes<T>(c.y), wf[0][1] = w4a_codes<T>(c.z), wf[1][1] = w4a_codes<T>(c.w);
            }
            if constexpr (PAIR) {
                w4a_f32x4 dot = w4a_mfma<T>(xa[1], wf[0][1], w4a_mfma<T>(xa[0], wf[0][0], zero));
                dot = w4a_mfma<T>(xa[3], wf[1][1], w4a_mfma<T>(xa[2], wf[1][0], dot));
#pragma unroll
                for (int i = 0; i < 4; ++i) acc[s][0][i] = fmaf(bi[0], xs[0][i], fmaf(sc[0], dot[i], acc[s][0][i]));
            } else {
#pragma unroll
                for (int t = 0; t < RB; ++t)
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        const w4a_f32x4 dot = w4a_mfma<T>(xa[2 * t + 1], wf[h][1], w4a_mfma<T>(xa[2 * t], wf[h][0], zero));
#pragma unroll
                        for (int i = 0; i < 4; ++i) acc[s][2 * t + h][i] = fmaf(bi[h], xs[t][i], fmaf(sc[h], dot[i], acc[s][2 * t + h][i]));
                    }
            }
        }
    };
    if (steps > 0) {
        int base = 0;
        for (; base + D < steps; base += D) {
#pragma unroll
            for (int d = 0; d < D; ++d) {
                compute(d);
                __builtin_amdgcn_sched_barrier(0);
                issue(d, base + d + D);
            }
        }
#pragma unroll
        for (int d = 0; d < D; ++d)
            if (base + d < steps) compute(d);
    }
    // a product's lane: columns 2 c16 (+ 1), rows 4 r16 .. + 3
#pragma unroll
    for (int s = 0; s < SPW; ++s)
#pragma unroll
        for (int t = 0; t < RB; ++t)
#pragma unroll
            for (int h = 0; h < (PAIR ? 1 : 2); ++h)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int row = 4 * r16 + i, m = PAIR ? row & 7 : 16 * t + row, col = 2 * c16 + (PAIR ? row >> 3 : h);
                    *reinterpret_cast<float *>(smem + (p * SPW + s) * BLK + (m * RSTR + col) * 4) = acc[s][PAIR ? 0 : 2 * t + h][i];
                }
    __syncthreads();
    const int EPI = a.epi;
    for (int o = threadIdx.x; o < MT * SPW * 4; o += 512) {  // a row's eight columns
        const int m = o / (4 * SPW), ts = (o >> 2) % SPW, ec = o & 3, col = 32 * (strip0 + ts) + 8 * ec;
        if (m >= a.M || ts >= n_strips) continue;
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
