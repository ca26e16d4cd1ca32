// w4a_gemm.hpp -- int4 (int8) g=64 x T GEMM for 3 to 16 (1 to 32) rows with the scales and biases applied to the sums: y = sum over groups of s (q . x) + b sum(x), the weights never rounded to T
// (mx.quantized_matmul's row-by-row arithmetic: models/llama/language.py:83,108,127).  (Included by w4m_gemm.hip.)
//
// k_w4r_gemm turns every weight into T in front of its product, 17 vector instructions per eight of them, and its waves wait for each other at every step for the x that they share.  For a
// few rows that is most of its time.  Here
//   * the codes are operands as they stand -- bf16: under the exponent of 128, one v_and_or for two, f16: less 1024 -- and a group's products are multiplied by its scale and joined by bias
//     times the group's sum of x (another product, by ones) in fp32;
//   * products are 16 x 16 x 32: sixteen rows and sixteen columns, the even or the odd ones of a strip, of int8 one half of it (a v_permlane16_swap of two words makes two such operands of a
//     tile's).  Up to eight rows, rows 8..15 of a product are the same rows against the strip's other columns (zeros in the others' place), so that no lane of the sums is idle;
//   * a wave's K-phase is its own: it loads the x of its groups as whole lines, eight lanes to a row, turns them into operands in LDS of its own without a barrier, and waits for nothing but its
//     loads, all of them ordinary ones, so that the compiler's waits are exact; the scales of a step's four strips are one load.  (x loaded straight into the operand's lanes: sixteen lanes side by
//     side are sixteen rows, and each takes the load pipe a turn of its own.  Waves that share a CU with few strips and walk a long K then wait for x: us, that / this, [2048, 5632] 8 int4 rows 8.0 / 6.8, 32 int8
//     rows 15.5 / 11.9, [10240, 8192] 8 int4 rows 13.7 / 12.6, 8 / 32 int8 rows 18.7 / 17.1, 27.0 / 24.0.  Two steps, [4096, 4096] in four splits, pay 0.1 to 0.3 us for the way through LDS: 4.5 / 4.6.)
// Bound by the stream and a launch (3 us).  us, weights from HBM, k_w4r_gemm / 32 x 32 products with x by LDS-DMA / this, 8 rows: gate|up [28672, 4096] 17.2 / 15.4 / 13.4, down [4096, 14336] 10.2 / 9.9 / 8.3,
// q|k|v [6144, 4096] 6.9 / 6.5 / 5.7, o [4096, 4096] 5.4 / 5.1 / 4.6, head [32768, 4096] 17.4 / 15.2 / 14.2; [16384, 3072] 9.2 / 9.3 / 7.5, [3072, 8192] 6.9 / 6.5 / 5.6, [2048, 5632] 8.6 / 7.6 / 6.8,
// [10240, 8192] 15.5 / 14.2 / 12.6.  16 rows, k_w4r_gemm / this: 17.3 / 14.9, 10.8 / 8.9, 7.1 / 6.2, 5.6 / 4.8, 19.6 / 15.6, 9.2 / 8.2, 7.0 / 6.2, 8.8 / 8.0, 16.0 / 14.3.  32 rows of int4 are k_w4r_gemm's (gate|up 18.5 / 21.4).
// Two steps in flight per wave are enough (three with one strip and eight rows: 256 strips of 8192 columns 10.5 / 9.7 us; three with four strips cost gate|up 1 us, sixteen waves gain nothing).  The last D
// steps of a wave load nothing; where D does not divide the steps, the round before them still issues the loads of a step or two past the end, which return nothing.  Both loops need the ring as whole vectors, see there.
// Error (2-norm, before the rounding to T, eight shapes, normal x) against 64 bits: 1.1e-6, that of the 32 x 32 products too; of weights rounded to bf16 1.7e-3.
#pragma once

constexpr int W4A_ROWS = 16, W8A_ROWS = 32;
constexpr int W8M_TILE_BYTES = 2176;  // W8M (below)
struct W4aArgs {
    const char *w4m;   // W4M (W8M) tiles of the [N, K] matrix
    const u16 *x;      // [M, K]
    int M, N, K;
    int halves;        // half strips (16 columns) per workgroup; int4: an even number
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

// Int8 codes, W8M tiles: as W4M, 32 rows x 64 columns, two pieces of 1 KiB and the 32 {scale, bias} words (of rows 0, 16, 1, 17, ..): lane l = 32 kh + n holds in piece h the codes of row n of k-steps 2 h and 2 h + 1, two words
// each, in the W8S word format (codes 0, 2, 1, 3).  Up to 255 a code is a bf16 and an f16 as it stands.
// The tile's halves are a product's two operands as they are read, so that a workgroup may take half strips of 16 columns and the lanes of the other half load nothing; a word of one half's scales
// lies beside the other half's.
// Bound by the stream, half the bytes of a 16-bit copy's.  us, the form with 32 x 32 products / this, 8 rows: gate|up 22.2 / 21.2, down 12.7 / 11.8, q|k|v 8.2 / 7.1, o 6.3 / 5.5, head 23.7 / 22.9, [2048, 5632] 7.8 / 7.6,
// [10240, 8192] 18.5 / 17.1; 32 rows: 25.7 / 25.8, 16.2 / 15.1, 11.1 / 9.9, 8.5 / 7.0, 27.3 / 27.0, 12.6 / 11.9, 24.7 / 24.0.  Slower than that form: 17 to 32 rows of 513 to 800 strips, by 2 to 3 %.
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
template <class T, int MT, int SPW, int D, int BITS = 4>
__global__ void __launch_bounds__(512) k_w4a_gemm(const W4aArgs a, const W4mRope rp) {
    constexpr int PC = BITS / 4, TILE = BITS == 8 ? W8M_TILE_BYTES : W4M_TILE_BYTES;  // code pieces (16 bytes a lane) of a tile; bytes of one
    constexpr int KW = 8, RB = (MT + 15) / 16;                  // K-phases = waves; blocks of 16 rows
    constexpr bool PAIR = MT == 8;                              // rows 8..15 of a product: the strip's other columns
    constexpr int XL = MT / 8, XB = MT * 128 + (PAIR ? 16 : 0); // loads of x per step, 1 KiB each; a wave's image of them
    constexpr int AC = PAIR ? 1 : 2 * RB;                       // accumulators of a strip: [block][operand]
    constexpr int RSTR = 36, BLK = MT * RSTR * 4;               // reduction: one (phase, strip) block, rows of 32 + 4 floats
    constexpr unsigned NOWHERE = 0x80000000u;
    static_assert(SPW <= 4 && D * (XL + 1 + SPW * PC) <= 63, "a strip to 16 lanes of the scales' load; loads in flight");
    constexpr bool APART = KW * (SPW * BLK + XB) <= 80 * 1024;  // the sums beside the images, two workgroups to a CU; else in their place
    __shared__ __attribute__((aligned(128))) char smem[KW * (APART ? SPW * BLK + XB : SPW * BLK > XB ? SPW * BLK : XB)];
    const int lane = threadIdx.x & 63, p = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int c16 = lane & 15, r16 = lane >> 4;
    const int all_groups = a.K >> 6;
    const int g_lo = blockIdx.y * a.groups + p, g_hi = min(all_groups, ((int)blockIdx.y + 1) * a.groups);  // this wave's groups: g_lo, g_lo + 8, ..
    const int steps = g_hi > g_lo ? (g_hi - g_lo + KW - 1) / KW : 0;
    const int h0 = blockIdx.x * a.halves, h1 = min(h0 + a.halves, a.N >> 4), strip0 = h0 >> 1, n_strips = ((h1 + 1) >> 1) - strip0;
    const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc(const_cast<char *>(a.w4m), 0, (a.N >> 5) * all_groups * TILE, 0x00020000);
    const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(const_cast<u16 *>(a.x), 0, a.M * a.K * 2, 0x00020000);
    // lanes by 16: one and the other operand's columns (int4: the even, the odd ones; int8: the strip's halves) of a k-step's first eight numbers, of its other eight; the scales of strips 0 .. 3, a column
    // of each operand
    const unsigned code_at = 16u * (BITS == 8 ? lane : 32 * (r16 >> 1) + 2 * c16 + (r16 & 1)), scale_at = r16 < n_strips ? (unsigned)(r16 * all_groups * TILE) + 1024u * PC + 8u * c16 : NOWHERE;
    unsigned strip_at[SPW], gone[SPW];
#pragma unroll
    for (int s = 0; s < SPW; ++s) {
        const int h = 2 * (strip0 + s) + (BITS == 8 ? r16 & 1 : 0);
        strip_at[s] = (unsigned)((strip0 + s) * all_groups + g_lo) * TILE, gone[s] = h >= h0 && h < h1 ? 0u : NOWHERE;
    }
    // A group of eight rows of x is one load of whole lines, eight lanes to a row; the wave's own LDS turns it into the operands: runs of eight columns 0, 2, 1, 3 of one half of a group (as the tile's
    // words lie), a run to 16 lanes; a row's pieces rotated by the row.  PAIR: the lanes of the other rows read zeros
    unsigned x_at[XL];
#pragma unroll
    for (int i = 0; i < XL; ++i) {
        const int r = 8 * i + (lane >> 3);
        x_at[i] = r < a.M ? (unsigned)(r * a.K + 8 * (lane & 7)) * 2u : NOWHERE;  // (rows past the end are zeros)
    }
    char *x_lds = smem + (APART ? KW * SPW * BLK : 0) + p * XB;
    char *x_put = x_lds + (lane >> 3) * 128 + (((lane & 7) ^ (lane >> 3)) << 4);
    const int run = 2 * (r16 & 1) + (r16 >> 1), xrow = PAIR ? c16 & 7 : c16;
    const char *x_get[2];  // a half of the group each
#pragma unroll
    for (int h = 0; h < 2; ++h) x_get[h] = x_lds + xrow * 128 + (((4 * h + run) ^ (xrow & 7)) << 4);
    if (PAIR && lane < 4) *reinterpret_cast<u32 *>(x_lds + MT * 128 + 4 * lane) = 0;
    typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
    typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
    u32x4 xv[D][XL], cw[D][SPW][PC];  // (as vectors: split into words they would be copied from round to round, waited for right behind their loads)
    u32x2 sb[D];
    auto issue = [&](int d, int j) {
        const unsigned dead = j < steps ? 0u : NOWHERE, o = (unsigned)j * (KW * TILE), xo = (unsigned)(g_lo + j * KW) * 128u;
#pragma unroll
        for (int t = 0; t < XL; ++t) xv[d][t] = __builtin_amdgcn_raw_buffer_load_b128(xr, x_at[t] | dead, xo, 0);
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
        uint4 xa[PAIR ? 4 : 2 * RB];  // [block][half]; PAIR: the group's halves as rows 0..7, as rows 8..15
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // (the wave's lanes meet in LDS, whose operations go in order)
#pragma unroll
        for (int t = 0; t < XL; ++t) *reinterpret_cast<u32x4 *>(x_put + 1024 * t) = xv[d][t];
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int t = 0; t < (PAIR ? 4 : 2 * RB); ++t) {
            const char *q = PAIR ? (t >> 1) == (c16 >> 3) ? x_get[t & 1] : x_lds + MT * 128 : x_get[t & 1] + 2048 * (t >> 1);
            xa[t] = *reinterpret_cast<const uint4 *>(q);
        }
        w4a_f32x4 xs[RB];
#pragma unroll
        for (int t = 0; t < RB; ++t) xs[t] = w4a_mfma<T>(xa[2 * t + 1], ones, w4a_mfma<T>(xa[2 * t], ones, zero));
        if constexpr (PAIR) xs[0] = w4a_mfma<T>(xa[3], ones, w4a_mfma<T>(xa[2], ones, xs[0]));
        u32 sw[4][2];  // every lane's scale word of a strip's column of one, of the other operand; PAIR: the one of the rows that it sums
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
            uint4 wf[2][2];  // [operand][half of the group]
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
    if (!APART) __syncthreads();
    // a product's lane: columns 2 c16 (+ 1), int8 c16 (+ 16), rows 4 r16 .. + 3
#pragma unroll
    for (int s = 0; s < SPW; ++s)
#pragma unroll
        for (int t = 0; t < RB; ++t)
#pragma unroll
            for (int h = 0; h < (PAIR ? 1 : 2); ++h)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int row = 4 * r16 + i, m = PAIR ? row & 7 : 16 * t + row, o = PAIR ? row >> 3 : h, col = BITS == 8 ? c16 + 16 * o : 2 * c16 + o;
                    *reinterpret_cast<float *>(smem + (p * SPW + s) * BLK + (m * RSTR + col) * 4) = acc[s][PAIR ? 0 : 2 * t + h][i];
                }
    __syncthreads();
    const int EPI = a.epi;
    for (int o = threadIdx.x; o < MT * SPW * 4; o += 512) {  // a row's eight columns
        const int m = o / (4 * SPW), ts = (o >> 2) % SPW, ec = o & 3, col = 32 * (strip0 + ts) + 8 * ec;
        if (m >= a.M || col >> 4 < h0 || col >> 4 >= h1) continue;
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
