// prefill_attn.hpp -- causal flash attention for prompt chunks on the MFMA units (head_dim 128 or 64).
//
// Replaces mx.fast.scaled_dot_product_attention(q, k, v, scale, mask=causal) at models/base.py:111-113 for L > 1
// (mask built by models/base.py:18-53: query row r at absolute position offset + r sees keys 0 .. offset + r).
// The VALU decode kernel run once per query row costs 27 wave-instructions per (query, key, kv-group): O(L^2) and the
// whole prefill beyond ~1k tokens.  Here one workgroup owns (32 query rows) x (one kv-head group); wave w owns q-head
// g*REP + w, so a staged K/V block serves all q-heads of the group.
//
// Per block of 64 keys (32 where fewer than four waves share it), per wave (v_mfma_f32_32x32x16, fp32 accumulators):
//   S^T[key, row]  = K . Q^T        2 x 8 MFMAs, two chains side by side;  A = K rows from the LDS image (ds_read_b128), B = Q fragments kept in VGPRs.
//                                   Orientation chosen so the softmax reduction runs over REGISTERS (keys), not lanes,
//                                   and so P^T is directly the B operand of the next product (no lane movement);
//   online softmax in fp32, base 2 (one fma and one v_exp_f32 per score; a block that every row sees whole -- all but a tile's last ones -- takes no mask),
//                                   running max / sum per query row = per lane pair;
//   O^T[dim, row] += V^T . P^T      A = V^T via ds_read_b64_tr_b16 (hardware transpose of the row-major V image),
//                                   B = P^T split into hi + lo halves of T (2 x 16 MFMAs, four chains): P keeps ~16 mantissa bits, the
//                                   "fp32 until one rounding" contract of the fused kernel within 2^-17.
// K/V blocks are fetched to registers one block ahead and written to one of two swizzled LDS images (the guide's dual-use
// layout (b): conflict-free for both the row reads and the transposed reads): one barrier per block.
// What bounds it: the vector instructions between the products, and, while few workgroups run, one block's chain of latencies.  Blocks of 32 keys masked element by element, two barriers
// and 25 instead of 12 instructions per pair of scores took, for 32 / 8 heads of 128: 4096 rows 303 us (now 227 = 0.9 PFLOP/s with the split P), 1024 rows 60 (38), 509 rows 30 (22),
// 37 rows behind 900 cached ones 54 (35; with the keys split 18).
#pragma once
#include "attention.hpp"
#include "common.hpp"

#include <type_traits>

typedef short v4i16_t __attribute__((ext_vector_type(4)));
typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_t;
typedef __attribute__((ext_vector_type(8))) _Float16 f16x8_t;
typedef __attribute__((ext_vector_type(16))) float f32x16_t;

struct PrefillAttnArgs {
    const u16 *q;                        // [M, Hq, D]
    const unsigned long long *kv_table;  // K buffers then V buffers, [Hkv, cap, D] each
    int layer, n_layers;
    const DecState *state;               // pos = offset of row 0, cap  (decoder) ...
    const u16 *k, *v;                    // ... or direct [Hkv, cap, D] buffers with host-side offset / capacity (op-level, state == nullptr)
    int offset, cap;
    int M, Hq, Hkv;
    float scale;
    u16 *out;                            // [M, Hq, D]
    // SEG instantiation (vision tower: block-diagonal, non-causal attention -- the mask of models/intern/vision.py:160-167):
    // query row r attends keys [seg_lo[r], seg_hi[r]); both int32 [M], non-decreasing in r.  Op level only (k, v, cap = M).
    const int *seg_lo, *seg_hi;
    int out_d;                           // SEG: columns of a head's output that are stored (a multiple of 4; 0: D): heads of 80, padded to 128 for the products, side by side again
    const int *block_table;              // paged KV (nullable, decoder only): kv_table holds the layers' slab K / V bases; key t
    int n_pages;                         //   lives in page block_table[t / 64] (each [Hkv, 64, D]) at row t % 64
    int before;                          // keys in front of the first row, as far as the host knows (plans the launch; the device's position decides)
    int splits;                          // SPLIT instantiation: workgroups along the keys (gridDim.y); their partial sums meet in k_prefill_combine
    float *part;                         //   [M, Hq, splits] x {[D] weighted sums}, then [M, Hq, splits] x {running max, sum}
    const u16 *rot_bias;                 // ROT instantiation: q = the qkv Linear's rows [M, 3, Hq, DR], without its bias; the bias
    const float *rot_cos, *rot_sin;      //   rotate-half angles, fp32 [M, DR / 2]
};

template <class T> struct MfmaT;
template <> struct MfmaT<BF16> {
    static __device__ __forceinline__ f32x16_t run(const uint4 &a, const uint4 &b, const f32x16_t &c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
    }
};
template <> struct MfmaT<F16> {
    static __device__ __forceinline__ f32x16_t run(const uint4 &a, const uint4 &b, const f32x16_t &c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b), c, 0, 0, 0);
    }
};

constexpr float PA_RISE = 8.0f;  // log2: see k_prefill_attn

// two fp32 -> one packed pair of T in a single v_cvt_pk
template <class T>
__device__ __forceinline__ u32 pa_pack2(float lo, float hi) {
    typedef float f2_t __attribute__((ext_vector_type(2)));
    typedef typename std::conditional<std::is_same<T, F16>::value, _Float16, __bf16>::type e_t;
    typedef e_t e2_t __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(u32, __builtin_convertvector((f2_t){lo, hi}, e2_t));
}

// byte offset of 16-byte chunk `ch` (0 .. D/8-1) of row `row` (0..31) in a [32][D x 16-bit] LDS tile: the guide's dual-use
// swizzle (b) for 256-byte rows; for D = 64 the same XOR folded to the row's 8 chunks (a bijection inside the row, which is
// all correctness needs -- both the writes and the two kinds of reads go through it)
template <int I, int N, class F>
__device__ __forceinline__ void pa_static_for(F &&f) {
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        pa_static_for<I + 1, N>(f);
    }
}

template <int D>
__device__ __forceinline__ int pa_off(int row, int ch) {
    return 2 * D * row + 16 * (ch ^ ((((row & 3) << 2) | ((row >> 2) & 3)) & (D / 8 - 1)));
}

// QT: 32-row query tiles per workgroup (1 or 2).  With QT = 2 the workgroup has 2*REP waves -- waves [0, REP) own the first
// tile, [REP, 2 REP) the second -- and one staged K/V block serves 64 query rows: half the L2 -> LDS traffic and barriers per
// unit of work, at the same number of waves per CU (one 8-wave workgroup instead of two 4-wave ones for REP = 4).
// SPLIT: blockIdx.y takes its share of the tile's key blocks and leaves its sums to k_prefill_combine (prefill_attn_splits says when).
// SHORT: blocks of 32 keys, for prompts that fill few of 64 (prefill_attn_short).
// KG = 2: two waves per head and tile, which take a staged block's first and second 64 keys and meet in LDS at the end: half the serial blocks, and a wave's softmax beside the other's
// products (prefill_attn_pairs says when).
// DR: a head's columns, side by side in memory (D: what a row takes in LDS).  Heads of 80 need five steps of 16 columns for their scores and three tiles of 32 for their sums, not the eight and four of 128,
// and no padding.  The 7B vision tower's widths, 1024 patches, us: windows of 64 7.9 -> 6.6, whole image 54 -> 46.
// ROT: windows straight from the qkv Linear's rows: bias and rotation on the way into LDS, by twice the waves (the second half of them does nothing else), queries and the first 64 keys asked for before anything
// waits; with the blocks of 32 keys of the others, so that the sums are theirs bit for bit.  Bound by the chain bounds -> rows -> LDS -> scores of one round of workgroups.  A window's keys are rotated once
// per 64 query rows that see them; rotated in a launch of their own, as a whole image's and long windows' still are (32 tiles would each rotate all keys), they cost 8 us beside the attention's 6.6, here 10.1 in all (12.0 with
// as many waves as tiles and no early queries).
template <class T, int D, int REP, int QT, bool SEG = false, bool SPLIT = false, bool SHORT = false, int KG = 1, int DR = D, bool ROT = false>
__global__ void __launch_bounds__(REP * QT * KG * 64 * (ROT ? 2 : 1), 2) k_prefill_attn(const PrefillAttnArgs a) {
    static_assert(DR == D || (SEG && DR % 16 == 0 && DR < D), "narrower rows: segments");
    static_assert(!ROT || (SEG && REP == 1), "rotation on the way in: segments of plain heads");
    static_assert(KG == 1 || (KG == 2 && QT == 1 && !SEG && !SHORT), "two waves per tile: causal, one tile");
    constexpr int NT = REP * QT * KG * 64 * (ROT ? 2 : 1), NB = (NT >= 256 && !SHORT && !ROT) || KG == 2 ? 2 : 1, BK = 32 * NB * KG;  // keys per block: 64 (a wave's) where enough threads share their loads
    constexpr int CH = DR / 8, KS = DR / 16, DT = (DR + 31) / 32;              // chunks per row, k-steps of Q.K^T, 32-dim output tiles (of columns past DR nothing is stored)
    constexpr int BM = 32 * QT;
    constexpr int CPT = (BK * CH + NT - 1) / NT;                                   // 16-byte chunks per thread and tile
    __shared__ __attribute__((aligned(16))) char kv_lds[2][2][BK * 2 * D];         // [block parity][K, V]
    const int lane = threadIdx.x & 63, wave_id = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const bool helper = ROT && wave_id >= REP * QT;  // (ROT: as many waves again, which only bring rows in)
    const int wave = KG == 2 ? wave_id % REP : ROT ? wave_id % (REP * QT) : wave_id, kg = KG == 2 ? wave_id / REP : 0;  // (kg: which half of a block's keys)
    const int c = lane & 31, h = lane >> 5;
    // XCD-aware tile mapping: workgroups go round-robin over the 8 XCDs by linear id, so the kv-head group is the FASTEST
    // index (id % Hkv): with 8 kv-heads every XCD's L2 only ever holds one group's K/V (4 MB at 4096 tokens) instead of all
    // of them.  Query tiles longest first (a tile's work grows with its position: causal).
    const int g = (int)blockIdx.x % a.Hkv, tile = (int)blockIdx.x / a.Hkv;
    const int wg_r0 = ((a.M + BM - 1) / BM - 1 - tile) * BM;                  // first query row of the workgroup
    const int r0 = wg_r0 + 32 * (wave / REP), hq = g * REP + wave % REP;     // this wave's 32-row tile and q-head
    // paged KV: a key block (BK = 32 or 64 rows) never straddles a 64-row page, so its page is one scalar table lookup per fetch (KG = 2: two);
    // the contiguous case is the same code with one "page" of `cap` rows (mask keeps every row bit, page offset 0)
    const bool paged = a.block_table != nullptr;
    const int pos0 = a.state ? a.state->pos : a.offset, cap = paged ? 64 : a.state ? a.state->cap : a.cap;
    const int row_mask = paged ? 63 : 0x7FFFFFFF;
    const size_t page_elems = (size_t)2 * 64 * a.Hkv * D;
    const int r_last = (wg_r0 + BM - 1 < a.M ? wg_r0 + BM - 1 : a.M - 1);
    // ROT: this workgroup's query rows, asked for before the bounds are known
    constexpr int HC = DR / 16, QI = ROT ? (BM * HC + NT - 1) / NT : 1;  // 16-byte pieces of half a head; (row, piece of the lower half)s per thread
    const size_t qkv_ld = (size_t)3 * a.Hq * DR;
    __shared__ __attribute__((aligned(16))) char q_lds[ROT ? BM * 2 * D : 16];
    uint4 q_half[QI][2];
    float4 q_turn[QI][4];
    auto turns = [&](int t, int c, float4(&o)[4]) {  // cosines, sines of piece c
        const float4 *cp = reinterpret_cast<const float4 *>(a.rot_cos + (size_t)t * (DR / 2) + 8 * c), *sp = reinterpret_cast<const float4 *>(a.rot_sin + (size_t)t * (DR / 2) + 8 * c);
        o[0] = cp[0], o[1] = cp[1], o[2] = sp[0], o[3] = sp[1];
    };
    if constexpr (ROT)
#pragma unroll
        for (int i = 0; i < QI; ++i) {
            const int x = min((int)threadIdx.x + i * NT, BM * HC - 1), c = x % HC, t = min(wg_r0 + x / HC, a.M - 1);
            const u16 *row = a.q + t * qkv_ld + (size_t)g * DR + 8 * c;
            q_half[i][0] = *reinterpret_cast<const uint4 *>(row), q_half[i][1] = *reinterpret_cast<const uint4 *>(row + DR / 2);
            turns(t, c, q_turn[i]);
        }
    // last / first key any row of this tile attends (segment bounds are non-decreasing in the row index)
    // (bounds clamped to the buffer: a bad segment table must not become a wild address)
    const int t_last = SEG ? max(min(a.seg_hi[r_last], a.cap), 1) - 1 : pos0 + r_last;
    const int n_all = t_last / BK + 1, share = SPLIT ? (n_all + a.splits - 1) / a.splits : n_all;  // (key blocks of the tile, and of this workgroup)
    const int b_first = SEG ? min(max(a.seg_lo[wg_r0], 0), t_last) / BK : SPLIT ? (int)blockIdx.y * share : 0;
    const int n_blocks = SPLIT ? min(b_first + share, n_all) : n_all;
    if constexpr (SPLIT)
        if (b_first >= n_blocks) {  // fewer blocks than workgroups: an empty share weighs nothing
            if (h == 0 && kg == 0 && r0 + c < a.M) {
                float *ml = a.part + (size_t)a.M * a.Hq * a.splits * D + (((size_t)(r0 + c) * a.Hq + hq) * a.splits + blockIdx.y) * 2;
                ml[0] = ATTN_NEG, ml[1] = 0.0f;
            }
            return;
        }
    const u16 *kbase = (a.state ? reinterpret_cast<const u16 *>(a.kv_table[a.layer]) : a.k) + (size_t)g * cap * DR;
    const u16 *vbase = (a.state ? reinterpret_cast<const u16 *>(a.kv_table[a.n_layers + a.layer]) : a.v) + (size_t)g * cap * DR;

    // staging: chunk id x = threadIdx.x + i*NT -> (row = x / CH, ch = x % CH); keys past t_last are clamped (masked later).
    // Eight NAMED register pairs, used up to CPT: as arrays (even with compile-time indices) the compiler parked them in
    // scratch memory and reloaded them every block (80-272 B per lane).
    uint4 k0, k1, k2, k3, k4, k5, k6, k7, v0, v1, v2, v3, v4, v5, v6, v7;
#define PA_FETCH1(i, kr, vr)                                                                   \
    if constexpr (i < CPT) {                                                                     \
        int x = threadIdx.x + i * NT;                                                            \
        x = x < BK * CH ? x : BK * CH - 1;                                                       \
        int t = b * BK + x / CH;                                                                 \
        t = t < t_last ? t : t_last;                                                             \
        const size_t po = KG == 2 && x >= 64 * CH ? pg_off1 : pg_off;                            \
        kr = *reinterpret_cast<const uint4 *>(kbase + po + (size_t)(t & row_mask) * DR + (x % CH) * 8); \
        vr = *reinterpret_cast<const uint4 *>(vbase + po + (size_t)(t & row_mask) * DR + (x % CH) * 8); \
    }
#define PA_PUBLISH1(i, kr, vr)                                                                 \
    if constexpr (i < CPT) {                                                                     \
        const int x = threadIdx.x + i * NT;                                                      \
        if (x < BK * CH) {                                                                       \
            *reinterpret_cast<uint4 *>(kv_lds[buf][0] + pa_off<D>(x / CH, x % CH)) = kr;                  \
            *reinterpret_cast<uint4 *>(kv_lds[buf][1] + pa_off<D>(x / CH, x % CH)) = vr;                  \
        }                                                                                        \
    }
    auto page_at = [&](int t) { return paged ? (size_t)min((unsigned)a.block_table[t >> 6], (unsigned)a.n_pages - 1u) * page_elems : (size_t)0; };
    auto fetch = [&](int b) {
        const size_t pg_off = page_at(b * BK), pg_off1 = KG == 2 ? page_at(min(b * BK + 64, t_last)) : 0;
        PA_FETCH1(0, k0, v0) PA_FETCH1(1, k1, v1) PA_FETCH1(2, k2, v2) PA_FETCH1(3, k3, v3)
        PA_FETCH1(4, k4, v4) PA_FETCH1(5, k5, v5) PA_FETCH1(6, k6, v6) PA_FETCH1(7, k7, v7)
    };
    auto publish = [&](int buf) {
        PA_PUBLISH1(0, k0, v0) PA_PUBLISH1(1, k1, v1) PA_PUBLISH1(2, k2, v2) PA_PUBLISH1(3, k3, v3)
        PA_PUBLISH1(4, k4, v4) PA_PUBLISH1(5, k5, v5) PA_PUBLISH1(6, k6, v6) PA_PUBLISH1(7, k7, v7)
    };
#undef PA_FETCH1
#undef PA_PUBLISH1
    static_assert(ROT || CPT <= 8, "staging registers");
    // ROT: eight columns of a Linear's row with its bias, and a pair of eights turned as apply_rotary_pos_emb_vision has them: the terms and roundings of k_vision_qkv_rope
    auto biased = [&](const uint4 &x, const u16 *bias, float(&o)[8]) {
        const uint4 b = *reinterpret_cast<const uint4 *>(bias);
        const u32 xw[4] = {x.x, x.y, x.z, x.w}, bw[4] = {b.x, b.y, b.z, b.w};
#pragma unroll
        for (int j = 0; j < 4; ++j) o[2 * j] = round_T<T>(lo_f32<T>(xw[j]) + lo_f32<T>(bw[j])), o[2 * j + 1] = round_T<T>(hi_f32<T>(xw[j]) + hi_f32<T>(bw[j]));
    };
    auto packed = [&](const float(&o)[8]) { return make_uint4(pack2<T>(o[0], o[1]), pack2<T>(o[2], o[3]), pack2<T>(o[4], o[5]), pack2<T>(o[6], o[7])); };
    auto turned = [&](char *rows, int r, int c, const uint4 &lower, const uint4 &upper, const u16 *bias, const float4(&t)[4]) {
        float lo[8], hi[8], o[8], p[8];
        biased(lower, bias + 8 * c, lo), biased(upper, bias + DR / 2 + 8 * c, hi);
        const float cc[8] = {t[0].x, t[0].y, t[0].z, t[0].w, t[1].x, t[1].y, t[1].z, t[1].w}, ss[8] = {t[2].x, t[2].y, t[2].z, t[2].w, t[3].x, t[3].y, t[3].z, t[3].w};
#pragma unroll
        for (int j = 0; j < 8; ++j) o[j] = __fadd_rn(__fmul_rn(lo[j], cc[j]), __fmul_rn(-hi[j], ss[j])), p[j] = __fadd_rn(__fmul_rn(hi[j], cc[j]), __fmul_rn(lo[j], ss[j]));
        *reinterpret_cast<uint4 *>(rows + pa_off<D>(r, c)) = packed(o), *reinterpret_cast<uint4 *>(rows + pa_off<D>(r, c + HC)) = packed(p);
    };
    auto rotate_in = [&](int b) {  // key blocks b and b + 1, into both images
        constexpr int B2 = 2 * BK, KI = (B2 * HC + NT - 1) / NT, VI = (B2 * CH + NT - 1) / NT;
        uint4 half[KI][2], vv[VI];
        float4 turn[KI][4];
#pragma unroll
        for (int i = 0; i < KI; ++i) {
            const int x = min((int)threadIdx.x + i * NT, B2 * HC - 1), c = x % HC, t = min(b * BK + x / HC, t_last);
            const u16 *row = a.q + t * qkv_ld + (size_t)(a.Hq + g) * DR + 8 * c;
            half[i][0] = *reinterpret_cast<const uint4 *>(row), half[i][1] = *reinterpret_cast<const uint4 *>(row + DR / 2);
            turns(t, c, turn[i]);
        }
#pragma unroll
        for (int i = 0; i < VI; ++i) {
            const int x = min((int)threadIdx.x + i * NT, B2 * CH - 1), t = min(b * BK + x / CH, t_last);
            vv[i] = *reinterpret_cast<const uint4 *>(a.q + t * qkv_ld + (size_t)(2 * a.Hq + g) * DR + 8 * (x % CH));
        }
        if (b == b_first)
#pragma unroll
            for (int i = 0; i < QI; ++i) {
                const int x = threadIdx.x + i * NT;
                if (x < BM * HC) turned(q_lds, x / HC, x % HC, q_half[i][0], q_half[i][1], a.rot_bias + (size_t)g * DR, q_turn[i]);
            }
#pragma unroll
        for (int i = 0; i < KI; ++i) {
            const int x = threadIdx.x + i * NT;
            if (x < B2 * HC) turned(kv_lds[x / HC / BK][0], x / HC % BK, x % HC, half[i][0], half[i][1], a.rot_bias + (size_t)(a.Hq + g) * DR, turn[i]);
        }
#pragma unroll
        for (int i = 0; i < VI; ++i) {
            const int x = threadIdx.x + i * NT;
            if (x >= B2 * CH) break;
            float v[8];
            biased(vv[i], a.rot_bias + (size_t)(2 * a.Hq + g) * DR + 8 * (x % CH), v);
            *reinterpret_cast<uint4 *>(kv_lds[x / CH / BK][1] + pa_off<D>(x / CH % BK, x % CH)) = packed(v);
        }
    };
    if constexpr (ROT) {
        rotate_in(b_first);
        __syncthreads();
    }
    if constexpr (!ROT) fetch(b_first);

    // Q fragments (B operand of K . Q^T): lane (row c, half h), k-step s holds Q[r0 + c][hq][16 s + 8 h .. + 8]
    const int qrow = r0 + c < a.M ? r0 + c : a.M - 1;
    uint4 qf[KS];
#pragma unroll
    for (int s = 0; s < KS; ++s)
        if constexpr (ROT) qf[s] = *reinterpret_cast<const uint4 *>(q_lds + pa_off<D>(32 * wave + c, 2 * s + h));
        else qf[s] = *reinterpret_cast<const uint4 *>(a.q + ((size_t)qrow * a.Hq + hq) * DR + 16 * s + 8 * h);
    // last (and, SEG, first) key this lane's query row attends (rows past M are padding: never stored)
    const int t_row = SEG ? a.seg_hi[qrow] - 1 : pos0 + r0 + c;
    const int t_lo = SEG ? a.seg_lo[qrow] : 0;
    const float sl2 = fabsf(a.scale) * ATTN_LOG2E;  // (a negative scale turns the sign of the queries: the largest score is the largest product)
    if (a.scale < 0.0f)
#pragma unroll
        for (int s = 0; s < KS; ++s) qf[s].x ^= 0x80008000u, qf[s].y ^= 0x80008000u, qf[s].z ^= 0x80008000u, qf[s].w ^= 0x80008000u;
    // keys that every row of this wave sees: such blocks need no mask (bounds are non-decreasing in the row)
    const int wr0 = r0 < a.M ? r0 : a.M - 1, wr1 = r0 + 31 < a.M ? r0 + 31 : a.M - 1;
    const int all_hi = SEG ? a.seg_hi[wr0] - 1 : pos0 + wr0, all_lo = SEG ? a.seg_lo[wr1] : 0;

    f32x16_t oacc[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int i = 0; i < 16; ++i) oacc[dt][i] = 0.0f;
    float m_run = ATTN_NEG, l_run = 0.0f;

    // transposed-read addressing (guide T10): lane 4q+p of a 16-lane group supplies row q, columns 4p..4p+3 of a
    // 4-row x 16-column block; lane i of the group receives column i, row q in element q
    const int grp = lane >> 4, tq = (lane & 15) >> 2, tp = lane & 3;

    if constexpr (!ROT) {
        publish(0);
        __syncthreads();
    }
    for (int b = b_first; b < n_blocks; ++b) {
        const int buf = (b - b_first) & 1;
        const char *k_lds = kv_lds[buf][0] + kg * (64 * 2 * D), *v_lds = kv_lds[buf][1] + kg * (64 * 2 * D);
        if constexpr (!ROT)
            if (b + 1 < n_blocks) fetch(b + 1);
        const int t0 = b * BK + (KG == 2 ? 64 * kg : 0);
        if ((KG == 1 || t0 <= t_last) && !helper) {

        // S^T = K . Q^T : rows = keys (registers), cols = query rows (lanes); the blocks of 32 keys are independent chains
        f32x16_t sc[NB];
#pragma unroll
        for (int n = 0; n < NB; ++n)
#pragma unroll
            for (int i = 0; i < 16; ++i) sc[n][i] = 0.0f;
#pragma unroll
        for (int s = 0; s < KS; ++s)
#pragma unroll
            for (int n = 0; n < NB; ++n) {
                const uint4 kf = *reinterpret_cast<const uint4 *>(k_lds + pa_off<D>(32 * n + c, 2 * s + h));
                sc[n] = MfmaT<T>::run(kf, qf[s], sc[n]);
            }
        // online softmax over keys: register i of block n <-> key t0 + 32 n + (i & 3) + 8 (i >> 2) + 4 h
        const bool masked = t0 + 32 * NB - 1 > all_hi || (SEG && t0 < all_lo);  // uniform for the wave
        auto sees = [&](int n, int i) {
            const int t = t0 + 32 * n + (i & 3) + 8 * (i >> 2) + 4 * h;
            return t <= t_row && (!SEG || t >= t_lo);
        };
        if (masked)
#pragma unroll
            for (int n = 0; n < NB; ++n)
#pragma unroll
                for (int i = 0; i < 16; ++i) sc[n][i] = sees(n, i) ? sc[n][i] : ATTN_NEG;
        float mloc = ATTN_NEG;
#pragma unroll
        for (int n = 0; n < NB; ++n)
#pragma unroll
            for (int i = 0; i < 16; ++i) mloc = fmaxf(mloc, sc[n][i]);
        const float top = xor32_max(mloc);  // the other half of the block's keys lives in the partner lane
        mloc = top * sl2;
        // A row's reference follows its maximum only every PA_RISE: with 32 rows to a wave some row's maximum grows in most blocks (two of three at 4096 keys), and the rescale is 64
        // products a lane.  (4096 tokens, four layers: 5623 -> 5570 us.)  bf16: the reference is set PA_RISE above the maximum -- no weight is above 1 then, and a V near the type's largest
        // keeps its sum in fp32; f16, whose V are no danger to fp32 but whose small weights have no low half, at the maximum, weights up to 2^PA_RISE.  The final division takes the factor out.
        constexpr float ABOVE = std::is_same<T, BF16>::value ? PA_RISE : 0.0f;
        if (mloc > m_run + (PA_RISE - ABOVE)) {
            const float m_new = mloc + ABOVE, alpha = attn_exp2(m_run - m_new);
            l_run *= alpha;
#pragma unroll
            for (int dt = 0; dt < DT; ++dt)
#pragma unroll
                for (int i = 0; i < 16; ++i) oacc[dt][i] *= alpha;
            m_run = m_new;
        }
        // one fma per score is exact against a maximum that is itself rounded: beyond 2^24 by more than one, which the exponential turns into 0 or infinity.  There
        // the scores are rounded like their maximum first (rare: a uniform branch; a row that sees no key of the block does not ask for it)
        float slope = sl2;
        if (__any(fabsf(m_run) > 16777216.0f && top > ATTN_NEG)) {
            slope = 1.0f;
#pragma unroll
            for (int n = 0; n < NB; ++n)
#pragma unroll
                for (int i = 0; i < 16; ++i) sc[n][i] *= sl2;
        }
        u32 phi[NB][8], plo[NB][8];
#pragma unroll
        for (int n = 0; n < NB; ++n)
#pragma unroll
            for (int i = 0; i < 16; i += 2) {
                float pa = attn_exp2(fmaf(sc[n][i], slope, -m_run)), pb = attn_exp2(fmaf(sc[n][i + 1], slope, -m_run));
                if (masked) pa = sees(n, i) ? pa : 0.0f, pb = sees(n, i + 1) ? pb : 0.0f;
                l_run += pa + pb;
                const u32 hi = pa_pack2<T>(pa, pb);
                phi[n][i >> 1] = hi;
                plo[n][i >> 1] = pa_pack2<T>(pa - lo_f32<T>(hi), pb - hi_f32<T>(hi));
            }
        // O^T += V^T . P^T : k-step s covers keys 16 s .. 16 s + 15 in the operand order 16 s + 8 (j >> 2) + 4 h + (j & 3)
#pragma unroll
        for (int s = 0; s < 2 * NB; ++s) {
            const int n = s >> 1, e = 4 * (s & 1);
            const uint4 bh = make_uint4(phi[n][e], phi[n][e + 1], phi[n][e + 2], phi[n][e + 3]);
            const uint4 bl = make_uint4(plo[n][e], plo[n][e + 1], plo[n][e + 2], plo[n][e + 3]);
            uint4 vf[DT];
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) {
                const int ch = 4 * dt + 2 * (grp & 1) + (tp >> 1);
                const v4i16_t lo4 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                    (__attribute__((address_space(3))) v4i16_t *)(v_lds + pa_off<D>(16 * s + 4 * h + tq, ch) + 8 * (tp & 1)));
                const v4i16_t hi4 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                    (__attribute__((address_space(3))) v4i16_t *)(v_lds + pa_off<D>(16 * s + 8 + 4 * h + tq, ch) + 8 * (tp & 1)));
                const uint2 a0 = __builtin_bit_cast(uint2, lo4), a1 = __builtin_bit_cast(uint2, hi4);
                vf[dt] = make_uint4(a0.x, a0.y, a1.x, a1.y);
            }
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) oacc[dt] = MfmaT<T>::run(vf[dt], bh, oacc[dt]);
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) oacc[dt] = MfmaT<T>::run(vf[dt], bl, oacc[dt]);
        }
        }
        if (b + 1 < n_blocks && (!ROT || buf)) {  // (the other image: its last readers passed the barrier in front of this block; ROT: both)
            if constexpr (ROT) {
                __syncthreads();
                rotate_in(b + 1);
            } else publish(buf ^ 1);
            __syncthreads();
        }
    }
    if (helper) return;
    if constexpr (KG == 2) {  // the second wave's sums join the first's: 16 floats of a lane at a time, lanes side by side
        static_assert(REP * 64 * (DT * 16 + 2) * 4 <= (int)sizeof(kv_lds), "the sums fit the images");
        float *meet = reinterpret_cast<float *>(kv_lds) + wave * (64 * (DT * 16 + 2)) + lane;
        __syncthreads();
        if (kg == 1) {
#pragma unroll
            for (int dt = 0; dt < DT; ++dt)
#pragma unroll
                for (int i = 0; i < 16; ++i) meet[(16 * dt + i) * 64] = oacc[dt][i];
            meet[DT * 16 * 64] = m_run, meet[(DT * 16 + 1) * 64] = l_run;
        }
        __syncthreads();
        if (kg == 1) return;
        const float m1 = meet[DT * 16 * 64], m_new = fmaxf(m_run, m1), w0 = attn_exp2(m_run - m_new), w1 = attn_exp2(m1 - m_new);
        l_run = l_run * w0 + meet[(DT * 16 + 1) * 64] * w1;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
            for (int i = 0; i < 16; ++i) oacc[dt][i] = oacc[dt][i] * w0 + meet[(16 * dt + i) * 64] * w1;
        m_run = m_new;
    }
    if constexpr (SPLIT) {
        const float l = xor32_sum(l_run);
        if (r0 + c < a.M) {
            const size_t at = ((size_t)(r0 + c) * a.Hq + hq) * a.splits + blockIdx.y;
            float *acc = a.part + at * D, *ml = a.part + (size_t)a.M * a.Hq * a.splits * D + at * 2;
#pragma unroll
            for (int dt = 0; dt < DT; ++dt)
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    *reinterpret_cast<float4 *>(acc + 32 * dt + 8 * k + 4 * h) = make_float4(oacc[dt][4 * k], oacc[dt][4 * k + 1], oacc[dt][4 * k + 2], oacc[dt][4 * k + 3]);
            if (h == 0) ml[0] = m_run, ml[1] = l;
        }
        return;
    }
    // normalise: the pair (lane, lane ^ 32) shares the query row and holds the two halves of the row sum
    const float inv = 1.0f / xor32_sum(l_run);
    if (r0 + c < a.M) {
        const int od = DR < D ? DR : SEG && a.out_d ? a.out_d : D;
        u16 *orow = a.out + ((size_t)(r0 + c) * a.Hq + hq) * od;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
            for (int k = 0; k < 4; ++k) {  // registers 4k .. 4k+3 <-> dims 32 dt + 8 k + 4 h + {0..3}
                const uint2 o = make_uint2(pack2<T>(oacc[dt][4 * k] * inv, oacc[dt][4 * k + 1] * inv),
                                           pack2<T>(oacc[dt][4 * k + 2] * inv, oacc[dt][4 * k + 3] * inv));
                if (!SEG || 32 * dt + 8 * k + 4 * h < od) *reinterpret_cast<uint2 *>(orow + 32 * dt + 8 * k + 4 * h) = o;
            }
    }
}

// The shares of a (row, head) merged in their order, one thread per four numbers: sum_z w_z acc_z / sum_z w_z l_z, w_z = exp2(m_z - max m).
template <class T, int D>
__global__ void __launch_bounds__(256) k_prefill_combine(const float *part, int splits, int pairs, u16 *out) {
    const int i = blockIdx.x * 256 + threadIdx.x, pair = i / (D / 4), d = i % (D / 4) * 4;
    if (pair >= pairs) return;
    const float *acc = part + (size_t)pair * splits * D + d, *ml = part + (size_t)pairs * splits * D + (size_t)pair * splits * 2;
    float m = ATTN_NEG, l = 0.0f;
    for (int z = 0; z < splits; ++z) m = fmaxf(m, ml[2 * z]);
    float4 o = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
#pragma unroll 4
    for (int z = 0; z < splits; ++z) {
        const float w = attn_exp2(ml[2 * z] - m), lz = ml[2 * z + 1];
        if (lz == 0.0f) continue;  // nothing seen: its sums were never written
        const float4 v = *reinterpret_cast<const float4 *>(acc + (size_t)z * D);
        l = fmaf(w, lz, l), o.x = fmaf(w, v.x, o.x), o.y = fmaf(w, v.y, o.y), o.z = fmaf(w, v.z, o.z), o.w = fmaf(w, v.w, o.w);
    }
    const float inv = 1.0f / l;
    *reinterpret_cast<uint2 *>(out + (size_t)pair * D + d) = make_uint2(pack2<T>(o.x * inv, o.y * inv), pack2<T>(o.z * inv, o.w * inv));
}

// Workgroups along the keys: rows behind a long cached prefix are few tiles with many blocks each (37 rows: 16 workgroups of 30 blocks).  `before`: keys in front of the first row.  Every
// share costs its sums (4 D bytes per row and head, twice): at least two blocks of 64 keys per share up to 64 rows, three beyond, up to two workgroups per CU.  us, 1 / 2 / 4 / 8 shares:
// 8 rows behind 500: 20 / 14 / 12 / 12; 37 behind 900: 35 / 24 / 18 / 17; 100: 38 / 26 / 21 / 23; 200: 41 / 30 / 26 / 30; 509: 53 / 42 / 40 / 46; 32 behind 4000: 131 / 73 / 42 / 29 (16: 28).
// Rows of a fresh prompt see half of the blocks on average and gain nothing (509 rows: 22 / 26).
// More than 256 rows of two to four heads a group may take two waves per tile instead (KG), one workgroup a CU (their images fill it for heads of 128), and so half as many shares where the chip and not the
// prefix sets their number.  Two heads a group and heads of 64 gain from it unless one share is left of three.  The others want as many shares, four, a full round of workgroups or, behind no more keys than rows come, most of one.  Prompts of four layers of
// attention alone, us, shares of one wave / of two, heads of 128: 32 / 8 heads, 509 rows behind 900 four / two 300 / 291, 400 behind 2000 four / two 328 / 332, 600 three / one 368 / 398; 24 / 8, 600 behind
// 4000 473 / 581; 12 / 4, 400 behind 2000 nine / four 291 / 276, 1250 behind 4000 three / one 508 / 639; 16 / 8, 1000 behind 2000 two / one 459 / 412; heads of 64, 32 / 8, 600 behind 2000 294 / 310.
static inline bool prefill_attn_duo(int rep) { return rep >= 2 && rep <= 4; }  // (four waves of 64 keys, 240 registers each, leave room for four more)
static inline bool prefill_attn_slim(int rep, int D) { return rep == 2 || D == 64; }
static inline int prefill_attn_shares(int M, int before, int Hkv, int chip) {  // chip: workgroups that run at once
    const int shares = before / 64 / (M <= 64 ? 2 : 3), room = chip / ((M + 31) / 32 * Hkv);
    const int s = shares < room ? shares : room;
    return s < 2 ? 1 : s > 16 ? 16 : s;
}
static inline bool prefill_attn_duo_shares(int M, int before, int Hq, int Hkv, int D) {  // whether shares are (or one is) of two waves per tile
    const int one = prefill_attn_shares(M, before, Hkv, 512), two = prefill_attn_shares(M, before, Hkv, 256), workgroups = (M + 31) / 32 * Hkv * two;
    if (M <= 256 || one < 2 || !prefill_attn_duo(Hq / Hkv)) return false;
    return prefill_attn_slim(Hq / Hkv, D) ? 8 * two >= 3 * one : 2 * two > one || two >= 4 || workgroups >= 240 || (two == 1 && workgroups >= 200 && before <= M);
}
static inline int prefill_attn_splits(int M, int before, int Hq, int Hkv, int D) { return prefill_attn_shares(M, before, Hkv, prefill_attn_duo_shares(M, before, Hq, Hkv, D) ? 256 : 512); }
// room for the sums of any split prompt: ceil(M / 32) Hkv splits <= 512
static inline size_t prefill_attn_part_bytes(int Hq, int Hkv, int D) { return (size_t)(512 / Hkv) * 32 * Hq * (D + 2) * sizeof(float); }

// A block of 64 keys costs its whole chain however few of them there are.  us in blocks of 32 / 64 keys, 32 / 8 heads of 128: 8 rows 5.7 / 6.7, 20 rows 6.5 / 7.6, 33 rows 7.4 / 8.4,
// 48 rows 7.6 / 8.4, 64 rows 8.8 / 8.4; 32 / 4 heads: 8 rows 6.4 / 7.6, 33 rows 9.6 / 10.6, 64 rows 10.7 / 10.5.
static inline bool prefill_attn_short(const PrefillAttnArgs &a) { return a.M + a.before <= 56; }

// Two waves per tile (KG) pay from about five blocks of 64 keys on, where they save blocks that wait for each other; below, and in shares of a few blocks, their meeting costs more.  us, one wave /
// two, 32 / 8 heads: 128 rows 9.1 / 9.8, 300 15.4 / 15.1, 509 21.9 / 19.0, 1000 39.5 / 32.3, 1900 76.9 / 66.7; 24 / 8: 509 24.9 / 19.3, 1000 49.5 / 33.4, 1900 92.9 / 62.6; 32 / 16: 300 15.3 / 13.0;
// 37 behind 900 in seven shares 17.2 / 17.9.  Beyond one round of workgroups not behind many more cached keys than rows come, where all tiles are long and a last round costs as much as a full one (four
// layers of attention alone, heads of 128, one wave / two: 32 / 8 heads, 1500 rows behind 900 532 / 508, behind 4000 884 / 920; 24 / 8, 1500 behind 2000 747 / 695, 2000 behind 4000 1085 / 1107); 16 / 8
// and heads of 64 gain there too (16 / 8, 1500 behind 4000 971 / 819).  Against two tiles per workgroup, where those fill the chip: two waves per SIMD either way, K and V staged once for both: fresh
// prompts (2000 rows 89.5 / 71.3, 2300 103 / 94, 3000 139 / 148; layers as above, 24 / 8 heads, 2050 551 / 536, 2400 574 / 591), behind cached keys hardly but heads of 64 (32 / 8
// heads of 128, 2050 behind 400 609 / 588, behind 900 696 / 718; 24 / 8, 2300 behind 400 627 / 678; 16 / 8 565 / 601; 32 / 8 heads of 64 520 / 491, behind 4000 1067 / 994).
static inline bool prefill_attn_pairs(const PrefillAttnArgs &a, int D) {
    const int rep = a.Hq / a.Hkv, tiles = (a.M + 31) / 32 * a.Hkv, doubles = (a.M + 63) / 64 * a.Hkv;
    if (a.splits > 1) return prefill_attn_duo_shares(a.M, a.before, a.Hq, a.Hkv, D);
    if (!prefill_attn_duo(rep) || a.M + a.before < 256 || doubles >= 320) return false;
    if (doubles >= 256) return D == 64 || (rep == 4 ? a.before <= (doubles < 288 ? a.M / 4 : 0) : a.before == 0 && doubles < 288);
    return prefill_attn_slim(rep, D) || tiles <= 256 || a.before <= (rep == 3 ? a.M + a.M / 2 : a.M);
}

template <class T, int D>
static int prefill_attn_launch_d(const PrefillAttnArgs &a, hipStream_t st) {
    const int rep = a.Hq / a.Hkv;
    const bool pairs = prefill_attn_pairs(a, D);
    if (a.splits > 1) {
        const dim3 grid((a.M + 31) / 32 * a.Hkv, a.splits);
#define PA_SPLIT(R)                                                                                                                                      \
    if (pairs && R >= 2 && R <= 4) hipLaunchKernelGGL((k_prefill_attn<T, D, R, 1, false, true, false, (R >= 2 && R <= 4 ? 2 : 1)>), grid, dim3(R * 128), 0, st, a); \
    else hipLaunchKernelGGL((k_prefill_attn<T, D, R, 1, false, true>), grid, dim3(R * 64), 0, st, a);                                                    \
    break
        switch (rep) {
            case 1: PA_SPLIT(1);
            case 2: PA_SPLIT(2);
            case 3: PA_SPLIT(3);
            case 4: PA_SPLIT(4);
            case 5: PA_SPLIT(5);
            case 6: PA_SPLIT(6);
            case 7: PA_SPLIT(7);
            case 8: PA_SPLIT(8);
            default: return pie::fail(PIE_E_SHAPE, "prefill attention: n_heads / n_kv_heads must be between 1 and 8");
        }
#undef PA_SPLIT
        PIE_LAUNCH_CHECK();
        const int rows = a.M * a.Hq;
        hipLaunchKernelGGL((k_prefill_combine<T, D>), dim3((unsigned)(((size_t)rows * (D / 4) + 255) / 256)), dim3(256), 0, st, a.part, a.splits, rows, a.out);
        PIE_LAUNCH_CHECK();
        return PIE_OK;
    }
    const int qt = pie_knob(PIE_KNOB_PREFILL_QT);  // test knob: 1 forces one 32-row query tile per workgroup, 2 forces two wherever they fit
    // 2 tiles need 2*rep <= 8 waves of up to 256 registers, and only pay while the halved grid still fills the 256 CUs
    // (8B model: 4096 tokens 54.9 -> 53.9 ms, 8000 tokens 126.3 -> 125.0 ms; at 1024 tokens it would idle half the chip)
    const bool two = rep <= 4 && a.M > 32 && (qt > 0 ? qt == 2 : ((a.M + 63) / 64) * a.Hkv >= 256 && !pairs), few = prefill_attn_short(a);
    const dim3 grid(((a.M + (two ? 63 : 31)) / (two ? 64 : 32)) * a.Hkv);
#define PA_LAUNCH(R)                                                                                         \
    if (two && R <= 4) hipLaunchKernelGGL((k_prefill_attn<T, D, R, (R <= 4 ? 2 : 1)>), grid, dim3(R * 128), 0, st, a); \
    else if (pairs && !few && R >= 2 && R <= 4) hipLaunchKernelGGL((k_prefill_attn<T, D, R, 1, false, false, false, (R >= 2 && R <= 4 ? 2 : 1)>), grid, dim3(R * 128), 0, st, a); \
    else if (few && R >= 4) hipLaunchKernelGGL((k_prefill_attn<T, D, R, 1, false, false, (R >= 4)>), grid, dim3(R * 64), 0, st, a); \
    else hipLaunchKernelGGL((k_prefill_attn<T, D, R, 1>), grid, dim3(R * 64), 0, st, a);                     \
    break
    switch (rep) {
        case 1: PA_LAUNCH(1);
        case 2: PA_LAUNCH(2);
        case 3: PA_LAUNCH(3);
        case 4: PA_LAUNCH(4);
        case 5: PA_LAUNCH(5);
        case 6: PA_LAUNCH(6);
        case 7: PA_LAUNCH(7);
        case 8: PA_LAUNCH(8);
        default: return pie::fail(PIE_E_SHAPE, "prefill attention: n_heads / n_kv_heads must be between 1 and 8");
    }
#undef PA_LAUNCH
    PIE_LAUNCH_CHECK();
    return PIE_OK;
}
// block-diagonal attention (SEG): multi-head only (Hq == Hkv, the vision tower), two query tiles per workgroup while the
// halved grid still fills the chip
template <class T, int D, int DR = D>
static int segment_attn_launch_d(const PrefillAttnArgs &a, hipStream_t st) {
    if (a.Hq != a.Hkv) return pie::fail(PIE_E_SHAPE, "segment attention: n_heads must equal n_kv_heads");
    const bool two = a.M > 32 && ((a.M + 63) / 64) * a.Hkv >= 512;
    const dim3 grid(((a.M + (two ? 63 : 31)) / (two ? 64 : 32)) * a.Hkv);
    if (two) hipLaunchKernelGGL((k_prefill_attn<T, D, 1, 2, true, false, false, 1, DR>), grid, dim3(128), 0, st, a);
    else hipLaunchKernelGGL((k_prefill_attn<T, D, 1, 1, true, false, false, 1, DR>), grid, dim3(64), 0, st, a);
    PIE_LAUNCH_CHECK();
    return PIE_OK;
}
// Windows of the vision tower whose q, k and v are still the Linear's rows (ROT): the bias and the rotation on the way into LDS, keys once per 64 query rows.
template <class T>
static int segment_rot_launch_t(const PrefillAttnArgs &a, int D, hipStream_t st) {
    const dim3 grid((a.M + 63) / 64 * a.Hkv);
    if (D == 80) hipLaunchKernelGGL((k_prefill_attn<T, 128, 1, 2, true, false, false, 1, 80, true>), grid, dim3(256), 0, st, a);
    else hipLaunchKernelGGL((k_prefill_attn<T, 64, 1, 2, true, false, false, 1, 64, true>), grid, dim3(256), 0, st, a);
    PIE_LAUNCH_CHECK();
    return PIE_OK;
}
// the same with grouped-query heads (several prompts prefilled in one pass: causal inside each prompt = seg_hi[r] = r + 1)
template <class T, int D>
static int segment_attn_gqa_launch_d(const PrefillAttnArgs &a, hipStream_t st) {
    const int rep = a.Hq / a.Hkv;
    const dim3 grid(((a.M + 31) / 32) * a.Hkv);
#define PA_SEG(R) hipLaunchKernelGGL((k_prefill_attn<T, D, R, 1, true>), grid, dim3(R * 64), 0, st, a); break
    switch (rep) {
        case 1: PA_SEG(1);
        case 2: PA_SEG(2);
        case 3: PA_SEG(3);
        case 4: PA_SEG(4);
        case 5: PA_SEG(5);
        case 6: PA_SEG(6);
        case 7: PA_SEG(7);
        case 8: PA_SEG(8);
        default: return pie::fail(PIE_E_SHAPE, "segment attention: n_heads / n_kv_heads must be between 1 and 8");
    }
#undef PA_SEG
    PIE_LAUNCH_CHECK();
    return PIE_OK;
}
template <class T>
static int segment_attn_gqa_launch_t(const PrefillAttnArgs &a, int D, hipStream_t st) {
    return D == 128 ? segment_attn_gqa_launch_d<T, 128>(a, st) : segment_attn_gqa_launch_d<T, 64>(a, st);
}

template <class T>
static int segment_attn_launch_t(const PrefillAttnArgs &a, int D, hipStream_t st) {
    if (D == 80) return segment_attn_launch_d<T, 128, 80>(a, st);
    return D == 128 ? segment_attn_launch_d<T, 128>(a, st) : segment_attn_launch_d<T, 64>(a, st);
}

template <class T>
static int prefill_attn_launch_t(const PrefillAttnArgs &a, int D, hipStream_t st) {
    return D == 128 ? prefill_attn_launch_d<T, 128>(a, st) : prefill_attn_launch_d<T, 64>(a, st);
}
