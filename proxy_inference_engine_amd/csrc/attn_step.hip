// attn_step.hip -- decode attention with its scores on the matrix units: a batch's step over T pages (RoPE, append and scores in one launch), and one sequence's step.
//
// Replaces mx.fast.scaled_dot_product_attention at models/base.py:111-113 for L = 1.
//
// attention.hpp's body scores on the vector units: a token's products per head, three or four DPP additions, a running maximum per 16 lanes whose rescale is taken by some lane of nearly
// every block; 211 vector instructions per four tokens and group of four heads of 128 (SQ_INSTS_VALU), 21 of the 33 us of 32 rows at 1000 cached positions, which are 20 us of stream.
// Here a wave takes 16 tokens at a time:
//   * scores S[token][head] = K q^T by v_mfma_f32_16x16x32, K rows straight from memory in operand order (lane: token lane % 16, dims 32 s + 8 (lane / 16) ..), the query heads as
//     the 16 columns (four or eight, repeated): no cross-lane additions, and a lane is left with four tokens' scores of ONE head, lane % 4 or lane % 8;
//   * the softmax of 16 tokens x 4 heads is then four exponentials a lane, not sixteen; a stream is rescaled only where a score exceeds its reference, which is set RISE above it (weights
//     of 2^-RISE and less lose nothing in fp32, none is above 1, so that a V near the type's largest has room in the sums, and the merge divides the factor out);
//   * P V stays fp32 products of the vector units, weights unrounded: lane (tokens 4 (lane / 16) .., dims 8 (lane % 16) ..; heads of 64: half of the tokens) finds its tokens' weights
//     in its own quad or the one beside (DPP).
// Blocks of 16 tokens begin at multiples of 16 (a page holds 64): a block lies in one page, its page number and its addresses are the wave's.
// With the scores that cheap, fewer and longer workgroups stream as fast: of four waves (eight measured the same), about one per CU (step_split).  Where a batch's row is in pieces the last
// to arrive merges them.  Four layers, sixteen steps, us, vector units -> this.  Llama-3-8B int4: 32 rows at 1000 positions 7596 -> 6350 (in two pieces each 6518, in four 6903), 8 rows at
// 200 5253 -> 4826; bf16, 8 rows at 1000 8460 -> 7900 (with a combine launch 8080); int4, one row of 8000 positions among 31 of 100 10622 -> 7111, 32 rows of 2000 8950 -> 7396.
// Llama-3.2-3B (three heads a group) int4: 24 rows at 700 6255 -> 5274, one at 600 2317 -> 2267, at 128 level.  TinyLlama-1.1B (eight heads of 64): 32 rows at 1000 6871 -> 5151, 8 at 300
// 4301 -> 3899, one at 128 2745 -> 2558, at 900 2950 -> 2643.
#include "attention.hpp"

namespace {

constexpr float RISE = 8.0f;  // log2: see above
constexpr int STEP_DEPTH = 2, STEP_WAVES = 4, MERGE = 4;  // (MERGE: splits' sums in flight)  Waves: 152 registers: three waves a SIMD, 24 KB of rows in flight on each

typedef float f32x4 __attribute__((ext_vector_type(4)));
template <class T>
__device__ __forceinline__ f32x4 mfma16(const uint4 &a, const uint4 &b, const f32x4 &c) {
    if constexpr (std::is_same<T, F16>::value) {
        typedef _Float16 v8 __attribute__((ext_vector_type(8)));
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8, a), __builtin_bit_cast(v8, b), c, 0, 0, 0);
    } else {
        typedef __bf16 v8 __attribute__((ext_vector_type(8)));
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8, a), __builtin_bit_cast(v8, b), c, 0, 0, 0);
    }
}
// lane h of every quad, to the quad
template <int h>
__device__ __forceinline__ float of_quad(float x) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), h * 0x55, 0xF, 0xF, true));
}
// With more than four heads a row's quads hold heads 0-3, 4-7, 0-3, 4-7: what the quad beside holds
template <int REP>
__device__ __forceinline__ float beside(float x) {
    if constexpr (REP <= 4) return x;
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x124, 0xF, 0xF, true));  // row_ror:4
}
// x: of head lane % 4, or of lane % 8 with more than four heads, other: beside(x) -> o[h]: head h's
template <int REP>
__device__ __forceinline__ void heads_of(float x, float other, float (&o)[REP]) {
    float lo = x, hi = 0.0f;
    if constexpr (REP > 4) {
        const bool upper = threadIdx.x & 4;
        lo = upper ? other : x, hi = upper ? x : other;
    }
    o[0] = of_quad<0>(lo);
    if constexpr (REP > 1) o[1] = of_quad<1>(lo);
    if constexpr (REP > 2) o[2] = of_quad<2>(lo);
    if constexpr (REP > 3) o[3] = of_quad<3>(lo);
    if constexpr (REP > 4) o[4] = of_quad<0>(hi);
    if constexpr (REP > 5) o[5] = of_quad<1>(hi);
    if constexpr (REP > 6) o[6] = of_quad<2>(hi);
    if constexpr (REP > 7) o[7] = of_quad<3>(hi);
}

// two floats, past the caches that the chip's XCDs do not share
__device__ __forceinline__ void agent_store(float *p, float x, float y) {
    __hip_atomic_store(reinterpret_cast<unsigned long long *>(p), __builtin_bit_cast(unsigned long long, make_float2(x, y)), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ float2 agent_load(const float *p) {
    return __builtin_bit_cast(float2, __hip_atomic_load(reinterpret_cast<const unsigned long long *>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
}

// How a row's positions are cut: into pieces of about what a CU gets of the batch's, one at least and most at most, that begin at multiples of 16.  The lengths are on the device, and
// so is the choice: rows of like lengths are one piece each where there are CUs for no more, a long row among short ones is spread.  (The lengths are summed once a step.)
__device__ __forceinline__ AttnSplit step_split(int T, int total, int Hkv, int most) {
    const int per_cu = (int)(((long long)total * Hkv) >> 8), share = max(per_cu, STEP_WAVES * 16);  // (256 CUs)
    const int n = max(1, min(most, (T + (share >> 1)) / share));
    AttnSplit s;
    s.chunk = max(((T + n - 1) / n + 15) & ~15, 16);
    s.active = T > 0 ? (T + s.chunk - 1) / s.chunk : 0;
    return s;
}

// STEP: the batch's step.  Else one sequence's, in buffers of its own or PAGED: q and the new row are in memory, the consumer merges the splits (attn_split's, beginning at multiples of 16; the
// neutral partial of one that is not active).
template <class T, int D, int REP, bool NTKV, bool STEP, bool PAGED>
__global__ void __launch_bounds__(STEP_WAVES * 64, REP <= 4 ? 3 : 2) k_attn_step(const AttnRopeArgs a) {
    constexpr int half = D / 2, HC = REP <= 4 ? 4 : 8;     // head of a lane: lane % HC
    constexpr int KS = D / 32, VL = D / 8, SUB = 16 / VL, VI = 4 / SUB;  // K pieces of a lane; lanes of a V row, rows of 16 lanes, V pieces of a lane
    constexpr int WAVES = STEP_WAVES, NT = WAVES * 64, NSTR = WAVES * 4;
    __shared__ __attribute__((aligned(16))) u16 s_q[REP * D], s_kv[2 * D];
    __shared__ float s_m[REP][NSTR], s_l[REP][NSTR];
    __shared__ __attribute__((aligned(16))) float s_acc[REP][NSTR][D];
    // The pieces that every row has are dealt to the CUs first, behind them those that few have -- a row's next one place on, or where the others leave at once they would all come to one CU.
    const int g = blockIdx.x, split = blockIdx.z, row = (blockIdx.y + split) % gridDim.y, q0 = g * REP;
    const int Ttot = STEP ? a.ctx_len[row] : a.state ? a.state->pos + 1 : a.T;
    AttnSplit sp;
    if constexpr (STEP) sp = step_split(Ttot, *a.total, a.Hkv, a.splits);
    else {
        sp = attn_split(Ttot, a.splits);
        sp.chunk = (sp.chunk + 15) & ~15, sp.active = (Ttot + sp.chunk - 1) / sp.chunk;
    }
    if (split >= sp.active) {  // uniform
        if (STEP && split == 0)  // an idle slot: zeros
            for (int o = threadIdx.x; o < REP * D; o += NT) a.out[((size_t)row * a.Hq + q0) * D + o] = 0;
        if (!STEP)
            for (int o = threadIdx.x; o < REP * half; o += NT) {
                const int h = o / half, d = (o % half) * 2;
                const size_t at = (size_t)(q0 + h) * a.splits + split;
                *reinterpret_cast<float2 *>(a.part_acc + at * D + d) = make_float2(0.0f, 0.0f);
                if (d == 0) *reinterpret_cast<float2 *>(a.part_ml + at * 2) = make_float2(ATTN_NEG, 0.0f);
            }
        return;
    }
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lo = lane & 15, hi = lane >> 4, vt = hi * 4 + lo / VL, vd = (lo % VL) * 8;  // (vt + SUB i: token of its V piece i)
    const int pos = Ttot - 1, t_begin = split * sp.chunk, t_end = min(Ttot, t_begin + sp.chunk);
    const bool newest = STEP && split == sp.active - 1;  // this split ends with the position that this launch writes
    const int *bt = PAGED ? a.block_table + (size_t)row * a.bt_stride : nullptr;
    const unsigned last_page = (unsigned)a.n_pages - 1u;
    const size_t page_elems = (size_t)2 * 64 * a.Hkv * D;
    const int cap = PAGED ? 64 : a.state ? a.state->cap : a.cap;
    const u16 *kbase = (STEP ? a.slab : a.k ? a.k : reinterpret_cast<const u16 *>(a.kv_table[a.layer])) + (size_t)g * cap * D;
    const u16 *vbase = STEP ? kbase + (size_t)a.Hkv * 64 * D : (a.k ? a.v : reinterpret_cast<const u16 *>(a.kv_table[a.n_layers + a.layer])) + (size_t)g * cap * D;

    const int first = t_begin + wave * 16;  // the wave's block b begins at first + 16 WAVES b
    const int n_blk = first < t_end ? (t_end - first + 16 * WAVES - 1) / (16 * WAVES) : 0;
    int pages = 0;  // lane i: page of block i, of the 64 that b is in; past the wave's last block that one's, whose row issue() reads again (t_end may lie a page further on)
    auto page_ids = [&](int b0) {
        const int t = first + min(b0 + lane, n_blk - 1) * 16 * WAVES;
        pages = (int)min((unsigned)bt[t >> 6], last_page);
    };
    uint4 kq[STEP_DEPTH][KS], vq[STEP_DEPTH][VI];
    const int t_mem = newest ? pos : t_end;  // rows before it are in memory
    auto issue = [&](int d, int b) {
        const int last = min(b, n_blk - 1), t0 = first + last * 16 * WAVES;
        // Rows beyond lim are not read, not even with weight 0.  (A block of the new row alone: its place, replaced below; past the last block: one row again.)
        const int lim = b == last ? max(t_mem - 1 - t0, 0) : 0;
        size_t at = (size_t)t0 * D;
        if constexpr (PAGED) {
            if (b && !(b & 63)) page_ids(b);
            at = (size_t)__builtin_amdgcn_readlane(pages, b & 63) * page_elems + (size_t)(t0 & 63) * D;
        }
        const u16 *kp = kbase + at, *vp = vbase + at;
        const int ko = min(lo, lim) * D + hi * 8;
#pragma unroll
        for (int s = 0; s < KS; ++s) kq[d][s] = attn_load_row<NTKV>(kp + ko + 32 * s);
#pragma unroll
        for (int i = 0; i < VI; ++i) vq[d][i] = attn_load_row<NTKV>(vp + min(vt + SUB * i, lim) * D + vd);
    };
    if (n_blk) {
        if constexpr (PAGED) page_ids(0);
#pragma unroll
        for (int d = 0; d < STEP_DEPTH; ++d) issue(d, d);
    }
    if constexpr (STEP) {  // RoPE of the group's query heads, by every split; of k and the append, by the newest: k_rope_append_rows, term for term
        const unsigned pg = min((unsigned)bt[pos >> 6], last_page);
        u16 *kdst = a.pages + (size_t)pg * page_elems + ((size_t)g * 64 + (pos & 63)) * D, *vdst = kdst + (size_t)a.Hkv * 64 * D;
        for (int p = threadIdx.x; p < (newest ? REP + 2 : REP) * half; p += NT) {
            const int h = p / half, ii = p % half;  // h: REP q heads, k, v
            const size_t at = (size_t)row * a.n_cols + (h < REP ? q0 + h : a.Hq + (h == REP ? g : a.Hkv + g)) * D + 2 * ii;
            const float2 cs = *reinterpret_cast<const float2 *>(a.rope_cs + ((size_t)row * half + ii) * 2);
            u32 pr;
            if (a.S > 1) {
                const size_t i[1] = {at};
                float2 v[1];
                slab_sum<float2, 1>(a.part, a.S, a.MN, i, v);
                pr = pack2<T>(v[0].x, v[0].y);
            } else pr = *reinterpret_cast<const u32 *>(a.qkv + at);
            if (h == REP + 1) {
                *reinterpret_cast<u32 *>(vdst + 2 * ii) = pr, *reinterpret_cast<u32 *>(s_kv + D + 2 * ii) = pr;
                continue;
            }
            const float ra = lo_f32<T>(pr), rb = hi_f32<T>(pr);
            const int i0 = a.traditional ? 2 * ii : ii, i1 = a.traditional ? 2 * ii + 1 : ii + half;
            const u16 o0 = T::from_f32(__fsub_rn(__fmul_rn(ra, cs.x), __fmul_rn(rb, cs.y))), o1 = T::from_f32(__fadd_rn(__fmul_rn(ra, cs.y), __fmul_rn(rb, cs.x)));
            u16 *dst = h < REP ? s_q + h * D : s_kv;
            dst[i0] = o0, dst[i1] = o1;
            if (h == REP) kdst[i0] = o0, kdst[i1] = o1;
        }
        __syncthreads();
    }
    uint4 qv[KS];
    const int qh = min(lane & (HC - 1), REP - 1);
#pragma unroll
    for (int s = 0; s < KS; ++s) qv[s] = *reinterpret_cast<const uint4 *>((STEP ? s_q + qh * D : a.q + (size_t)(q0 + qh) * D) + 32 * s + hi * 8);
    const float sl2 = a.scale * ATTN_LOG2E;
    float m = ATTN_NEG, l = 0.0f, acc[REP][8];
#pragma unroll
    for (int h = 0; h < REP; ++h)
#pragma unroll
        for (int j = 0; j < 8; ++j) acc[h][j] = 0.0f;

    auto score = [&](int d, int b, auto whole) {  // whole: of a block in front of the wave's last, whose tokens are all in memory and all count
        constexpr bool WHOLE = decltype(whole)::value;
        const int t0 = first + b * 16 * WAVES;
        if (!WHOLE && newest && t0 + 16 > pos) {  // the new row, and the rows past it of its block (weight 0, but 0 times what nobody wrote may be NaN)
            if (lo >= pos - t0)
#pragma unroll
                for (int s = 0; s < KS; ++s) kq[d][s] = *reinterpret_cast<const uint4 *>(s_kv + 32 * s + hi * 8);
#pragma unroll
            for (int i = 0; i < VI; ++i)
                if (vt + SUB * i >= pos - t0) vq[d][i] = *reinterpret_cast<const uint4 *>(s_kv + D + vd);
        }
        f32x4 s4 = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int s = 0; s < KS; ++s) s4 = mfma16<T>(kq[d][s], qv[s], s4);
        float sc[4], most = ATTN_NEG, p[4];
        bool in[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            in[i] = WHOLE || hi * 4 + i < t_end - t0;
            sc[i] = in[i] ? s4[i] * sl2 : ATTN_NEG;
            most = fmaxf(most, sc[i]);
        }
        const bool rise = most > m;
        if (__any(rise)) {  // (the whole wave: a quad's lanes hold its heads' factors)
            const float to = rise ? most + RISE : m, f = attn_exp2(m - to);
            float fh[REP];
            heads_of<REP>(f, beside<REP>(f), fh);
            l *= f, m = to;
#pragma unroll
            for (int h = 0; h < REP; ++h)
#pragma unroll
                for (int j = 0; j < 8; ++j) acc[h][j] *= fh[h];
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) p[i] = in[i] ? attn_exp2(sc[i] - m) : 0.0f, l += p[i];
#pragma unroll
        for (int i = 0; i < VI; ++i) {
            const u32 w[4] = {vq[d][i].x, vq[d][i].y, vq[d][i].z, vq[d][i].w};
            float ph[REP];
            if constexpr (SUB == 1) heads_of<REP>(p[i], beside<REP>(p[i]), ph);
            else {  // (the quad beside may be of the other half, which weighs the other token)
                const float even = p[2 * i & 3], odd = p[(2 * i + 1) & 3], even_b = beside<REP>(even), odd_b = beside<REP>(odd);
                heads_of<REP>(lo < VL ? even : odd, lo < VL ? even_b : odd_b, ph);
            }
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float v0 = lo_f32<T>(w[j]), v1 = hi_f32<T>(w[j]);
#pragma unroll
                for (int h = 0; h < REP; ++h) acc[h][2 * j] = fmaf(ph[h], v0, acc[h][2 * j]), acc[h][2 * j + 1] = fmaf(ph[h], v1, acc[h][2 * j + 1]);
            }
        }
    };
    // Between loads in flight and their use stands no branch around a load: behind one the compiler would wait for every load there is.  Behind the loop, the last two blocks, or
    // one of an odd number, load nothing, and only they can hold the new row or tokens past the end; of an odd number the loop's last round asks for a row of the last block again (one loop for all, with loads past the end: 168 registers instead of 152; sixteen steps of four layers, one f16 row of TinyLlama's 2561 / 2532 us, 8 int4 rows of
    // Llama-3-8B's at 200 positions 4040 / 3970, 32 at 1000 6262 / 6231).
    int b0 = 0;
    for (; b0 + STEP_DEPTH < n_blk; b0 += STEP_DEPTH)
#pragma unroll
        for (int d = 0; d < STEP_DEPTH; ++d) score(d, b0 + d, std::true_type{}), issue(d, b0 + d + STEP_DEPTH);
#pragma unroll
    for (int d = 0; d < STEP_DEPTH; ++d)
        if (b0 + d < n_blk) score(d, b0 + d, std::false_type{});

    // streams: 16 lanes of a wave share one
    const int str = wave * 4 + hi;
    if (lo < REP) s_m[lo][str] = m, s_l[lo][str] = l;
    if constexpr (SUB == 2)
#pragma unroll
        for (int h = 0; h < REP; ++h)
#pragma unroll
            for (int j = 0; j < 8; ++j) acc[h][j] += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, acc[h][j]), 0x128, 0xF, 0xF, true));  // row_ror:8
    if (lo < VL)
#pragma unroll
        for (int h = 0; h < REP; ++h) {
            *reinterpret_cast<float4 *>(&s_acc[h][str][vd]) = make_float4(acc[h][0], acc[h][1], acc[h][2], acc[h][3]);
            *reinterpret_cast<float4 *>(&s_acc[h][str][vd + 4]) = make_float4(acc[h][4], acc[h][5], acc[h][6], acc[h][7]);
        }
    __syncthreads();
    for (int o = threadIdx.x; o < REP * half; o += NT) {
        const int h = o / half, d = (o % half) * 2;
        float M = ATTN_NEG;
#pragma unroll
        for (int i = 0; i < NSTR; ++i) M = fmaxf(M, s_m[h][i]);
        float L = 0.0f, A0 = 0.0f, A1 = 0.0f;
#pragma unroll
        for (int i = 0; i < NSTR; ++i) {
            const float w = attn_exp2(s_m[h][i] - M);
            const float2 av = *reinterpret_cast<const float2 *>(&s_acc[h][i][d]);
            L = fmaf(w, s_l[h][i], L), A0 = fmaf(w, av.x, A0), A1 = fmaf(w, av.y, A1);
        }
        const size_t hq = (size_t)row * a.Hq + q0 + h;
        if constexpr (!STEP) {
            *reinterpret_cast<float2 *>(a.part_acc + (hq * a.splits + split) * D + d) = make_float2(A0, A1);
            if (d == 0) *reinterpret_cast<float2 *>(a.part_ml + (hq * a.splits + split) * 2) = make_float2(M, L);
            continue;
        }
        if (sp.active == 1) {
            *reinterpret_cast<u32 *>(a.out + hq * D + d) = pack2<T>(A0 / L, A1 / L);
            continue;
        }
        agent_store(a.part_acc + (hq * a.splits + split) * D + d, A0, A1);
        if (d == 0) agent_store(a.part_ml + (hq * a.splits + split) * 2, M, L);
    }
    if (!STEP || sp.active == 1) return;
    // The last of the row's splits to arrive merges them.  Their sums go past the caches of an XCD (agent scope), and have arrived there when their workgroup says so.
    __shared__ int s_last;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    int *arrived = a.arrived + row * a.Hkv + g;
    if (threadIdx.x == 0) s_last = __hip_atomic_fetch_add(arrived, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == sp.active - 1;
    __syncthreads();
    if (!s_last) return;
    if (threadIdx.x == 0) __hip_atomic_store(arrived, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    for (int o = threadIdx.x; o < REP * half; o += NT) {
        const int h = o / half, d = (o % half) * 2;
        const size_t hq = (size_t)row * a.Hq + q0 + h;
        const float *acc_of = a.part_acc + hq * a.splits * D + d, *ml_of = a.part_ml + hq * a.splits * 2;
        float M = ATTN_NEG, L = 0.0f, A0 = 0.0f, A1 = 0.0f;
        for (int j0 = 0; j0 < sp.active; j0 += MERGE) {
            float2 ml[MERGE], av[MERGE];
#pragma unroll
            for (int u = 0; u < MERGE; ++u) {
                const int j = min(j0 + u, sp.active - 1);
                ml[u] = agent_load(ml_of + 2 * j), av[u] = agent_load(acc_of + (size_t)j * D);
            }
            float to = M;
#pragma unroll
            for (int u = 0; u < MERGE; ++u) to = fmaxf(to, ml[u].x);
            const float f = attn_exp2(M - to);
            L *= f, A0 *= f, A1 *= f, M = to;
#pragma unroll
            for (int u = 0; u < MERGE; ++u) {
                const float w = j0 + u < sp.active ? attn_exp2(ml[u].x - M) : 0.0f;
                L = fmaf(w, ml[u].y, L), A0 = fmaf(w, av[u].x, A0), A1 = fmaf(w, av[u].y, A1);
            }
        }
        *reinterpret_cast<u32 *>(a.out + hq * D + d) = pack2<T>(A0 / L, A1 / L);
    }
}

template <class T, int D, bool NTKV, bool STEP, bool PAGED>
int step_go(int rep, const AttnRopeArgs &a, hipStream_t st) {
    const dim3 grid(a.Hkv, STEP ? a.rows : 1, a.splits), block(STEP_WAVES * 64);
#define STEP_GO(R) \
    case R: hipLaunchKernelGGL((k_attn_step<T, D, R, NTKV, STEP, PAGED>), grid, block, 0, st, a); break
    switch (rep) {
        STEP_GO(1);
        STEP_GO(2);
        STEP_GO(3);
        STEP_GO(4);
        STEP_GO(5);
        STEP_GO(6);
        STEP_GO(7);
        STEP_GO(8);
        default: return pie::fail(PIE_E_SHAPE, "sdpa_decode: n_heads / n_kv_heads must be between 1 and 8");
    }
#undef STEP_GO
    PIE_LAUNCH_CHECK();
    return PIE_OK;
}

}  // namespace

int attn_rope_decode_launch(int dtype, int D, const AttnRopeArgs &a, hipStream_t st) {
    PIE_REQUIRE(a.Hkv > 0 && a.Hq % a.Hkv == 0, PIE_E_SHAPE, "sdpa_decode: Hq must be a multiple of Hkv");
    PIE_REQUIRE(a.splits >= 1 && a.splits <= ATTN_MAX_SPLITS, PIE_E_ARG, "sdpa_decode: bad split count");
    PIE_REQUIRE(a.total && (a.splits == 1 || a.arrived), PIE_E_ARG, "sdpa_decode: a step needs the sum of its lengths, a split one its counters");
    const int rep = a.Hq / a.Hkv;
#define STEP_D(T_, D_) return a.nt_kv ? step_go<T_, D_, true, true, true>(rep, a, st) : step_go<T_, D_, false, true, true>(rep, a, st)
    if (dtype == PIE_BF16 && D == 128) STEP_D(BF16, 128);
    if (dtype == PIE_BF16 && D == 64) STEP_D(BF16, 64);
    if (dtype == PIE_F16 && D == 128) STEP_D(F16, 128);
    if (dtype == PIE_F16 && D == 64) STEP_D(F16, 64);
#undef STEP_D
    return pie::fail(PIE_E_SHAPE, "sdpa_decode: head_dim must be 64 or 128 and dtype bf16/f16");
}

int attn_one_launch(int dtype, int D, const AttnArgs &args, hipStream_t st) {  // (attn_decode_launch has looked at the arguments)
    AttnRopeArgs a = {};
    static_cast<AttnArgs &>(a) = args;
    const int rep = a.Hq / a.Hkv;
#define STEP_D(T_, D_) return a.block_table ? step_go<T_, D_, false, false, true>(rep, a, st) : step_go<T_, D_, false, false, false>(rep, a, st)
    if (dtype == PIE_BF16 && D == 128) STEP_D(BF16, 128);
    if (dtype == PIE_BF16) STEP_D(BF16, 64);
    if (D == 128) STEP_D(F16, 128);
    STEP_D(F16, 64);
#undef STEP_D
}
