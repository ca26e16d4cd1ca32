// vision.hip -- op-level kernels of the Qwen2.5-VL vision tower (reference models/intern/vision.py:87-442).
//
// The tower is dense 16-bit GEMMs (the hand-written MFMA GEMM of w16_gemm.hpp on W16M-tiled weights: pie_linear_w16m, with the bias and
// the MLP's SiLU * up in its epilogue) plus four hand-written pieces: the rotate-half rotary embedding with per-patch (row, column) angles fused with the q / k / v re-layout the attention
// kernel wants, block-diagonal non-causal attention on the MFMA units (prefill_attn.hpp, SEG instantiation: full-image and
// 64-patch-window layers are the same kernel with different segment tables), bias add for any column count, and erf-GELU.
// RMSNorm, SiLU*up and residual adds are the ops the text tower already has (ops.hip).
#include "prefill_attn.hpp"

// nn.GELU() (exact): x * (1 + erf(x / sqrt 2)) / 2  (PatchMerger.mlp[1], vision.py:130)
template <class T>
__global__ void k_gelu(const u16 *x, size_t n, u16 *y) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float v = T::to_f32(x[i]);
    y[i] = T::from_f32(v * (1.0f + erff(v * 0.70710678118654752440f)) * 0.5f);
}

// Attention.__call__, vision.py:152-158 + the layout step: qkv [N, 3, H, D] (the qkv Linear's output) ->
//   q [N, H, DP] = rope(q), k [H, N, DP] = rope(k), v [H, N, DP] = v, head dims D..DP-1 zero (DP = 64 or 128: the MFMA
//   attention's head sizes; zero columns change neither the scores nor the output's first D dims).
// rope = apply_rotary_pos_emb_vision (vision.py:55-70): x * cos + rotate_half(x) * sin in fp32, one rounding;
// cos / sin fp32 [N, D/2] (the row's angles, tiled twice over the head dim).  One thread per (row, head, pair d < D/2).
// `bias` (nullable, [3 * H * D]): the qkv Linear's bias, added here -- T(x + b), the Linear's own rounding -- instead of in a pass
// of its own over the GEMM output.
template <class T>
__global__ void k_vision_qkv_rope(const u16 *qkv, const u16 *bias, const float *cs, const float *sn, int N, int H, int D, int DP, u16 *q, u16 *k,
                                  u16 *v) {
    const int half = D >> 1, hp = DP >> 1;
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (size_t)N * H * hp) return;
    const int d = (int)(i % hp), hh = (int)((i / hp) % H), n = (int)(i / ((size_t)hp * H));
    u16 *qo = q + ((size_t)n * H + hh) * DP, *ko = k + ((size_t)hh * N + n) * DP, *vo = v + ((size_t)hh * N + n) * DP;
    if (d >= half) {  // padding pairs: columns D + 2 (d - half), + 1
        const int c0 = D + 2 * (d - half);
        if (c0 + 1 < DP) qo[c0] = qo[c0 + 1] = ko[c0] = ko[c0 + 1] = vo[c0] = vo[c0 + 1] = 0;
        return;
    }
    const u16 *row = qkv + (size_t)n * 3 * H * D + (size_t)hh * D;
    const u16 *brow = bias ? bias + (size_t)hh * D : nullptr;
    auto ld = [&](int part, int col) {  // element `col` of this head's q (0) / k (1) / v (2) row, bias applied
        const float x = T::to_f32(row[(size_t)part * H * D + col]);
        return brow ? round_T<T>(x + T::to_f32(brow[(size_t)part * H * D + col])) : x;
    };
    const float c = cs[(size_t)n * half + d], s = sn[(size_t)n * half + d];
    {
        const float a = ld(0, d), b = ld(0, d + half);
        qo[d] = T::from_f32(__fadd_rn(__fmul_rn(a, c), __fmul_rn(-b, s)));
        qo[d + half] = T::from_f32(__fadd_rn(__fmul_rn(b, c), __fmul_rn(a, s)));
    }
    {
        const float a = ld(1, d), b = ld(1, d + half);
        ko[d] = T::from_f32(__fadd_rn(__fmul_rn(a, c), __fmul_rn(-b, s)));
        ko[d + half] = T::from_f32(__fadd_rn(__fmul_rn(b, c), __fmul_rn(a, s)));
    }
    vo[d] = T::from_f32(ld(2, d)), vo[d + half] = T::from_f32(ld(2, d + half));
}

// The same, four pairs per thread with 8-byte accesses (D % 8 == 0: every head size the tower uses); the scalar kernel above is
// the fallback.  At 4096 patches: 50 -> see DESIGN.md 2d (the scalar form moved 2 bytes per lane per access).
template <class T>
__global__ void k_vision_qkv_rope_v4(const u16 *qkv, const u16 *bias, const float *cs, const float *sn, int N, int H, int D, int DP, u16 *q, u16 *k,
                                     u16 *v) {
    const int half = D >> 1, hp4 = DP >> 3;  // groups of 4 pairs per padded head
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (size_t)N * H * hp4) return;
    const int d0 = (int)(i % hp4) * 4, hh = (int)((i / hp4) % H), n = (int)(i / ((size_t)hp4 * H));
    u16 *qo = q + ((size_t)n * H + hh) * DP, *ko = k + ((size_t)hh * N + n) * DP, *vo = v + ((size_t)hh * N + n) * DP;
    if (d0 >= half) {  // 8 padding columns
        const int c0 = D + 2 * (d0 - half);
        const uint4 z = make_uint4(0, 0, 0, 0);
        *reinterpret_cast<uint4 *>(qo + c0) = z, *reinterpret_cast<uint4 *>(ko + c0) = z, *reinterpret_cast<uint4 *>(vo + c0) = z;
        return;
    }
    const u16 *row = qkv + (size_t)n * 3 * H * D + (size_t)hh * D;
    const u16 *brow = bias ? bias + (size_t)hh * D : nullptr;
    const float4 c = *reinterpret_cast<const float4 *>(cs + (size_t)n * half + d0), s = *reinterpret_cast<const float4 *>(sn + (size_t)n * half + d0);
    const float cc[4] = {c.x, c.y, c.z, c.w}, ss[4] = {s.x, s.y, s.z, s.w};
    auto ld4 = [&](int part, int col, float *o) {  // 4 elements of this head's q / k / v row, bias applied
        const uint2 x = *reinterpret_cast<const uint2 *>(row + (size_t)part * H * D + col);
        o[0] = lo_f32<T>(x.x), o[1] = hi_f32<T>(x.x), o[2] = lo_f32<T>(x.y), o[3] = hi_f32<T>(x.y);
        if (brow) {
            const uint2 b = *reinterpret_cast<const uint2 *>(brow + (size_t)part * H * D + col);
            o[0] = round_T<T>(o[0] + lo_f32<T>(b.x)), o[1] = round_T<T>(o[1] + hi_f32<T>(b.x));
            o[2] = round_T<T>(o[2] + lo_f32<T>(b.y)), o[3] = round_T<T>(o[3] + hi_f32<T>(b.y));
        }
    };
    auto st4 = [&](u16 *dst, const float *o) { *reinterpret_cast<uint2 *>(dst) = make_uint2(pack2<T>(o[0], o[1]), pack2<T>(o[2], o[3])); };
#pragma unroll
    for (int part = 0; part < 2; ++part) {
        float a[4], b[4], lo[4], hi[4];
        ld4(part, d0, a), ld4(part, d0 + half, b);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            lo[j] = __fadd_rn(__fmul_rn(a[j], cc[j]), __fmul_rn(-b[j], ss[j]));
            hi[j] = __fadd_rn(__fmul_rn(b[j], cc[j]), __fmul_rn(a[j], ss[j]));
        }
        u16 *dst = part == 0 ? qo : ko;
        st4(dst + d0, lo), st4(dst + d0 + half, hi);
    }
    float a[4], b[4];
    ld4(2, d0, a), ld4(2, d0 + half, b);
    st4(vo + d0, a), st4(vo + d0 + half, b);
}

// MLP.__call__ (vision.py:196-197) between the GEMMs: act = T(T(silu(T(g + bg))) * T(u + bu)); two columns per thread.
template <class T>
__global__ void k_bias_silu_mul(const u16 *g, const u16 *u, const u16 *bg, const u16 *bu, int M, int N, int ld, u16 *y) {
    const int n2 = (N + 1) >> 1;
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (size_t)M * n2) return;
    const int n = (int)(i % n2) * 2;
    const size_t o = (i / n2) * (size_t)N + n, oi = (i / n2) * (size_t)ld + n;  // output / input (row stride ld) offsets
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        if (n + j >= N) break;
        const float gv = round_T<T>(T::to_f32(g[oi + j]) + T::to_f32(bg[n + j])), uv = round_T<T>(T::to_f32(u[oi + j]) + T::to_f32(bu[n + j]));
        y[o + j] = T::from_f32(round_T<T>(gv / (1.0f + expf(-gv))) * uv);
    }
}

// four columns per thread, 8-byte accesses (N % 4 == 0)
template <class T>
__global__ void k_bias_silu_mul_v4(const u16 *g, const u16 *u, const u16 *bg, const u16 *bu, int M, int N, int ld, u16 *y) {
    const int n4 = N >> 2;
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (size_t)M * n4) return;
    const int n = (int)(i % n4) * 4;
    const size_t o = (i / n4) * (size_t)N + n, oi = (i / n4) * (size_t)ld + n;
    const uint2 gv = *reinterpret_cast<const uint2 *>(g + oi), uv = *reinterpret_cast<const uint2 *>(u + oi);
    const uint2 bgv = *reinterpret_cast<const uint2 *>(bg + n), buv = *reinterpret_cast<const uint2 *>(bu + n);
    const float gg[4] = {lo_f32<T>(gv.x), hi_f32<T>(gv.x), lo_f32<T>(gv.y), hi_f32<T>(gv.y)};
    const float uu[4] = {lo_f32<T>(uv.x), hi_f32<T>(uv.x), lo_f32<T>(uv.y), hi_f32<T>(uv.y)};
    const float bgg[4] = {lo_f32<T>(bgv.x), hi_f32<T>(bgv.x), lo_f32<T>(bgv.y), hi_f32<T>(bgv.y)};
    const float buu[4] = {lo_f32<T>(buv.x), hi_f32<T>(buv.x), lo_f32<T>(buv.y), hi_f32<T>(buv.y)};
    float r[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const float a = round_T<T>(gg[j] + bgg[j]), b = round_T<T>(uu[j] + buu[j]);
        r[j] = round_T<T>(a / (1.0f + expf(-a))) * b;
    }
    *reinterpret_cast<uint2 *>(y + o) = make_uint2(pack2<T>(r[0], r[1]), pack2<T>(r[2], r[3]));
}

// hidden_states + Linear(...) (vision.py:212-218) with the Linear's bias folded in: y = T(x + T(r + b)).
template <class T>
__global__ void k_add_bias(const u16 *x, const u16 *r, const u16 *b, int M, int N, u16 *y) {
    const int n2 = (N + 1) >> 1;
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (size_t)M * n2) return;
    const int n = (int)(i % n2) * 2;
    const size_t o = (i / n2) * (size_t)N + n;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        if (n + j >= N) break;
        y[o + j] = T::from_f32(T::to_f32(x[o + j]) + round_T<T>(T::to_f32(r[o + j]) + T::to_f32(b[n + j])));
    }
}

// The residual add (with the preceding Linear's bias) and the RMSNorm that follows it in one pass over the row (vision.py:212-218 ->
// :213 / :218's norm): y = T(x + T(r + b)), xn = w * T(y * rsqrt(mean(y^2) + eps)).  One workgroup per row, H % 8 == 0, H <= 8192.
template <class T>
__global__ void __launch_bounds__(256) k_add_bias_rms_norm(const u16 *x, const u16 *r, const u16 *b, const u16 *w, float eps, int H, u16 *y, u16 *xn) {
    __shared__ float red[4];
    const size_t base = (size_t)blockIdx.x * H;
    constexpr int MAXP = 4;
    uint4 hv[MAXP];
    float ssq = 0.0f;
#pragma unroll
    for (int p = 0; p < MAXP; ++p) {
        const int i = (threadIdx.x + p * 256) * 8;
        if (i < H) {
            const uint4 a = *reinterpret_cast<const uint4 *>(x + base + i), c = *reinterpret_cast<const uint4 *>(r + base + i);
            const uint4 bb = *reinterpret_cast<const uint4 *>(b + i);
            const u32 av[4] = {a.x, a.y, a.z, a.w}, cv[4] = {c.x, c.y, c.z, c.w}, bv[4] = {bb.x, bb.y, bb.z, bb.w};
            u32 o[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                o[j] = pack2<T>(lo_f32<T>(av[j]) + round_T<T>(lo_f32<T>(cv[j]) + lo_f32<T>(bv[j])),
                                hi_f32<T>(av[j]) + round_T<T>(hi_f32<T>(cv[j]) + hi_f32<T>(bv[j])));
                const float lo = lo_f32<T>(o[j]), hi = hi_f32<T>(o[j]);
                ssq = fmaf(lo, lo, ssq);
                ssq = fmaf(hi, hi, ssq);
            }
            hv[p] = make_uint4(o[0], o[1], o[2], o[3]);
            *reinterpret_cast<uint4 *>(y + base + i) = hv[p];
        }
    }
    ssq = wave_sum(ssq);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = ssq;
    __syncthreads();
    const float inv = 1.0f / sqrtf((red[0] + red[1] + red[2] + red[3]) / (float)H + eps);
#pragma unroll
    for (int p = 0; p < MAXP; ++p) {
        const int i = (threadIdx.x + p * 256) * 8;
        if (i < H) {
            const uint4 g = *reinterpret_cast<const uint4 *>(w + i);
            const u32 vv[4] = {hv[p].x, hv[p].y, hv[p].z, hv[p].w}, gg[4] = {g.x, g.y, g.z, g.w};
            u32 o[4];
#pragma unroll
            for (int j = 0; j < 4; ++j)
                o[j] = pack2<T>(round_T<T>(lo_f32<T>(vv[j]) * inv) * lo_f32<T>(gg[j]), round_T<T>(hi_f32<T>(vv[j]) * inv) * hi_f32<T>(gg[j]));
            *reinterpret_cast<uint4 *>(xn + base + i) = make_uint4(o[0], o[1], o[2], o[3]);
        }
    }
}

template <class F16F, class BF16F>
static int by_dt(int dtype, F16F &&f16, BF16F &&bf16, const char *who) {
    if (dtype == PIE_F16) f16();
    else if (dtype == PIE_BF16) bf16();
    else return pie::fail(PIE_E_ARG, std::string(who) + ": dtype must be PIE_BF16 or PIE_F16");
    PIE_LAUNCH_CHECK();
    return PIE_OK;
}

// DP: 64, 128, or D itself (no padding)
static int qkv_rope(const void *qkv, const void *bias, const float *cos_t, const float *sin_t, int N, int H, int D, int DP, int dtype, void *q, void *k, void *v, void *stream) {
    hipStream_t st = (hipStream_t)stream;
    if (D % 8 == 0 && pie_aligned(qkv, 8) && pie_aligned(q, 16) && pie_aligned(k, 16) && pie_aligned(v, 16) && (!bias || pie_aligned(bias, 8)) &&
        pie_aligned(cos_t, 16) && pie_aligned(sin_t, 16)) {
        const size_t n4 = (size_t)N * H * (DP / 8);
        const dim3 grid4((unsigned)((n4 + 255) / 256)), block4(256);
        return by_dt(
            dtype,
            [&] { hipLaunchKernelGGL(k_vision_qkv_rope_v4<F16>, grid4, block4, 0, st, (const u16 *)qkv, (const u16 *)bias, cos_t, sin_t, N, H, D, DP, (u16 *)q, (u16 *)k, (u16 *)v); },
            [&] { hipLaunchKernelGGL(k_vision_qkv_rope_v4<BF16>, grid4, block4, 0, st, (const u16 *)qkv, (const u16 *)bias, cos_t, sin_t, N, H, D, DP, (u16 *)q, (u16 *)k, (u16 *)v); },
            "pie_vision_qkv_rope");
    }
    const size_t n = (size_t)N * H * (DP / 2);
    const dim3 grid((unsigned)((n + 255) / 256)), block(256);
    return by_dt(
        dtype,
        [&] { hipLaunchKernelGGL(k_vision_qkv_rope<F16>, grid, block, 0, st, (const u16 *)qkv, (const u16 *)bias, cos_t, sin_t, N, H, D, DP, (u16 *)q, (u16 *)k, (u16 *)v); },
        [&] { hipLaunchKernelGGL(k_vision_qkv_rope<BF16>, grid, block, 0, st, (const u16 *)qkv, (const u16 *)bias, cos_t, sin_t, N, H, D, DP, (u16 *)q, (u16 *)k, (u16 *)v); },
        "pie_vision_qkv_rope");
}

extern "C" {

int pie_gelu(const void *x, size_t n, int dtype, void *y, void *stream) {
    PIE_REQUIRE(x && y, PIE_E_ARG, "pie_gelu: null pointer");
    PIE_REQUIRE(n > 0, PIE_E_SHAPE, "pie_gelu: empty input");
    hipStream_t st = (hipStream_t)stream;
    const dim3 grid((unsigned)((n + 255) / 256)), block(256);
    return by_dt(
        dtype, [&] { hipLaunchKernelGGL(k_gelu<F16>, grid, block, 0, st, (const u16 *)x, n, (u16 *)y); },
        [&] { hipLaunchKernelGGL(k_gelu<BF16>, grid, block, 0, st, (const u16 *)x, n, (u16 *)y); }, "pie_gelu");
}

int pie_vision_qkv_rope(const void *qkv, const void *bias, const float *cos_t, const float *sin_t, int N, int H, int D, int DP, int dtype, void *q,
                        void *k, void *v, void *stream) {
    PIE_REQUIRE(qkv && cos_t && sin_t && q && k && v, PIE_E_ARG, "pie_vision_qkv_rope: null pointer");
    PIE_REQUIRE(N > 0 && H > 0 && D > 0 && D % 2 == 0 && (DP == 64 || DP == 128) && D <= DP, PIE_E_SHAPE,
                "pie_vision_qkv_rope: head_dim must be even and fit the padded size 64 or 128");
    return qkv_rope(qkv, bias, cos_t, sin_t, N, H, D, DP, dtype, q, k, v, stream);
}

int pie_bias_silu_mul(const void *gate, const void *up, const void *bias_gate, const void *bias_up, int M, int N, int ld, int dtype, void *y,
                      void *stream) {
    PIE_REQUIRE(gate && up && bias_gate && bias_up && y, PIE_E_ARG, "pie_bias_silu_mul: null pointer");
    PIE_REQUIRE(M > 0 && N > 0, PIE_E_SHAPE, "pie_bias_silu_mul: empty input");
    if (ld == 0) ld = N;
    PIE_REQUIRE(ld >= N, PIE_E_SHAPE, "pie_bias_silu_mul: row stride smaller than the row");
    hipStream_t st = (hipStream_t)stream;
    if (N % 4 == 0 && ld % 4 == 0 && pie_aligned(gate, 8) && pie_aligned(up, 8) && pie_aligned(bias_gate, 8) && pie_aligned(bias_up, 8) && pie_aligned(y, 8)) {
        const size_t n4 = (size_t)M * (N / 4);
        const dim3 grid4((unsigned)((n4 + 255) / 256)), block4(256);
        return by_dt(
            dtype,
            [&] { hipLaunchKernelGGL(k_bias_silu_mul_v4<F16>, grid4, block4, 0, st, (const u16 *)gate, (const u16 *)up, (const u16 *)bias_gate, (const u16 *)bias_up, M, N, ld, (u16 *)y); },
            [&] { hipLaunchKernelGGL(k_bias_silu_mul_v4<BF16>, grid4, block4, 0, st, (const u16 *)gate, (const u16 *)up, (const u16 *)bias_gate, (const u16 *)bias_up, M, N, ld, (u16 *)y); },
            "pie_bias_silu_mul");
    }
    const size_t n = (size_t)M * ((N + 1) >> 1);
    const dim3 grid((unsigned)((n + 255) / 256)), block(256);
    return by_dt(
        dtype,
        [&] { hipLaunchKernelGGL(k_bias_silu_mul<F16>, grid, block, 0, st, (const u16 *)gate, (const u16 *)up, (const u16 *)bias_gate, (const u16 *)bias_up, M, N, ld, (u16 *)y); },
        [&] { hipLaunchKernelGGL(k_bias_silu_mul<BF16>, grid, block, 0, st, (const u16 *)gate, (const u16 *)up, (const u16 *)bias_gate, (const u16 *)bias_up, M, N, ld, (u16 *)y); },
        "pie_bias_silu_mul");
}

int pie_add_bias(const void *x, const void *r, const void *bias, int M, int N, int dtype, void *y, void *stream) {
    PIE_REQUIRE(x && r && bias && y, PIE_E_ARG, "pie_add_bias: null pointer");
    PIE_REQUIRE(M > 0 && N > 0, PIE_E_SHAPE, "pie_add_bias: empty input");
    hipStream_t st = (hipStream_t)stream;
    const size_t n = (size_t)M * ((N + 1) >> 1);
    const dim3 grid((unsigned)((n + 255) / 256)), block(256);
    return by_dt(
        dtype, [&] { hipLaunchKernelGGL(k_add_bias<F16>, grid, block, 0, st, (const u16 *)x, (const u16 *)r, (const u16 *)bias, M, N, (u16 *)y); },
        [&] { hipLaunchKernelGGL(k_add_bias<BF16>, grid, block, 0, st, (const u16 *)x, (const u16 *)r, (const u16 *)bias, M, N, (u16 *)y); }, "pie_add_bias");
}

int pie_add_bias_rms_norm(const void *x, const void *r, const void *bias, const void *norm_w, float eps, int M, int N, int dtype, void *y, void *xn,
                          void *stream) {
    PIE_REQUIRE(x && r && bias && norm_w && y && xn, PIE_E_ARG, "pie_add_bias_rms_norm: null pointer");
    PIE_REQUIRE(M > 0 && N > 0 && N % 8 == 0 && N <= 8192, PIE_E_SHAPE, "pie_add_bias_rms_norm: N must be a multiple of 8, at most 8192");
    PIE_REQUIRE(pie_aligned(x, 16) && pie_aligned(r, 16) && pie_aligned(bias, 16) && pie_aligned(norm_w, 16) && pie_aligned(y, 16) && pie_aligned(xn, 16),
                PIE_E_ALIGN, "pie_add_bias_rms_norm: 16-byte alignment required");
    hipStream_t st = (hipStream_t)stream;
    return by_dt(
        dtype,
        [&] { hipLaunchKernelGGL(k_add_bias_rms_norm<F16>, dim3(M), dim3(256), 0, st, (const u16 *)x, (const u16 *)r, (const u16 *)bias, (const u16 *)norm_w, eps, N, (u16 *)y, (u16 *)xn); },
        [&] { hipLaunchKernelGGL(k_add_bias_rms_norm<BF16>, dim3(M), dim3(256), 0, st, (const u16 *)x, (const u16 *)r, (const u16 *)bias, (const u16 *)norm_w, eps, N, (u16 *)y, (u16 *)xn); },
        "pie_add_bias_rms_norm");
}

}  // extern "C"

// D: 64, 128, or 80 (rows without padding); out: rows of H heads of out_d columns (0: D)
static int segment_attn(const void *q, const void *k, const void *v, const int32_t *seg_lo, const int32_t *seg_hi, int N, int H, int D, int out_d, float scale, int dtype, void *out, void *stream) {
    PIE_REQUIRE(q && k && v && seg_lo && seg_hi && out, PIE_E_ARG, "pie_sdpa_segments: null pointer");
    PIE_REQUIRE(N > 0 && H > 0, PIE_E_SHAPE, "pie_sdpa_segments: empty input");
    PIE_REQUIRE(pie_aligned(q, 16) && pie_aligned(k, 16) && pie_aligned(v, 16) && pie_aligned(out, 8), PIE_E_ALIGN, "pie_sdpa_segments: misaligned pointer");
    PrefillAttnArgs a = {};
    a.q = (const u16 *)q, a.k = (const u16 *)k, a.v = (const u16 *)v, a.offset = 0, a.cap = N;
    a.seg_lo = seg_lo, a.seg_hi = seg_hi;
    a.M = N, a.Hq = H, a.Hkv = H, a.scale = scale, a.out = (u16 *)out, a.out_d = out_d;
    if (dtype == PIE_BF16) return segment_attn_launch_t<BF16>(a, D, (hipStream_t)stream);
    if (dtype == PIE_F16) return segment_attn_launch_t<F16>(a, D, (hipStream_t)stream);
    return pie::fail(PIE_E_ARG, "pie_sdpa_segments: dtype must be PIE_BF16 or PIE_F16");
}

// The attention of a block over windows, from the qkv Linear's rows (no bias yet): heads of 64 and 80, windows that a tile of 64 query rows covers.  A longer one's keys are rotated again by every tile
// of its rows, 64 at a time behind a barrier with no loads in flight.  us a block of the tower's 16 heads of 80, rotation in a launch of its own / here, 256 / 1024 / 2304 / 4096 patches: windows of 64 two / four / one /
// six less here; of 100 level, level, 6 and 12 more; of 144 level, 1, 8 and 16 more; of 256 1, level, 11 and 10 more; of 1024 level, 12, 25 and 77 more.  Heads of 64: of 64 five to seven less here, of 100 to 256 three less
// to five more.
static bool segment_rot_serves(int window, int head_dim, const void *bias, const float *cos_t, const float *sin_t) {
    return window > 0 && window <= 64 && (head_dim == 64 || head_dim == 80) && pie_aligned(bias, 16) && pie_aligned(cos_t, 16) && pie_aligned(sin_t, 16);
}
static int segment_rot(const void *qkv, const void *bias, const float *cos_t, const float *sin_t, const int32_t *seg_lo, const int32_t *seg_hi, int N, int H, int D, float scale, int dtype, void *out, void *stream) {
    PIE_REQUIRE(dtype == PIE_BF16 || dtype == PIE_F16, PIE_E_ARG, "segment attention: dtype must be PIE_BF16 or PIE_F16");
    PrefillAttnArgs a = {};
    a.q = (const u16 *)qkv, a.cap = N, a.seg_lo = seg_lo, a.seg_hi = seg_hi, a.M = N, a.Hq = H, a.Hkv = H, a.scale = scale, a.out = (u16 *)out;
    a.rot_bias = (const u16 *)bias, a.rot_cos = cos_t, a.rot_sin = sin_t;
    return dtype == PIE_BF16 ? segment_rot_launch_t<BF16>(a, D, (hipStream_t)stream) : segment_rot_launch_t<F16>(a, D, (hipStream_t)stream);
}

// Scratch of pie_vision_blocks, in order; every part a multiple of 256 bytes.  The qkv rows and the MLP's activation are never alive together.
struct VisionScratch {
    size_t wide, head, out, gemm;  // bytes of: qkv / activation rows, q (k, v) rows, the products' output and the attention's rows (each), slabs of a product that splits K
    size_t total() const { return wide + 3 * head + 2 * out + gemm; }
};
static int vision_head_row(int head_dim) { return head_dim <= 64 ? 64 : head_dim == 80 ? 80 : 128; }  // columns of a q, k or v row between the rotation and the attention (k_prefill_attn's DR)
static VisionScratch vision_scratch(int rows, int hidden, int inter, int heads, int head_dim) {
    auto up = [](size_t n) { return (n + 255) & ~(size_t)255; };
    auto most = [](size_t a, size_t b) { return a > b ? a : b; };
    const int act = (inter + 63) & ~63, DP = vision_head_row(head_dim);
    const size_t slabs = most(most(pie_linear_w16m_workspace(rows, 3 * hidden, hidden), pie_linear_w16m_workspace(rows, hidden, hidden)), pie_linear_w16m_workspace(rows, hidden, inter));
    return {up((size_t)rows * (3 * hidden > act ? 3 * hidden : act) * 2), up((size_t)rows * heads * DP * 2), up((size_t)rows * hidden * 2), up(slabs)};
}
static bool vision_shape(int rows, int hidden, int inter, int heads, int head_dim) {
    return rows > 0 && hidden > 0 && hidden % 64 == 0 && hidden <= 8192 && inter > 0 && inter % 4 == 0 && heads > 0 && head_dim % 4 == 0 && head_dim <= 128 && heads * head_dim == hidden;
}

extern "C" {

int pie_sdpa_segments(const void *q, const void *k, const void *v, const int32_t *seg_lo, const int32_t *seg_hi, int N, int H, int D, float scale,
                      int dtype, void *out, void *stream) {
    PIE_REQUIRE(D == 64 || D == 128, PIE_E_SHAPE, "pie_sdpa_segments: head_dim must be 64 or 128");
    return segment_attn(q, k, v, seg_lo, seg_hi, N, H, D, 0, scale, dtype, out, stream);
}

size_t pie_vision_blocks_workspace(int rows, int hidden, int inter, int heads, int head_dim) {
    return vision_shape(rows, hidden, inter, heads, head_dim) ? vision_scratch(rows, hidden, inter, heads, head_dim).total() : 0;
}

// One call for all blocks: seven or eight launches each, which a host that calls op by op starts in 12 us apiece (0.92 ms for eight blocks of the 7B tower's widths, the time of an image up to 448 x 448)
// and this one in 2-3.
int pie_vision_blocks(const pie_vision_block *blocks, int n_blocks, int rows, int hidden, int inter, int heads, int head_dim, float eps, const float *cos_t, const float *sin_t, const int32_t *full_lo,
                      const int32_t *full_hi, const int32_t *win_lo, const int32_t *win_hi, int dtype, void *x, void *xn, void *workspace, size_t workspace_bytes, void *stream) {
    PIE_REQUIRE(blocks && cos_t && sin_t && full_lo && full_hi && win_lo && win_hi && x && xn && workspace, PIE_E_ARG, "pie_vision_blocks: null pointer");
    PIE_REQUIRE(n_blocks > 0 && vision_shape(rows, hidden, inter, heads, head_dim), PIE_E_SHAPE,
                "pie_vision_blocks: hidden = heads * head_dim, a multiple of 64 up to 8192; inter and head_dim multiples of 4, head_dim up to 128");
    PIE_REQUIRE(pie_aligned(workspace, 256), PIE_E_ALIGN, "pie_vision_blocks: the workspace needs 256-byte alignment");
    const VisionScratch z = vision_scratch(rows, hidden, inter, heads, head_dim);
    PIE_REQUIRE(workspace_bytes >= z.total(), PIE_E_ARG, "pie_vision_blocks: workspace smaller than pie_vision_blocks_workspace()");
    const int DP = vision_head_row(head_dim), act_ld = (inter + 63) & ~63;
    char *p = (char *)workspace;
    char *wide = p, *q = wide + z.wide, *k = q + z.head, *v = k + z.head, *att = v + z.head, *r = att + z.out, *slabs = r + z.out;
    const float scale = (float)(1.0 / sqrt((double)head_dim));
    auto linear = [&](const void *in, int ldx, const void *w, int N, int K, void *y) {
        return pie_linear_w16m(in, ldx, w, nullptr, rows, N, K, dtype, y, N, 0, z.gemm ? slabs : nullptr, z.gemm, stream);
    };
    for (int i = 0; i < n_blocks; ++i) {
        const pie_vision_block &b = blocks[i];
        PIE_REQUIRE(b.qkv_w && b.qkv_b && b.proj_w && b.proj_b && b.norm2 && b.gateup_w && b.gateup_b && b.down_w && b.down_b && b.next_norm, PIE_E_ARG, "pie_vision_blocks: null weight");
        int rc = linear(xn, hidden, b.qkv_w, 3 * hidden, hidden, wide);
        if (!rc && !b.full && segment_rot_serves(b.window, head_dim, b.qkv_b, cos_t, sin_t)) rc = segment_rot(wide, b.qkv_b, cos_t, sin_t, win_lo, win_hi, rows, heads, head_dim, scale, dtype, att, stream);
        else {
            if (!rc) rc = qkv_rope(wide, b.qkv_b, cos_t, sin_t, rows, heads, head_dim, DP, dtype, q, k, v, stream);
            if (!rc) rc = segment_attn(q, k, v, b.full ? full_lo : win_lo, b.full ? full_hi : win_hi, rows, heads, DP, head_dim, scale, dtype, att, stream);
        }
        if (!rc) rc = linear(att, hidden, b.proj_w, hidden, hidden, r);
        if (!rc) rc = pie_add_bias_rms_norm(x, r, b.proj_b, b.norm2, eps, rows, hidden, dtype, x, xn, stream);
        if (!rc) rc = pie_linear_w16m(xn, hidden, b.gateup_w, b.gateup_b, rows, 2 * inter, hidden, dtype, wide, act_ld, act_ld == inter ? 1 : PIE_SWIGLU_ZERO_REST, nullptr, 0, stream);
        if (!rc) rc = linear(wide, act_ld, b.down_w, hidden, inter, r);
        if (!rc) rc = pie_add_bias_rms_norm(x, r, b.down_b, b.next_norm, eps, rows, hidden, dtype, x, xn, stream);
        if (rc) return rc;
    }
    return PIE_OK;
}

}  // extern "C"
