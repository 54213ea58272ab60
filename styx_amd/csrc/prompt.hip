// prompt.hip -- the decode path's arithmetic for many prompt tokens at once
// (gfx950): what styx_moe_generate runs for every prompt token but the last.
//
// Token-at-a-time prefill (crates/model/examples/generate_moe.rs:44-56) reads
// every dense matrix, the LM head and k expert slabs per layer again for each
// token.  Here a batch of up to PROMPT_MAX_T tokens goes through a layer
// together, so that each matrix and each routed expert's slab is read once
// per 32 tokens that use it, and the contraction runs on the matrix cores:
//
//   k_prompt_embed   residual rows of the tokens; clears the batch's odd flag
//   k_prompt_pack    a row's RMSNorm / SwiGLU / combine, and its f16 pieces
//   k_prompt_gemm    split-layout quant matrix x token rows (dense matrices,
//                    or the tokens of each routed expert)
//   k_prompt_rope    per-head q/k RMSNorm, rope, K/V rows into the cache
//   k_prompt_attn    causal attention of the batch over the paged cache
//   k_prompt_router, k_prompt_topk, k_prompt_plan
//                    router logits, top-k, tokens grouped by expert
//
// Precision.  A row of K/V left here is as close to 64-bit arithmetic as the
// single-token path's.  Quant values times their 6-bit (q4_K, q5_K) sub-block
// scale are integers below 2048, q8_0 and q6_K quants are integers below 128:
// all exact in f16 (q6_K's 12-bit products with its 8-bit scale are an f16
// plus an exact remainder).  An activation row is scaled by a power of two so
// that its largest value lies in [2^13, 2^14) and written as three f16 pieces
// x = p1 + p2 + p3, p1 a multiple of 16, p2 and p3 each the rounding of what
// is left: 23 bits of every value, to 39 bits below the row's maximum.  v_mfma_f32_16x16x32_f16 forms exact products, and sums of
// integers below 2^24 are exact in its f32 accumulator, so p1's products of
// 256 values (integers times 16) are summed without an error to speak of; the
// products of p2 and p3 go into an accumulator of their own.  (With a first
// piece that is just x's rounding, the low bits of every addition to its sum
// were dropped downwards by the matrix core.)  A matrix's f16
// block factor multiplies the block's sum, and blocks are added up, in f64.
// Layer-0 V rows against 64 bits, relative L2, here and token by token: q8_0
// 7.1e-8, 8.6e-8; q4_K 9.6e-8, 1.02e-7; q5_K 9.6e-8, 1.06e-7; q6_K 5.9e-8,
// 9.0e-8 (2048 columns, 300 tokens).
#include "attn16.h"
#include "deq.h"
#include "head.h"
#include "kernels.h"
#include "qdot.h"
#include "topk.h"

#include <algorithm>

namespace styx {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef double d4 __attribute__((ext_vector_type(4)));

constexpr int PWG = 256;                 // threads of every kernel here but the plan
constexpr int KC = 256;                  // values of a row per GEMM step
constexpr int XROW = KC * 2 + 16;        // bytes of a token's piece of a step in LDS

// ------------------------------------------------------------ embedding ----
__global__ void __launch_bounds__(PWG) k_prompt_embed(int t, const uint8_t *w, int64_t nrows,
                                                      int ncols, const uint32_t *tok, float *x,
                                                      int *odd)
{
    if (blockIdx.x == 0 && threadIdx.x == 0) *odd = 0;
    const int be = blk_elems(t), nb = ncols / be;
    const Mat m = mat_at(w, t, nrows * nb);
    const int64_t r = tok[blockIdx.x];
    float *o = x + (int64_t)blockIdx.x * ncols;
    for (int b = threadIdx.x; b < nb; b += PWG) deq_block(t, m, r * nb + b, o + (int64_t)b * be);
}

hipError_t launch_prompt_embed(hipStream_t st, int t, const uint8_t *w, int64_t nrows, int ncols,
                               const uint32_t *tok, int T, float *x, int *odd)
{
    if (T < 1 || !odd || ncols % blk_elems(t)) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_prompt_embed, dim3(T), dim3(PWG), 0, st, t, w, nrows, ncols, tok, x, odd);
    return hipGetLastError();
}

// ----------------------------------------------------------------- pack ----
// One row per workgroup:
//   PACK_PLAIN    v = src
//   PACK_NORM     v = rms_norm(src) * norm_w
//   PACK_SWIGLU   v = silu(src) * u
//   PACK_COMBINE  src += sum_s w_s y[inv[row k + s]] (s ascending,
//                 moe_reduce_f32.comp:8-13), += sigmoid(gate) y_sh
//                 (axpy_sig_f32.comp), written back; then as PACK_NORM
// and the pieces of v, the sums of its runs of 32 (the minimum terms of
// q4_K / q5_K; formed in f64) as pieces scaled by a further 2^-6, the third
// piece first, and 2^-e of the row.
__device__ __forceinline__ float pack_max(float v, float *red)
{
    v = wave_max(v);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    return fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
}

// v = a + b + c: a a multiple of 16, b the rounding of the rest, c of that
// rest's (|v| < 2^14)
template <typename F> __device__ __forceinline__ void pieces3(F v, _Float16 &a, _Float16 &b, _Float16 &c)
{
    // adding and taking off 1.5 2^p u, p the mantissa's length, rounds to a
    // multiple of u
    constexpr F mid = sizeof(F) == 4 ? (F)12582912.0 : (F)6755399441055744.0;
    const F p1 = (v + mid * (F)16) - mid * (F)16, r1 = v - p1;
    a = (_Float16)(float)p1;
    b = (_Float16)(float)r1;
    c = (_Float16)(float)(r1 - (F)b);
}
// v of the lane that the DPP control CTRL names
template <int CTRL> __device__ __forceinline__ double dpp_d(double v)
{
    const uint64_t u = (uint64_t)__double_as_longlong(v);
    return __longlong_as_double((long long)join64(dpp_u<CTRL>((uint32_t)(u >> 32)), dpp_u<CTRL>((uint32_t)u)));
}

template <int MODE> __global__ void __launch_bounds__(PWG) k_prompt_pack(PromptPack a)
{
    extern __shared__ __align__(16) float xs[];  // [n]
    __shared__ float red[16];
    const int64_t row = blockIdx.x;
    float *src = a.src + row * a.n;
    float mx = 0.0f, ss = 0.0f;
    for (int i = threadIdx.x * 4; i < a.n; i += PWG * 4) {
        f4 v = *(const f4 *)(src + i);
        if constexpr (MODE == PACK_SWIGLU) {
            const f4 u = *(const f4 *)(a.u + row * a.n + i);
#pragma unroll
            for (int j = 0; j < 4; j++) v[j] = v[j] / (1.0f + expf(-v[j])) * u[j];
        }
        if constexpr (MODE == PACK_COMBINE) {
            // eight slots' rows in flight at once; an absent slot reads row 0
            // and adds nothing
            f4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
            for (int s0 = 0; s0 < a.k; s0 += 8) {
                f4 y[8];
                float w[8];
                bool on[8];
#pragma unroll
                for (int s = 0; s < 8; s++) {
                    const int p = s0 + s < a.k ? a.inv[row * a.k + s0 + s] : -1;
                    on[s] = p >= 0;
                    w[s] = s0 + s < a.k ? a.wts[row * MAX_TOPK + s0 + s] : 0.0f;
                    y[s] = *(const f4 *)(a.y + (int64_t)max(p, 0) * a.n + i);
                }
#pragma unroll
                for (int s = 0; s < 8; s++)
                    if (on[s])
#pragma unroll
                        for (int j = 0; j < 4; j++) acc[j] += w[s] * y[s][j];
            }
            v += acc;
            if (a.y_sh) {
                const float sg = 1.0f / (1.0f + expf(-a.gate[row]));
                const f4 y = *(const f4 *)(a.y_sh + row * a.n + i);
#pragma unroll
                for (int j = 0; j < 4; j++) v[j] += sg * y[j];
            }
            *(f4 *)(src + i) = v;
        }
#pragma unroll
        for (int j = 0; j < 4; j++) {
            ss += v[j] * v[j];
            mx = fmaxf(mx, fabsf(v[j]));
        }
        *(f4 *)(xs + i) = v;
    }
    if constexpr (MODE == PACK_NORM || MODE == PACK_COMBINE) {
        ss = block_sum<PWG>(ss, red);
        const float scale = 1.0f / sqrtf(ss / (float)a.n + a.eps);
        float g = 0.0f;
        mx = 0.0f;
        for (int i = threadIdx.x * 4; i < a.n; i += PWG * 4) {
            f4 v = *(const f4 *)(xs + i);
            const f4 w = *(const f4 *)(a.norm_w + i);
#pragma unroll
            for (int j = 0; j < 4; j++) {
                v[j] = (v[j] * scale) * w[j];
                mx = fmaxf(mx, fabsf(v[j]));
            }
            *(f4 *)(xs + i) = v;
            if (a.xn) *(f4 *)(a.xn + row * a.n + i) = v;
            if (a.gate_w) {
                const f4 gw = *(const f4 *)(a.gate_w + i);
#pragma unroll
                for (int j = 0; j < 4; j++) g += gw[j] * v[j];
            }
        }
        if (a.gate_w) {
            g = block_sum<PWG>(g, red);
            if (threadIdx.x == 0) a.gate_out[row] = g;
        }
    }
    mx = pack_max(mx, red);
    // 2^e with max 2^e in [2^13, 2^14) (0, denormal or non-finite maxima
    // keep a usable factor)
    const int ex = (__float_as_int(mx) >> 23) & 255;
    const int e = ex == 0 || ex == 255 ? 0 : min(126, max(-126, 13 - (ex - 127)));
    const float up = __int_as_float((e + 127) << 23);
    if (threadIdx.x == 0) a.v.scale[row] = __int_as_float((127 - e) << 23);
    const int np = a.v.np;
    _Float16 *p1 = (_Float16 *)a.v.p + row * np, *p2 = p1 + a.v.rows * np, *p3 = p2 + a.v.rows * np;
    for (int g = threadIdx.x; g < np / 8; g += PWG) {
        float v[8];
        double s8 = 0.0;
        h8 c1, c2, c3;
#pragma unroll
        for (int i = 0; i < 8; i++) {
            v[i] = 8 * g < a.n ? xs[8 * g + i] : 0.0f;
            s8 += v[i];
            _Float16 x, y, z;
            pieces3(v[i] * up, x, y, z);
            c1[i] = x;
            c2[i] = y;
            c3[i] = z;
        }
        *(h8 *)(p1 + 8 * g) = c1;
        *(h8 *)(p2 + 8 * g) = c2;
        *(h8 *)(p3 + 8 * g) = c3;
        // the run of 32 is held by four neighbouring lanes
        s8 += dpp_d<0xB1>(s8);
        s8 += dpp_d<0x4E>(s8);
        if ((g & 3) == 0) {
            _Float16 x, y, z;
            pieces3(s8 * (double)up * 0.015625, x, y, z);
            const int sb = g >> 2;
            _Float16 *s = (_Float16 *)a.v.sums + (row * (np / KC) + (sb >> 3)) * 32 + (sb & 7);
            s[0] = z;
            s[8] = y;
            s[16] = x;
            s[24] = (_Float16)0.0f;
        }
    }
}

hipError_t launch_prompt_pack(hipStream_t st, int mode, const PromptPack &a, int rows)
{
    if (rows < 1 || a.n < 32 || a.n % 32 || a.n > PROMPT_MAX_N || a.v.n != a.n || rows > a.v.rows)
        return hipErrorInvalidValue;
    const dim3 g(rows), b(PWG);
    const size_t lds = (size_t)a.n * 4;
    switch (mode) {
    case PACK_PLAIN: hipLaunchKernelGGL(k_prompt_pack<PACK_PLAIN>, g, b, lds, st, a); break;
    case PACK_NORM: hipLaunchKernelGGL(k_prompt_pack<PACK_NORM>, g, b, lds, st, a); break;
    case PACK_SWIGLU: hipLaunchKernelGGL(k_prompt_pack<PACK_SWIGLU>, g, b, lds, st, a); break;
    case PACK_COMBINE: hipLaunchKernelGGL(k_prompt_pack<PACK_COMBINE>, g, b, lds, st, a); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

// ----------------------------------------------------------------- GEMM ----
// Matrix-core operands of a weight row: lane (n = lane & 15, g = lane >> 4)
// holds row n's values that the lane's unit loads bring (qdot.h uw_load), so
// every quant byte is loaded once per wave in 16-byte pieces; the step that
// multiplies them takes the activation run of the same eight values.  A step
// s of the 8 per KC values holds, at lane group g, the run of 8 values run<T>(g, s).
template <int T> __device__ __forceinline__ int x_run(int g, int s)
{
    if constexpr (T == T_Q8_0) return 4 * s + 2 * (g & 1) + (g >> 1);
    if constexpr (T == T_Q6_K) return 16 * (g >> 1) + 2 * (g & 1) + 4 * (s >> 1) + (s & 1);
    return 8 * g + s;
}

__device__ __forceinline__ h2 as_h2(uint32_t v) { return __builtin_bit_cast(h2, v); }
__device__ __forceinline__ h2 dup_h2(float v)
{
    const _Float16 h = (_Float16)v;
    return h2{h, h};
}

// Bytes 0,1 and 2,3 of a dword as f16 values 1024 + byte (0x6400 | byte).
__device__ __forceinline__ void bytes_1024(uint32_t v, h2 &a, h2 &b)
{
    a = as_h2(__builtin_amdgcn_perm(0x64646464u, v, 0x04010400u));
    b = as_h2(__builtin_amdgcn_perm(0x64646464u, v, 0x04030402u));
}

__device__ __forceinline__ h8 cat8(h2 a, h2 b, h2 c, h2 d)
{
    return h8{a[0], a[1], b[0], b[1], c[0], c[1], d[0], d[1]};
}

// Buffer loads (a uniform base, 32-bit byte offsets, reads past the end give
// zeros): the 64-bit address of every pending load would otherwise take the
// registers that hold the loads themselves.
struct Buf {
    __amdgpu_buffer_rsrc_t r;
    __device__ __forceinline__ Buf(const void *p, int64_t bytes)
    {
        // the base is uniform: kept in scalar registers whatever it was read from
        const uint64_t u = (uint64_t)(uintptr_t)p;
        const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)u);
        const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(u >> 32));
        r = __builtin_amdgcn_make_buffer_rsrc((void *)(uintptr_t)((uint64_t)hi << 32 | lo), 0,
                                              (int)bytes, 0x00020000);
    }
    __device__ __forceinline__ styx_u4 b128(uint32_t v, uint32_t s = 0) const
    {
        return __builtin_amdgcn_raw_buffer_load_b128(r, v, s, 0);
    }
    __device__ __forceinline__ styx_u2 b64(uint32_t v) const
    {
        return __builtin_amdgcn_raw_buffer_load_b64(r, v, 0, 0);
    }
    __device__ __forceinline__ uint32_t b16(uint32_t v) const
    {
        return __builtin_amdgcn_raw_buffer_load_b16(r, v, 0, 0);
    }
};

// Byte offsets of a matrix's regions (common.h split_of).
struct Reg {
    uint32_t r1, r2, r3;
};

// One row's KC values as loaded: lane group g's unit of K-block blk
// (uw_load's loads).  D8: rows of whole groups of 8 blocks (q8_0; every other
// type loads alike).  Nothing here looks at a loaded value, so the next
// step's loads stay in flight over this step's products.
template <int T, bool D8> struct PW;
template <bool D8> struct PW<T_Q4_K, D8> {
    styx_u4 q0, q1, hd;
    __device__ __forceinline__ void load(const Buf &m, const Reg &o, uint32_t row, int nb, int c, int g)
    {
        const uint32_t blk = row * nb + c, q = (uint32_t)ilv2(blk) + 16 * g;
        q0 = m.b128(q);
        q1 = m.b128(q + 128);
        hd = m.b128(o.r1 + blk * 16);
    }
};
template <bool D8> struct PW<T_Q5_K, D8> {
    styx_u4 q0, q1, h0, h1, hd;
    __device__ __forceinline__ void load(const Buf &m, const Reg &o, uint32_t row, int nb, int c, int g)
    {
        const uint32_t blk = row * nb + c, q = (uint32_t)ilv2(blk) + 16 * g, h = o.r1 + (uint32_t)ilv8(blk);
        q0 = m.b128(q);
        q1 = m.b128(q + 128);
        h0 = m.b128(h);
        h1 = m.b128(h + 128);
        hd = m.b128(o.r2 + blk * 16);
    }
};
template <bool D8> struct PW<T_Q6_K, D8> {
    styx_u4 p0, p1, qh;
    styx_u2 sc;
    uint32_t d;
    __device__ __forceinline__ void load(const Buf &m, const Reg &o, uint32_t row, int nb, int c, int g)
    {
        const uint32_t blk = row * nb + c, q = (uint32_t)ilv2(blk) + 16 * g;
        p0 = m.b128(q);
        p1 = m.b128(q + 128);
        qh = m.b128(o.r1 + blk * 64 + 16 * g);
        sc = m.b64(o.r2 + blk * 16 + 8 * (g >> 1));
        d = m.b16(o.r3 + blk * 2);
    }
};
// q8_0: lane group g loads the half (g & 1) of block 2 i + (g >> 1) of the
// step, i < 4; the swap of halves between the lanes of each pair of groups
// then gives both blocks' operands.  Blocks past the row's end read its
// first block of the step: the activations there are zeros.
template <bool D8> struct PW<T_Q8_0, D8> {
    styx_u4 q[4];
    uint32_t d[D8 ? 4 : 8];
    __device__ __forceinline__ void load(const Buf &m, const Reg &o, uint32_t row, int nb, int c, int g)
    {
        const uint32_t b0 = row * nb + 8 * c;
        const int left = nb - 8 * c;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int b = 2 * i + (g >> 1);
            q[i] = m.b128((uint32_t)ilv8(b0 + (D8 || b < left ? b : 0)) + 128 * (g & 1));
        }
        if constexpr (D8) {
            const styx_u4 v = m.b128(o.r1 + 2 * b0);
            d[0] = v.x, d[1] = v.y, d[2] = v.z, d[3] = v.w;
        } else {
#pragma unroll
            for (int i = 0; i < 8; i++) d[i] = m.b16(o.r1 + 2 * (b0 + (i < left ? i : 0)));
        }
    }
    __device__ __forceinline__ float factor(int b) const
    {
        return f16f(D8 ? d[D8 ? b >> 1 : b] >> (16 * (b & 1)) : d[D8 ? 0 : b]);
    }
};
__device__ __forceinline__ void u4v_to(const styx_u4 v, uint32_t *o)
{
    o[0] = v.x, o[1] = v.y, o[2] = v.z, o[3] = v.w;
}

// acc += the products of a step: xop(t, piece, s) gives the activation
// operand of token tile t, sop(t) its run sums' (q4_K, q5_K).
template <int T, bool D8, int NG, int TT, typename XOp, typename SOp>
__device__ __forceinline__ void gemm_step(const PW<T, D8> (&w)[NG], XOp xop, SOp sop, d4 (&acc)[NG][TT])
{
    const int lane = threadIdx.x & 63, g = lane >> 4;
    auto mm = [](h8 a, h8 b, f4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0); };
    const f4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
    auto widen = [](f4 v) { return __builtin_convertvector(v, d4); };
    if constexpr (T == T_Q8_0) {
        f4 tot[NG][TT];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            h8 op[NG][2];
#pragma unroll
            for (int r = 0; r < NG; r++) {
                // both blocks' operands: lower lanes' high halves against
                // upper lanes' low halves
                const styx_u4 v = w[r].q[i];
                const auto a = __builtin_amdgcn_permlane32_swap(v.x, v.z, false, false);
                const auto b = __builtin_amdgcn_permlane32_swap(v.y, v.w, false, false);
#pragma unroll
                for (int j = 0; j < 2; j++) {
                    h2 e[4];
                    bytes_1024(a[j] ^ 0x80808080u, e[0], e[1]);
                    bytes_1024(b[j] ^ 0x80808080u, e[2], e[3]);
                    const h2 off = dup_h2(-1152.0f);
                    op[r][j] = cat8(e[0] + off, e[1] + off, e[2] + off, e[3] + off);
                }
            }
#pragma unroll
            for (int j = 0; j < 2; j++) {
#pragma unroll
                for (int t = 0; t < TT; t++) {
                    const h8 x1 = xop(t, 0, 2 * i + j), x2 = xop(t, 1, 2 * i + j), x3 = xop(t, 2, 2 * i + j);
#pragma unroll
                    for (int r = 0; r < NG; r++) {
                        const float d = w[r].factor(2 * i + j);
                        const f4 s = mm(x1, op[r][j], zero) + mm(x2, op[r][j], mm(x3, op[r][j], zero));
                        tot[r][t] = (i & 1) + j == 0 ? d * s : tot[r][t] + d * s;
                        // added up here, not kept as products until the end
                        // of the step: left to itself the compiler spills
                        asm volatile("" : "+v"(tot[r][t]));
                        if ((i & 1) + j == 2) acc[r][t] += widen(tot[r][t]);
                    }
                }
            }
        }
    } else {
        f4 big[NG][TT], small[NG][TT];
#pragma unroll
        for (int r = 0; r < NG; r++)
#pragma unroll
            for (int t = 0; t < TT; t++) big[r][t] = small[r][t] = zero;
        uint32_t q[NG][8], hb[NG][8];
        h2 sc[NG][4], sb[NG][4];
#pragma unroll
        for (int r = 0; r < NG; r++) {
            if constexpr (T == T_Q6_K) {
                const auto &u = w[r];
                const int h = g & 1;
                u4v_to(u.p0, q[r]);
                u4v_to(u.p1, q[r] + 4);
                u4v_to(u.qh, hb[r]);
                sc[r][0] = dup_h2((float)(int8_t)(u.sc.x >> (8 * h)));
                sc[r][1] = dup_h2((float)(int8_t)(u.sc.x >> (8 * h + 16)));
                sc[r][2] = dup_h2((float)(int8_t)(u.sc.y >> (8 * h)));
                sc[r][3] = dup_h2((float)(int8_t)(u.sc.y >> (8 * h + 16)));
            } else {
                const auto &u = w[r];
                u4v_to(u.q0, q[r]);
                u4v_to(u.q1, q[r] + 4);
                if constexpr (T == T_Q5_K) {
                    u4v_to(u.h0, hb[r]);
                    u4v_to(u.h1, hb[r] + 4);
                }
                // scales of sub-blocks 2 g and 2 g + 1
                const uint32_t lo = u.hd.y & 0x3F3F3F3Fu;
                const uint32_t hi = (u.hd.w & 0x0F0F0F0Fu) | ((u.hd.y >> 2) & 0x30303030u);
                const uint32_t s2 = (g < 2 ? lo : hi) >> (16 * (g & 1));
                const float s0 = (float)(s2 & 255u), s1 = (float)((s2 >> 8) & 255u);
                sc[r][0] = dup_h2(s0), sc[r][1] = dup_h2(s1);
                sb[r][0] = dup_h2(-1024.0f * s0), sb[r][1] = dup_h2(-1024.0f * s1);
            }
        }
#pragma unroll
        for (int s = 0; s < 8; s++) {
            h8 op[NG], rem[NG];
#pragma unroll
            for (int r = 0; r < NG; r++) {
                uint32_t v[2];
                h2 e[4];
                if constexpr (T == T_Q6_K) {
                    const int run = s >> 1, half = s & 1;
#pragma unroll
                    for (int j = 0; j < 2; j++) {
                        const int i = 2 * half + j;
                        const uint32_t p = q[r][4 * (run & 1) + i], h = hb[r][i];
                        v[j] = (run < 2 ? p & 0x0F0F0F0Fu : (p >> 4) & 0x0F0F0F0Fu) |
                               ((run == 0 ? h << 4 : run == 1 ? h << 2 : run == 2 ? h : h >> 2) & 0x30303030u);
                    }
                    bytes_1024(v[0], e[0], e[1]);
                    bytes_1024(v[1], e[2], e[3]);
                    h2 o[4], m[4];
#pragma unroll
                    for (int j = 0; j < 4; j++) {
                        const h2 c = e[j] + dup_h2(-1056.0f);  // 1024 + q - (1024 + 32)
                        o[j] = c * sc[r][run];
                        m[j] = __builtin_elementwise_fma(c, sc[r][run], -o[j]);  // exact
                    }
                    op[r] = cat8(o[0], o[1], o[2], o[3]);
                    rem[r] = cat8(m[0], m[1], m[2], m[3]);
                } else {
                    const int hi = s >> 2, i0 = 2 * (s & 3);
#pragma unroll
                    for (int j = 0; j < 2; j++) {
                        v[j] = (hi ? q[r][i0 + j] >> 4 : q[r][i0 + j]) & 0x0F0F0F0Fu;
                        if constexpr (T == T_Q5_K)
                            v[j] |= ((hb[r][i0 + j] >> (2 * g + hi)) & 0x01010101u) << 4;
                    }
                    bytes_1024(v[0], e[0], e[1]);
                    bytes_1024(v[1], e[2], e[3]);
                    // (1024 + q) s - 1024 s, one rounding of an exact value
#pragma unroll
                    for (int j = 0; j < 4; j++) e[j] = __builtin_elementwise_fma(e[j], sc[r][hi], sb[r][hi]);
                    op[r] = cat8(e[0], e[1], e[2], e[3]);
                }
            }
#pragma unroll
            for (int t = 0; t < TT; t++) {
                const h8 x1 = xop(t, 0, s), x2 = xop(t, 1, s), x3 = xop(t, 2, s);
#pragma unroll
                for (int r = 0; r < NG; r++) {
                    big[r][t] = mm(x1, op[r], big[r][t]);
                    small[r][t] = mm(x3, op[r], small[r][t]);
                    small[r][t] = mm(x2, op[r], small[r][t]);
                    if constexpr (T == T_Q6_K) small[r][t] = mm(x1, rem[r], mm(x2, rem[r], small[r][t]));
                }
            }
            if (s & 1) __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int r = 0; r < NG; r++) {
            if constexpr (T == T_Q6_K) {
                const double d = f16f(w[r].d);
#pragma unroll
                for (int t = 0; t < TT; t++) acc[r][t] += d * widen(big[r][t] + small[r][t]);
            } else {
                // minimum terms: sum_j m_j s_j of the 8 sub-blocks, the third
                // to first pieces of s_j in lane groups 0..2 (group 3
                // multiplies zeros); the first, exactly, and the other two
                // summed apart
                const uint32_t z = w[r].hd.z, hw = w[r].hd.w;
                h2 e[4];
                bytes_1024(z & 0x3F3F3F3Fu, e[0], e[1]);
                bytes_1024(((hw >> 4) & 0x0F0F0F0Fu) | ((z >> 2) & 0x30303030u), e[2], e[3]);
                const h2 off = dup_h2(-1024.0f);
                const h8 mv = cat8(e[0] + off, e[1] + off, e[2] + off, e[3] + off);
                const h8 mz = {}, mhi = g < 2 ? mz : mv, mlo = g < 2 ? mv : mz;
                const double d = f16f(w[r].hd.x), dm = -64.0 * f16f(w[r].hd.x >> 16);
#pragma unroll
                for (int t = 0; t < TT; t++) {
                    const h8 sx = sop(t);
                    const f4 mn = mm(sx, mhi, zero) + mm(sx, mlo, zero);
                    acc[r][t] += d * widen(big[r][t] + small[r][t]);
                    acc[r][t] += dm * widen(mn);
                }
            }
        }
    }
}

// Y[pos][r] = sum_c W[r][c] x[row(pos)][c] for a tile of 16 TT positions and
// 16 NG rows per wave of a workgroup of NW, the activation pieces of a
// step in LDS (shared by the waves), each wave's weights in its registers
// one step ahead.  With tiles, tile i holds positions [start, start + count)
// of one expert (its slab) and row(pos) = order[pos] / xdiv or pos; without,
// positions are the T rows of one or more dense matrices.
//
// Bound: the weight stream while an expert has few tokens, the matrix cores
// (three or four f16 products per value) beyond; 16 TT = 32 tokens keeps an
// expert's tile near the 24 tokens an expert meets in 384-token prompts at
// k / E = 8 / 128 and two workgroups on a CU (the second launch bound, in
// waves per SIMD).  At 383 tokens of the 30B-A3B shape: q/k/v (5120 x 2048
// q8_0) 49 us, o-proj (2048 x 4096) 59, gate (q4_K) 85, up (q5_K) 104, down
// (q6_K) 100 us for 417 MB of slabs; a 384-token prompt through two such
// layers took 50.7 ms token by token and takes 1.0 ms (with two generated
// tokens), the batch itself 0.53 ms.
template <int T, bool D8, int TT, int NG, int NW>
__global__ void __launch_bounds__(64 * NW, NW / 2) k_prompt_gemm(PromptGemm a)
{
    constexpr int TM = 16 * TT, XT = 2 * NW, XR = TM / XT;  // rows staged per pass, passes
    static_assert(TM % XT == 0, "whole passes");
    __shared__ __align__(16) uint8_t s_x[3 * TM * XROW];
    __shared__ __align__(16) uint8_t s_sum[TM * 64];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, n = lane & 15, g = lane >> 4;
    // consecutive workgroups go to the 8 XCDs in turn: an expert's row tiles
    // stay on one XCD (they share its tokens' pieces in that L2), a dense
    // row tile's token tiles likewise (they share its weights)
    const int bid = blockIdx.x, xcd = bid & 7, j = bid >> 3;
    int tile, rt;
    if (a.tiles) {
        tile = xcd + 8 * (j / a.nrt);
        rt = j % a.nrt;
        if (tile >= *a.ntiles) return;
    } else {
        const int nx = (a.nrt + 7) / 8;
        rt = xcd + 8 * (j % nx);
        tile = j / nx;
        if (rt >= a.nrt) return;
    }
    int seg = 0;
    while (seg + 1 < a.nseg && rt >= a.rt0[seg + 1]) seg++;
    rt -= a.rt0[seg];
    const int rows = a.rows[seg];
    int start = tile * TM, count = min(TM, a.T - start);
    const uint8_t *base = a.w[seg];
    if (a.tiles) {
        const int4 ti = a.tiles[tile];
        start = ti.y;
        count = ti.z;
        const uint32_t h = a.remap ? a.remap[ti.x] : (uint32_t)ti.x;
        const ExpSrc &e = a.src[seg];
        if (h != SKIP)
            base = e.hot + (int64_t)h * e.hot_slab;
        else if (const int c = a.stage ? a.cold_slot[ti.x] : a.stage_slots; c < a.stage_slots)
            base = a.stage + (int64_t)c * e.gtt_slab;
        else
            base = e.gtt + (int64_t)ti.x * e.gtt_slab;
    }
    auto xrow = [&](int i) {  // activation row of position start + i (clamped to the tile)
        const int p = start + min(i, count - 1);
        return a.order ? a.order[p] / a.xdiv : p;
    };
    const int nb = a.x.n / blk_elems(T), nc = a.x.np / KC;
    const Split sl = split_of(T);
    const int64_t nblk = (int64_t)rows * nb;
    const Buf m(base, nblk * blk_bytes(T));
    const Reg ro{(uint32_t)region_off(sl, 1, nblk), (uint32_t)region_off(sl, 2, nblk),
                 (uint32_t)region_off(sl, 3, nblk)};
    const int r0 = (rt * NW + wave) * 16 * NG;
    PW<T, D8> w[NG];
    auto wload = [&](int c) {
#pragma unroll
        for (int r = 0; r < NG; r++) w[r].load(m, ro, min(r0 + 16 * r + n, rows - 1), nb, c, g);
    };
    // this thread's 16-byte columns of XR rows of each piece
    uint32_t xo[XR];
#pragma unroll
    for (int i = 0; i < XR; i++) xo[i] = (uint32_t)xrow((tid >> 5) + XT * i) * a.x.np * 2 + (tid & 31) * 16;
    const int64_t plane = a.x.rows * (int64_t)a.x.np * 2;
    const Buf xb[3] = {{a.x.p, plane}, {(const uint8_t *)a.x.p + plane, plane}, {(const uint8_t *)a.x.p + 2 * plane, plane}};
    const Buf sb(a.x.sums, a.x.rows * nc * 64);
    const uint32_t so = (uint32_t)xrow(tid >> 2) * nc * 64 + (tid & 3) * 16;
    styx_u4 xr[3 * XR], sr;
    auto xload = [&](int c) {
#pragma unroll
        for (int p = 0; p < 3; p++)
#pragma unroll
            for (int i = 0; i < XR; i++) xr[p * XR + i] = xb[p].b128(xo[i], c * KC * 2);
        if (T == T_Q4_K || T == T_Q5_K)
            if (tid < TM * 4) sr = sb.b128(so, c * 64);
    };
    d4 acc[NG][TT];
#pragma unroll
    for (int r = 0; r < NG; r++)
#pragma unroll
        for (int t = 0; t < TT; t++) acc[r][t] = d4{0.0, 0.0, 0.0, 0.0};
    xload(0);
    wload(0);
    for (int c = 0; c < nc; c++) {
        __syncthreads();
#pragma unroll
        for (int p = 0; p < 3; p++)
#pragma unroll
            for (int i = 0; i < XR; i++)
                *(styx_u4 *)(s_x + (p * TM + (tid >> 5) + XT * i) * XROW + (tid & 31) * 16) = xr[p * XR + i];
        if (T == T_Q4_K || T == T_Q5_K)
            if (tid < TM * 4) *(styx_u4 *)(s_sum + tid * 16) = sr;
        __syncthreads();
        PW<T, D8> wc[NG];
#pragma unroll
        for (int r = 0; r < NG; r++) wc[r] = w[r];
        // (the activations first: loads return in order, and the LDS stores
        // of the next step then leave its weights in flight)
        if (c + 1 < nc) {
            xload(c + 1);
            wload(c + 1);
        }
        gemm_step<T, D8, NG, TT>(
            wc,
            [&](int t, int p, int s) {
                return *(const h8 *)(s_x + (p * TM + 16 * t + n) * XROW + 16 * x_run<T>(g, s));
            },
            [&](int t) { return *(const h8 *)(s_sum + (16 * t + n) * 64 + 16 * g); }, acc);
    }
#pragma unroll
    for (int t = 0; t < TT; t++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int p = 16 * t + 4 * g + i;
            if (p >= count) continue;
            const float sc = a.x.scale[xrow(p)];
#pragma unroll
            for (int r = 0; r < NG; r++) {
                const int row = r0 + 16 * r + n;
                if (row >= rows) continue;
                float *y = a.y[seg] + (int64_t)(start + p) * rows + row;
                const float v = (float)acc[r][t][i] * sc;
                *y = a.add ? *y + v : v;
            }
        }
}

// The same for a dense matrix and at most 32 positions, 16 rows per
// workgroup: each wave takes every fourth step of the columns with its
// activations straight from the L2, and the waves' sums meet in LDS.  A
// workgroup of the kernel above walks all steps in turn, each a memory round
// trip of about 3 us while few workgroups share a CU: q8_0 q/k/v (5120 x
// 2048) 26 us at up to 32 tokens, here 14 up to 16 and 25 above; o-proj
// (2048 x 4096) 48, here 15 and 27.  From 33 tokens on the
// activations' L2 traffic (every workgroup reads them all) outweighs it.
template <int T, bool D8, int TT> __global__ void __launch_bounds__(PWG, 2) k_prompt_gemm_few(PromptGemm a)
{
    __shared__ d4 s_acc[4][TT][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, n = lane & 15, g = lane >> 4;
    int rt = blockIdx.x, seg = 0;
    while (seg + 1 < a.nseg && rt >= a.rt0[seg + 1]) seg++;
    rt -= a.rt0[seg];
    const int rows = a.rows[seg], nb = a.x.n / blk_elems(T), nc = a.x.np / KC;
    const Split sl = split_of(T);
    const int64_t nblk = (int64_t)rows * nb;
    const Buf m(a.w[seg], nblk * blk_bytes(T));
    const Reg ro{(uint32_t)region_off(sl, 1, nblk), (uint32_t)region_off(sl, 2, nblk),
                 (uint32_t)region_off(sl, 3, nblk)};
    const int64_t plane = a.x.rows * (int64_t)a.x.np * 2;
    const Buf xb[3] = {{a.x.p, plane}, {(const uint8_t *)a.x.p + plane, plane}, {(const uint8_t *)a.x.p + 2 * plane, plane}};
    const Buf sb(a.x.sums, a.x.rows * nc * 64);
    uint32_t xo[TT], so[TT];
#pragma unroll
    for (int t = 0; t < TT; t++) {
        const uint32_t row = min(16 * t + n, a.T - 1);
        xo[t] = row * a.x.np * 2;
        so[t] = row * nc * 64 + 16 * g;
    }
    const uint32_t row = min(rt * 16 + n, rows - 1);
    // (the sums stay in LDS between steps: the step's loads need the registers)
#pragma unroll
    for (int t = 0; t < TT; t++) s_acc[wave][t][lane] = d4{0.0, 0.0, 0.0, 0.0};
    for (int c = wave; c < nc; c += 4) {
        // every load of the step before any product: one round trip a step
        PW<T, D8> w[1];
        w[0].load(m, ro, row, nb, c, g);
        styx_u4 x[TT][3][8], xs[TT];
#pragma unroll
        for (int t = 0; t < TT; t++) {
#pragma unroll
            for (int s = 0; s < 8; s++)
#pragma unroll
                for (int p = 0; p < 3; p++) x[t][p][s] = xb[p].b128(xo[t] + 16 * x_run<T>(g, s), c * KC * 2);
            if (T == T_Q4_K || T == T_Q5_K) xs[t] = sb.b128(so[t], c * 64);
        }
        __builtin_amdgcn_sched_barrier(0);
        d4 acc[1][TT];
#pragma unroll
        for (int t = 0; t < TT; t++) acc[0][t] = d4{0.0, 0.0, 0.0, 0.0};
        gemm_step<T, D8, 1, TT>(
            w, [&](int t, int p, int s) { return __builtin_bit_cast(h8, x[t][p][s]); },
            [&](int t) { return __builtin_bit_cast(h8, xs[t]); }, acc);
#pragma unroll
        for (int t = 0; t < TT; t++) s_acc[wave][t][lane] += acc[0][t];
    }
    __syncthreads();
    if (wave >= TT) return;
    const int t = wave;
    const d4 v = (s_acc[0][t][lane] + s_acc[1][t][lane]) + (s_acc[2][t][lane] + s_acc[3][t][lane]);
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int p = 16 * t + 4 * g + i;
        if (p >= a.T || rt * 16 + n >= rows) continue;
        float *y = a.y[seg] + (int64_t)p * rows + rt * 16 + n;
        const float r = (float)v[i] * a.x.scale[p];
        *y = a.add ? *y + r : r;
    }
}

template <int T, bool D8> static hipError_t gemm_few(hipStream_t st, PromptGemm &a)
{
    a.nrt = 0;
    for (int s = 0; s < a.nseg; s++) {
        a.rt0[s] = a.nrt;
        a.nrt += (a.rows[s] + 15) / 16;
    }
    if (a.T <= 16)
        hipLaunchKernelGGL((k_prompt_gemm_few<T, D8, 1>), dim3(a.nrt), dim3(PWG), 0, st, a);
    else
        hipLaunchKernelGGL((k_prompt_gemm_few<T, D8, 2>), dim3(a.nrt), dim3(PWG), 0, st, a);
    return hipGetLastError();
}

template <int T, bool D8, int TT, int NG, int NW> static hipError_t gemm_go(hipStream_t st, PromptGemm &a)
{
    a.nrt = 0;
    for (int s = 0; s < a.nseg; s++) {
        a.rt0[s] = a.nrt;
        a.nrt += (a.rows[s] + 16 * NW * NG - 1) / (16 * NW * NG);
    }
    a.ntt = (a.T + 16 * TT - 1) / (16 * TT);
    const int64_t n = a.tiles ? (int64_t)((a.max_tiles + 7) / 8 * 8) * a.nrt
                              : (int64_t)((a.nrt + 7) / 8 * 8) * a.ntt;
    if (n > 0x7FFFFFFF) return hipErrorInvalidValue;
    hipLaunchKernelGGL((k_prompt_gemm<T, D8, TT, NG, NW>), dim3((unsigned)n), dim3(64 * NW), 0, st, a);
    return hipGetLastError();
}

template <int T, bool D8 = true> static hipError_t gemm_t(hipStream_t st, PromptGemm &a)
{
    // 32 positions a tile unless 16 hold them all; eight waves of 16 rows
    // unless that would leave CUs without a workgroup, then four.  q4_K and
    // q5_K take four waves of two row tiles each (half the LDS reads per
    // product): the gate slabs (q4_K) of 383 tokens of the 30B-A3B shape 87
    // us, 93 with eight waves, whose 128 registers do not hold q5_K's
    // unpacking at all (24 spilled).  q6_K: 92 that way, 89 with eight.
    const int64_t rows = (int64_t)a.rows[0] + (a.nseg > 1 ? a.rows[1] : 0) + (a.nseg > 2 ? a.rows[2] : 0);
    if (!a.tiles && a.T <= 32) return gemm_few<T, D8>(st, a);
    const int tm = a.tile_tokens;
    const int64_t wg = (rows + 127) / 128 * (a.tiles ? a.max_tiles : (a.T + tm - 1) / tm);
    if (tm == 16) return wg < 256 ? gemm_go<T, D8, 1, 1, 4>(st, a) : gemm_go<T, D8, 1, 1, 8>(st, a);
    if (wg < 256) return gemm_go<T, D8, 2, 1, 4>(st, a);
    if constexpr (T == T_Q4_K || T == T_Q5_K) return gemm_go<T, D8, 2, 2, 4>(st, a);
    return gemm_go<T, D8, 2, 1, 8>(st, a);
}

hipError_t launch_prompt_gemm(hipStream_t st, int t, PromptGemm a)
{
    if (a.nseg < 1 || a.nseg > 3 || a.T < 1 || a.x.n % blk_elems(t) ||
        (a.tile_tokens != 16 && a.tile_tokens != 32) || (a.order && a.xdiv < 1) ||
        (a.tiles && (!a.ntiles || a.max_tiles < 1)))
        return hipErrorInvalidValue;
    // byte offsets into a matrix and into a piece of the rows are 32-bit
    for (int s = 0; s < a.nseg; s++)
        if (a.rows[s] < 1 || (int64_t)a.rows[s] * (a.x.n / blk_elems(t)) * blk_bytes(t) > 0x7FFFFFFF)
            return hipErrorInvalidValue;
    if (a.x.rows * (int64_t)a.x.np * 2 > 0x7FFFFFFF) return hipErrorInvalidValue;
    switch (t) {
    case T_Q8_0: return a.x.n % 256 ? gemm_t<T_Q8_0, false>(st, a) : gemm_t<T_Q8_0>(st, a);
    case T_Q4_K: return gemm_t<T_Q4_K>(st, a);
    case T_Q5_K: return gemm_t<T_Q5_K>(st, a);
    case T_Q6_K: return gemm_t<T_Q6_K>(st, a);
    default: return hipErrorInvalidValue;
    }
}

// ------------------------------------------------------- rope, K/V rows ----
// One workgroup per token: its q heads normalised and rotated in place, its
// k heads into the K cache, its v heads into the V cache; *odd set if one of
// their values is not finite.
template <int PPL> __global__ void __launch_bounds__(PWG) k_prompt_rope(PromptAttn a)
{
    const int t = blockIdx.x, pos = a.pos0 + t, wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    double2 cs[PPL];
    cs_load<PPL>(cs, a.rope + (int64_t)pos * (a.hd / 2), a.hd);
    const int64_t pg = a.page_table[pos / a.page_tokens];
    const int tp = pos % a.page_tokens;
    auto at = [&](int h) { return ((pg * a.nkv + h) * a.page_tokens + tp) * (int64_t)a.hd; };
    for (int h = wave; h < (a.q ? a.nh : 0); h += 4) {
        float *q = a.q + ((int64_t)t * a.nh + h) * a.hd;
        HeadIn<PPL> in;
        head_load<PPL>(in, q, a.q_norm, a.hd);
        head_finish<PPL>(in, cs, a.q_norm != nullptr, a.eps, a.hd, q);
    }
    for (int h = wave; h < a.nkv; h += 4) {
        const int64_t o = ((int64_t)t * a.nkv + h) * a.hd;
        HeadIn<PPL> in;
        head_load<PPL>(in, a.k + o, a.k_norm, a.hd);
        head_finish<PPL>(in, cs, a.k_norm != nullptr, a.eps, a.hd, a.kpool + at(h));
        for (int i = lane; i < a.hd; i += 64) {
            const float v = a.v[o + i];
            a.vpool[at(h) + i] = v;
            if (!(fabsf(v) < INFINITY)) *a.odd = 1;
        }
    }
}

// ------------------------------------------------------------ attention ----
// Causal attention of T tokens at positions pos0.. over cached keys: a
// workgroup takes 16 query rows (token, head) of one kv head and a chunk of
// the keys (blockIdx.z); its four waves take every fourth block of 32 keys,
// each with its own online softmax (attn16.h), and merge in LDS.  With more
// than one chunk the results are partials, merged by launch_attn_merge: few
// tokens over a long context make few row tiles, whose waves each walk a
// quarter of the keys in turn.  A prompt of five tokens after 32000 keys
// through four layers of the 30B-A3B shape took 7.5 ms unsplit (2.8 ms token
// by token), so 1.2; after 4000 keys 1.31, 1.31 and 0.77 ms.
//
// The matrix products give every query of a tile every V row up to the
// largest key met, those it does not see times 0.  Where the batch wrote a V
// value that is not finite (a.odd), 0 times it would put NaN into the tokens
// before it: each query is then taken by a wave of its own, over the keys it
// sees only (prompt_attn_rows).
__device__ __forceinline__ void prompt_attn_emit(const PromptAttn &a, int HD, int64_t o, int d, float O, float L, float M)
{
    if (gridDim.z == 1) {
        a.out[o * HD + d] = O / L;
        return;
    }
    float *p = a.part + (o * gridDim.z + blockIdx.z) * (HD + 2);
    p[2 + d] = O;
    if (d == 0) p[0] = M, p[1] = L;
}

template <int HD> __device__ __forceinline__ void prompt_attn_rows(const PromptAttn &a)
{
    const int lane = threadIdx.x & 63, gqa = a.nh / a.nkv, kvh = blockIdx.y, r0 = blockIdx.x * 16;
    const int r1 = min(r0 + 16, a.T * gqa), c0 = blockIdx.z * a.chunk;
    auto row_at = [&](int key) {
        return (((int64_t)a.page_table[key / a.page_tokens] * a.nkv + kvh) * a.page_tokens + key % a.page_tokens) * HD;
    };
    for (int r = r0 + (threadIdx.x >> 6); r < r1; r += PWG / 64) {
        const int64_t oi = (int64_t)(r / gqa) * a.nh + kvh * gqa + r % gqa;
        const int last = min(a.pos0 + r / gqa, c0 + a.chunk - 1);
        const float *q = a.q + oi * HD;
        float m = -INFINITY, l = 0.0f, o[HD / 64] = {};
        for (int k0 = c0; k0 <= last; k0 += 64) {
            const float *kp = a.kpool + row_at(min(k0 + lane, last));
            float s = 0.0f;
#pragma unroll 2
            for (int d = 0; d < HD; d += 4) {
                const f4 x = ld4(q + d), k = ld4(kp + d);
                s += (x.x * k.x + x.y * k.y) + (x.z * k.z + x.w * k.w);
            }
            s = k0 + lane <= last ? s * a.scale : -INFINITY;
            const float mn = fmaxf(m, wave_max(s)), mz = mn == -INFINITY ? 0.0f : mn;
            const float corr = expf(m - mz), p = expf(s - mz);
            m = mn;
            l = l * corr + wave_sum(p);
#pragma unroll
            for (int i = 0; i < HD / 64; i++) o[i] *= corr;
            for (int j = 0; j < min(64, last - k0 + 1); j++) {
                const float *vp = a.vpool + row_at(k0 + j) + lane;
                const float pj = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(p), j));
#pragma unroll
                for (int i = 0; i < HD / 64; i++) o[i] += pj * vp[64 * i];
            }
        }
#pragma unroll
        for (int i = 0; i < HD / 64; i++) prompt_attn_emit(a, HD, oi, lane + 64 * i, o[i], l, m);
    }
}

template <int HD> __global__ void __launch_bounds__(PWG) k_prompt_attn(PromptAttn a)
{
    __shared__ __align__(16) Merge16<HD> s;
    if (*a.odd) {
        prompt_attn_rows<HD>(a);
        return;
    }
    const int wave = threadIdx.x >> 6, n = threadIdx.x & 15;
    const int gqa = a.nh / a.nkv, kvh = blockIdx.y, nrow = a.T * gqa, r0 = blockIdx.x * 16;
    const int row = min(r0 + n, nrow - 1);
    const int tok = row / gqa, head = kvh * gqa + row % gqa, qpos = a.pos0 + tok;
    const int c0 = blockIdx.z * a.chunk;
    // largest key met
    const int last = min(a.pos0 + min(r0 + 15, nrow - 1) / gqa, c0 + a.chunk - 1);
    Attn16<HD> at;
    at.init(a.q + ((int64_t)tok * a.nh + head) * HD);
    for (int k0 = c0 + wave * A16_KB; k0 <= last; k0 += 4 * A16_KB) {
        // page_tokens is a multiple of A16_KB: a key block lies in one page
        const int64_t pg = a.page_table[k0 / a.page_tokens];
        const int64_t base = ((pg * a.nkv + kvh) * a.page_tokens + k0 % a.page_tokens) * (int64_t)HD;
        at.block(a.kpool + base, a.vpool + base, HD, last - k0, qpos - k0 + 1, a.scale);
    }
    attn16_merge<HD>(at, s, [&](int r, int d, float O, float L, float M) {
        const int qr = r0 + r;
        if (qr >= nrow) return;
        prompt_attn_emit(a, HD, (int64_t)(qr / gqa) * a.nh + kvh * gqa + qr % gqa, d, O, L, M);
    });
}

static bool attn_ok(const PromptAttn &a)
{
    return a.odd && a.T >= 1 && a.nkv >= 1 && a.nh >= a.nkv && a.nh % a.nkv == 0 && a.pos0 >= 0 &&
           (a.hd == 64 || a.hd == 128 || a.hd == 256) && a.page_tokens >= A16_KB && a.page_tokens % A16_KB == 0;
}

hipError_t launch_prompt_rope(hipStream_t st, const PromptAttn &a)
{
    if (!attn_ok(a)) return hipErrorInvalidValue;
    if (a.hd == 256)
        hipLaunchKernelGGL(k_prompt_rope<2>, dim3(a.T), dim3(PWG), 0, st, a);
    else
        hipLaunchKernelGGL(k_prompt_rope<1>, dim3(a.T), dim3(PWG), 0, st, a);
    return hipGetLastError();
}

hipError_t launch_prompt_attn(hipStream_t st, PromptAttn a)
{
    if (!attn_ok(a) || !a.q || !a.out) return hipErrorInvalidValue;
    const int tiles = (a.T * (a.nh / a.nkv) + 15) / 16, n_t = a.pos0 + a.T;
    a.chunk = (int)attn_chunk_keys(n_t, (uint64_t)tiles * a.nkv, (uint64_t)a.T * a.nh, a.hd, a.part ? a.part_floats : 0);
    const int chunks = (n_t + a.chunk - 1) / a.chunk;
    const dim3 grid(tiles, a.nkv, chunks);
    switch (a.hd) {
    case 64: hipLaunchKernelGGL(k_prompt_attn<64>, grid, dim3(PWG), 0, st, a); break;
    case 128: hipLaunchKernelGGL(k_prompt_attn<128>, grid, dim3(PWG), 0, st, a); break;
    default: hipLaunchKernelGGL(k_prompt_attn<256>, grid, dim3(PWG), 0, st, a); break;
    }
    if (chunks > 1) return launch_attn_merge(st, a.part, a.out, a.T * a.nh, chunks, a.hd);
    return hipGetLastError();
}

// --------------------------------------------------------------- router ----
// logits[t][e] = W[e] . xn[t] (+ bias) in f32 (matvec_strided_f32.comp): 16
// tokens x 16 experts per workgroup, the four waves a quarter of the columns
// each, four accumulators per wave.
__global__ void __launch_bounds__(PWG) k_prompt_router(const float *xn, const float *W,
                                                       const float *bias, float *logits, int T,
                                                       int E, int H)
{
    __shared__ float part[4][16][16];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, n = lane & 15, g = lane >> 4;
    const int t0 = blockIdx.x * 16, e0 = blockIdx.y * 16, q = H / 4;
    const float *xp = xn + (int64_t)min(t0 + n, T - 1) * H + wave * q + 4 * g;
    const float *wp = W + (int64_t)min(e0 + n, E - 1) * H + wave * q + 4 * g;
    const f4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
    d4 tot = {0.0, 0.0, 0.0, 0.0};
    // 64 columns' products summed in f32, those sums in f64
    for (int i = 0; i < q; i += 64) {
        f4 acc[4] = {zero, zero, zero, zero};
#pragma unroll
        for (int j = 0; j < 64; j += 16) {
            const f4 x = *(const f4 *)(xp + i + j), w = *(const f4 *)(wp + i + j);
#pragma unroll
            for (int e = 0; e < 4; e++)
                acc[e] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[e], w[e], acc[e], 0, 0, 0);
        }
        tot += __builtin_convertvector((acc[0] + acc[1]) + (acc[2] + acc[3]), d4);
    }
#pragma unroll
    for (int i = 0; i < 4; i++) part[wave][4 * g + i][n] = (float)tot[i];
    __syncthreads();
    const int t = threadIdx.x >> 4, e = threadIdx.x & 15;
    if (t0 + t >= T || e0 + e >= E) return;
    const float v = (part[0][t][e] + part[1][t][e]) + (part[2][t][e] + part[3][t][e]);
    logits[(int64_t)(t0 + t) * E + e0 + e] = bias ? v + bias[e0 + e] : v;
}

__global__ void __launch_bounds__(64) k_prompt_topk(const float *logits, int E, int k, int renorm,
                                                    float *wts, int32_t *ids)
{
    const int64_t t = blockIdx.x;
    topk_wave(logits + t * E, E, k, renorm, nullptr, nullptr, 0, 0, wts + t * MAX_TOPK, ids + t * IDS_ROW);
}

// The (token, slot) pairs p = token k + slot grouped by expert: order lists
// them, inv[p] is p's place there (-1: no such expert), tiles the runs of at
// most tm places of one expert.
constexpr int PLAN_WG = 1024;
__global__ void __launch_bounds__(PLAN_WG) k_prompt_plan(const int32_t *ids, int T, int k, int E,
                                                         int tm, int *order, int *inv, int4 *tiles,
                                                         int *ntiles, const uint32_t *remap,
                                                         int *cold_slot, int *cold_list, int *ncold)
{
    __shared__ int cnt[MAX_EXPERTS], off[MAX_EXPERTS], til[MAX_EXPERTS], cold[MAX_EXPERTS];
    const int tid = threadIdx.x;
    if (tid < MAX_EXPERTS) cnt[tid] = 0;
    __syncthreads();
    for (int p = tid; p < T * k; p += PLAN_WG) {
        const uint32_t e = (uint32_t)ids[(int64_t)(p / k) * IDS_ROW + p % k];
        if (e < (uint32_t)E) atomicAdd(&cnt[e], 1);
    }
    __syncthreads();
    // inclusive scans of the counts, of the tiles they make and of the met
    // experts that are not in HBM
    int c = 0, t = 0, host = 0;
    if (tid < MAX_EXPERTS) {
        off[tid] = c = cnt[tid];
        til[tid] = t = (c + tm - 1) / tm;
        cold[tid] = host = remap && c > 0 && remap[tid] == SKIP;
    }
    __syncthreads();
    for (int d = 1; d < MAX_EXPERTS; d *= 2) {
        int a = 0, b = 0, h = 0;
        if (tid < MAX_EXPERTS && tid >= d) a = off[tid - d], b = til[tid - d], h = cold[tid - d];
        __syncthreads();
        if (tid < MAX_EXPERTS) off[tid] += a, til[tid] += b, cold[tid] += h;
        __syncthreads();
    }
    if (host) {
        cold_slot[tid] = cold[tid] - 1;
        cold_list[cold[tid] - 1] = tid;
    }
    if (remap && tid == 0) *ncold = cold[MAX_EXPERTS - 1];
    if (tid < MAX_EXPERTS) {
        const int o = off[tid] - c, i0 = til[tid] - t;
        for (int i = 0; i < t; i++) tiles[i0 + i] = make_int4(tid, o + i * tm, min(tm, c - i * tm), 0);
        if (tid == MAX_EXPERTS - 1) *ntiles = til[tid];
        cnt[tid] = o;  // the expert's next free place
    }
    __syncthreads();
    for (int p = tid; p < T * k; p += PLAN_WG) {
        const uint32_t e = (uint32_t)ids[(int64_t)(p / k) * IDS_ROW + p % k];
        int at = -1;
        if (e < (uint32_t)E) {
            at = atomicAdd(&cnt[e], 1);
            order[at] = p;
        }
        inv[p] = at;
    }
}

// Slabs of the first `slots` cold experts from pinned host memory to the
// staging buffer: blockIdx.y the slot, 64 KiB per workgroup, four 16-byte
// loads in flight per thread.  The GEMM's own loads of host memory (64-byte
// pieces of 16 rows) reach about half the link's rate, these 52 GB/s: a
// 96-token prompt with half of the experts cold (about 55 slabs of each
// matrix) 6.7 -> 4.0 ms.
constexpr int64_t STAGE_CHUNK = 64 * 1024;
__global__ void __launch_bounds__(PWG) k_prompt_stage(const int *list, const int *ncold, const uint8_t *src,
                                                      int64_t slab, uint8_t *dst)
{
    const int s = blockIdx.y;
    if (s >= *ncold) return;
    const styx_u4 *p = (const styx_u4 *)(src + (int64_t)list[s] * slab);
    styx_u4 *q = (styx_u4 *)(dst + (int64_t)s * slab);
    const int64_t c0 = blockIdx.x * (STAGE_CHUNK / 16), c1 = min(slab / 16, c0 + STAGE_CHUNK / 16);
    int64_t i = c0 + threadIdx.x;
    for (; i + 3 * PWG < c1; i += 4 * PWG) {
        const styx_u4 a = p[i], b = p[i + PWG], c = p[i + 2 * PWG], d = p[i + 3 * PWG];
        q[i] = a, q[i + PWG] = b, q[i + 2 * PWG] = c, q[i + 3 * PWG] = d;
    }
    for (; i < c1; i += PWG) q[i] = p[i];
}

hipError_t launch_prompt_stage(hipStream_t st, const int *list, const int *ncold, const uint8_t *src,
                               int64_t slab, uint8_t *dst, int slots)
{
    if (slab < 16 || slab % 16 || slots < 1) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_prompt_stage, dim3((unsigned)((slab + STAGE_CHUNK - 1) / STAGE_CHUNK), slots),
                       dim3(PWG), 0, st, list, ncold, src, slab, dst);
    return hipGetLastError();
}

hipError_t launch_prompt_route(hipStream_t st, const PromptRoute &a)
{
    if (a.T < 1 || a.E < a.k || a.E > MAX_EXPERTS || a.k < 1 || a.k > MAX_TOPK || a.H % 256)
        return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_prompt_router, dim3((a.T + 15) / 16, (a.E + 15) / 16), dim3(PWG), 0, st, a.xn,
                       a.W, a.bias, a.logits, a.T, a.E, a.H);
    hipLaunchKernelGGL(k_prompt_topk, dim3(a.T), dim3(64), 0, st, a.logits, a.E, a.k, a.renorm, a.wts,
                       a.ids);
    hipLaunchKernelGGL(k_prompt_plan, dim3(1), dim3(PLAN_WG), 0, st, a.ids, a.T, a.k, a.E, a.tile_tokens,
                       a.order, a.inv, a.tiles, a.ntiles, a.remap, a.cold_slot, a.cold_list, a.ncold);
    return hipGetLastError();
}

}  // namespace styx
