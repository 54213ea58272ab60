// kernels_ref.hip -- kernels with the reference pipelines' exact interface,
// for the generic dispatch path (styx_batch_dispatch).  Each takes the
// bindings and push-constant block of the shader or vendored kernel it
// stands in for, with the same workgroup grid.  Quant weights are read in
// GGUF block layout, as the reference uploads them.
#include "attn16.h"
#include "kernels.h"
#include "qdot.h"
#include "refk.h"
#include "topk.h"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <type_traits>

namespace styx {

#pragma clang fp contract(off)

// shaders/moe_reduce_f32.comp: x[i] += sum_s w[s]*d[s*ne+i]
__global__ void __launch_bounds__(256) kr_moe_reduce(const float *d, const float *w, float *x,
                                                     uint32_t ne, uint32_t k)
{
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i >= ne) return;
    float acc = 0.0f;
    for (uint32_t s = 0; s < k; s++) acc += w[s] * d[s * ne + i];
    x[i] += acc;
}

// shaders/add_flat_f32.comp
__global__ void __launch_bounds__(256) kr_add(const float *a, const float *b, float *d, uint32_t n)
{
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) d[i] = a[i] + b[i];
}

// shaders/axpy_sig_f32.comp
__global__ void __launch_bounds__(256) kr_axpy_sig(const float *a, const float *g, float *d,
                                                   uint32_t n)
{
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    const float s = 1.0f / (1.0f + expf(-g[0]));
    if (i < n) d[i] += s * a[i];
}

#pragma clang fp contract(on)

// shaders/matvec_strided_f32.comp: one row per wave.  A router row is a few
// KB and a launch has few rows, so a row's time is its memory round trip:
// every lane has its loads of a 2048-value pass (8 of the row, 8 of x) in
// flight at once.  128 rows of 2048: 21.6 us with 32 lanes and one load at a
// time, 2.6 so.
__global__ void __launch_bounds__(64) kr_matvec_strided(const float *A, const float *x, float *d,
                                                        uint32_t ncols, uint32_t stride)
{
    const uint32_t row = blockIdx.x, tid = threadIdx.x;
    const float *a = A + (int64_t)row * stride;
    float sum = 0.0f;
    uint32_t c0 = 0;
    for (; c0 + 2048 <= ncols; c0 += 2048) {
        f4 av[8], xv[8];
#pragma unroll
        for (int j = 0; j < 8; j++) {
            av[j] = ld4(a + c0 + 256 * j + 4 * tid);
            xv[j] = ld4(x + c0 + 256 * j + 4 * tid);
        }
        float p[8];
#pragma unroll
        for (int j = 0; j < 8; j++)
            p[j] = av[j].x * xv[j].x + av[j].y * xv[j].y + av[j].z * xv[j].z + av[j].w * xv[j].w;
        sum += ((p[0] + p[1]) + (p[2] + p[3])) + ((p[4] + p[5]) + (p[6] + p[7]));
    }
    for (; c0 + 256 <= ncols; c0 += 256) {
        const f4 av = ld4(a + c0 + 4 * tid), xv = ld4(x + c0 + 4 * tid);
        sum += av.x * xv.x + av.y * xv.y + av.z * xv.z + av.w * xv.w;
    }
    for (uint32_t c = c0 + tid; c < ncols; c += 64) sum += a[c] * x[c];
    sum = wave_sum(sum);
    if (tid == 0) d[row] = sum;
}

#pragma clang fp contract(off)

// shaders/attn_decode_f32.comp:31-79 (one workgroup of 128 per query head),
// for head dimensions without a matrix-core kernel and for the shortest
// contexts, empty ones among them.
__global__ void __launch_bounds__(128) kr_attn_decode(const float *Q, const float *K,
                                                      const float *V, float *O, uint32_t n_t,
                                                      uint32_t hd, uint32_t kv_dim, uint32_t gqa,
                                                      float scale)
{
    __shared__ float sh_q[256];
    __shared__ float sh_red[128];
    __shared__ float sh_prob, sh_m, sh_l, sh_corr;
    const uint32_t h = blockIdx.x, tid = threadIdx.x;
    const uint32_t kvoff = (h / gqa) * hd, qbase = h * hd;
    for (uint32_t i = tid; i < hd; i += 128) sh_q[i] = Q[qbase + i];
    __syncthreads();
    float acc0 = 0.0f, acc1 = 0.0f, m = -INFINITY, l = 0.0f;
    for (uint32_t t = 0; t < n_t; t++) {
        const int64_t krow = (int64_t)t * kv_dim + kvoff;
        float part = 0.0f;
        for (uint32_t i = tid; i < hd; i += 128) part += sh_q[i] * K[krow + i];
        sh_red[tid] = part;
        __syncthreads();
        for (uint32_t s = 64; s > 0; s >>= 1) {
            if (tid < s) sh_red[tid] += sh_red[tid + s];
            __syncthreads();
        }
        if (tid == 0) {
            const float sc = sh_red[0] * scale;
            const float m_new = fmaxf(m, sc);
            const float corr = expf(m - m_new);
            const float pr = expf(sc - m_new);
            sh_l = l * corr + pr;
            sh_m = m_new;
            sh_prob = pr;
            sh_corr = corr;
        }
        __syncthreads();
        const float pr = sh_prob, corr = sh_corr;
        m = sh_m;
        l = sh_l;
        if (tid < hd) acc0 = acc0 * corr + pr * V[krow + tid];
        if (tid + 128 < hd) acc1 = acc1 * corr + pr * V[krow + tid + 128];
        __syncthreads();
    }
    const float inv_l = 1.0f / l;
    if (tid < hd) O[qbase + tid] = acc0 * inv_l;
    if (tid + 128 < hd) O[qbase + tid + 128] = acc1 * inv_l;
}

#pragma clang fp contract(on)

// attn_decode_f32 for head dimensions 64, 128 and 256: 16 query heads of one
// kv head per workgroup (attn16.h), so that each K/V row is read once per
// kv head, four waves on every fourth block of 32 keys.  Bound by the keys'
// round trips: a long context is cut into `chunk` keys per workgroup
// (blockIdx.x) whose (m, l, o) go to part [head][chunks][hd + 2] and are
// merged by kr_attn_merge.  Against one workgroup per query head and a
// barrier tree per key: 145 keys 167 -> 16 us, 4000 keys 5360 -> 12 and 4 us
// (32 heads, 4 kv heads of 128).
struct AttnRef {
    const float *Q, *K, *V;
    float *O, *part;  // part: null with one chunk
    uint32_t n_t, kv_dim, gqa, nh, tiles, chunk;  // tiles: of 16 heads per kv head
    float scale;
};

template <int HD> __global__ void __launch_bounds__(256) kr_attn16(AttnRef a)
{
    __shared__ __align__(16) Merge16<HD> s;
    const uint32_t kvh = blockIdx.y / a.tiles, h0 = kvh * a.gqa + blockIdx.y % a.tiles * 16;
    const uint32_t nrow = min(min(a.gqa - blockIdx.y % a.tiles * 16, 16u), a.nh - min(h0, a.nh));
    if (nrow == 0) return;
    const uint32_t c0 = blockIdx.x * a.chunk, nk = min(a.n_t - c0, a.chunk);
    Attn16<HD> at;
    at.init(a.Q + (int64_t)(h0 + min((uint32_t)(threadIdx.x & 15), nrow - 1)) * HD);
    // keys left to this wave, counted down: n_t may be anything up to 2^32 - 1
    // (rows that overlap, kv_dim 0), past which a key position would wrap
    const uint32_t k0 = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) * A16_KB;
    int64_t base = (int64_t)(c0 + k0) * a.kv_dim + (int64_t)kvh * HD;
    for (uint32_t rem = nk - min(nk, k0); rem > 0; rem -= min(rem, 4u * A16_KB), base += 4 * A16_KB * (int64_t)a.kv_dim) {
        const int left = (int)min(rem, (uint32_t)A16_KB);
        at.block(a.K + base, a.V + base, a.kv_dim, left - 1, left, a.scale);
    }
    attn16_merge<HD>(at, s, [&](int r, int d, float O, float L, float M) {
        if ((uint32_t)r >= nrow) return;
        const int64_t h = h0 + r;
        // the last block's missing keys are 0 times its last row: where that
        // holds an infinity, the keys' own sum
        if (O != O && isinf(a.V[(int64_t)(c0 + nk - 1) * a.kv_dim + (int64_t)kvh * HD + d])) {
            O = 0.0f;
            for (uint32_t k = 0; k < nk; k++) {
                const int64_t row = (int64_t)(c0 + k) * a.kv_dim + (int64_t)kvh * HD;
                float x = 0.0f;
#pragma unroll 4
                for (int i = 0; i < HD; i++) x += a.Q[h * HD + i] * a.K[row + i];
                O += expf(x * a.scale - M) * a.V[row + d];
            }
        }
        if (!a.part) {
            a.O[h * HD + d] = O / L;
            return;
        }
        float *p = a.part + (h * gridDim.x + blockIdx.x) * (HD + 2);
        p[2 + d] = O;
        if (d == 0) p[0] = M, p[1] = L;
    });
}

// One workgroup per query row: the chunks' factors in LDS, then 512 / hd
// thread groups over every (512 / hd)th chunk, one thread per dimension,
// eight chunks' loads in flight each (32 chunks: one thread per dimension over
// all of them took 11 us, this 3.9).  Up to 512 chunks.
constexpr int AM_WG = 512;
__global__ void __launch_bounds__(AM_WG) kr_attn_merge(const float *part, float *O, int chunks, int hd)
{
    __shared__ float s_f[AM_WG], red[16], s_o[AM_WG];
    const int tid = threadIdx.x, d = tid % hd, grp = tid / hd, ng = AM_WG / hd;
    const float *p = part + (int64_t)blockIdx.x * chunks * (hd + 2);
    const float m = tid < chunks ? p[(int64_t)tid * (hd + 2)] : -INFINITY;
    const float l = tid < chunks ? p[(int64_t)tid * (hd + 2) + 1] : 0.0f;
    float M = wave_max(m);
    if ((tid & 63) == 0) red[tid >> 6] = M;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < AM_WG / 64; w++) M = fmaxf(M, red[w]);
    const float f = m == -INFINITY ? 0.0f : expf(m - M);
    s_f[tid] = f;
    const float L = block_sum<AM_WG>(l * f, red);  // (its barriers cover s_f)
    float o = 0.0f;
#pragma unroll 8
    for (int c = grp; c < chunks; c += ng) o += p[(int64_t)c * (hd + 2) + 2 + d] * s_f[c];
    s_o[tid] = o;
    __syncthreads();
    if (tid >= hd) return;
    for (int g = 1; g < ng; g++) o += s_o[g * hd + d];
    O[(int64_t)blockIdx.x * hd + d] = o / L;
}

hipError_t launch_attn_merge(hipStream_t st, const float *part, float *O, int rows, int chunks, int hd)
{
    if (!part || rows < 1 || chunks < 1 || chunks > AM_WG || hd < 1 || AM_WG % hd) return hipErrorInvalidValue;
    hipLaunchKernelGGL(kr_attn_merge, dim3(rows), dim3(AM_WG), 0, st, part, O, chunks, hd);
    return hipGetLastError();
}

static hipError_t attn_go(hipStream_t st, AttnRef a, uint32_t hd, const RefScratch *s)
{
    a.tiles = (a.gqa + 15) / 16;
    const uint64_t ny = (uint64_t)((a.nh + a.gqa - 1) / a.gqa) * a.tiles;
    if (ny > 65535) return hipErrorNotSupported;
    a.chunk = attn_chunk_keys(a.n_t, ny, a.nh, hd, s && s->p ? s->floats : 0);
    const uint32_t chunks = (uint32_t)(((uint64_t)a.n_t + a.chunk - 1) / a.chunk);
    a.part = chunks > 1 ? s->p : nullptr;
    const dim3 grid(chunks, (unsigned)ny);
    if (hd == 64)
        hipLaunchKernelGGL(kr_attn16<64>, grid, dim3(256), 0, st, a);
    else if (hd == 128)
        hipLaunchKernelGGL(kr_attn16<128>, grid, dim3(256), 0, st, a);
    else
        hipLaunchKernelGGL(kr_attn16<256>, grid, dim3(256), 0, st, a);
    if (chunks > 1) return launch_attn_merge(st, a.part, a.O, (int)a.nh, (int)chunks, (int)hd);
    return hipGetLastError();
}

#pragma clang fp contract(off)

// swiglu_f32 split mode over n values (GluPush.n).
__global__ void __launch_bounds__(256) kr_swiglu(const float *g, const float *u, float *d, uint32_t n)
{
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) d[i] = g[i] / (1.0f + expf(-g[i])) * u[i];
}

// rms_norm_f32 (generic_binary_head, do_multiply spec): one row per
// workgroup, the row's first 2048 values kept in registers (all their loads,
// and the weights', in flight at once: a 2048-value row 7.3 -> 3.0 us).
__global__ void __launch_bounds__(256) kr_rms_norm(const float *a, const float *w, float *d,
                                                   uint32_t ncols, uint32_t a_row, uint32_t d_row,
                                                   float eps, int mul)
{
    __shared__ float red[16];
    const float *x = a + (int64_t)blockIdx.x * a_row;
    float xv[8], wv[8], ss = 0.0f;
#pragma unroll
    for (int j = 0; j < 8; j++) {
        const uint32_t c = threadIdx.x + 256 * j;
        xv[j] = c < ncols ? x[c] : 0.0f;
        wv[j] = mul && c < ncols ? w[c] : 1.0f;
    }
#pragma unroll
    for (int j = 0; j < 8; j++) ss += xv[j] * xv[j];
    for (uint32_t c = threadIdx.x + 2048; c < ncols; c += 256) ss += x[c] * x[c];
    ss = block_sum<256>(ss, red);
    const float scale = 1.0f / sqrtf(ss / (float)ncols + eps);
    float *y = d + (int64_t)blockIdx.x * d_row;
#pragma unroll
    for (int j = 0; j < 8; j++) {
        const uint32_t c = threadIdx.x + 256 * j;
        if (c < ncols) y[c] = mul ? (scale * xv[j]) * wv[j] : scale * xv[j];
    }
    for (uint32_t c = threadIdx.x + 2048; c < ncols; c += 256) y[c] = mul ? (scale * x[c]) * w[c] : scale * x[c];
}

#pragma clang fp contract(on)

// mul_mat_vec_{t} / mul_mat_vec_id_{t} over GGUF-layout rows.  A row is cut
// into units of 32 values (one q8_0 block, or an eighth of a K-quant block:
// 16 bytes of quants hold its low-nibble values and, 32 or 64 values on, its
// high-nibble ones), so that a lane group of cols / 32 lanes reads a row's
// blocks end to end in 16-byte loads.  A lane keeps its units' activations
// in registers over the rows its group visits and has the next row's loads
// in flight over this row's products: f32 FMAs of weights dequantized one by
// one, as the reference's.  (Factors taken out of the sums, d (s sum q x - m
// sum x), save a third of the products' instructions, which shows in long
// matrices of q6_K only, 151936 x 2048 59 us, so 73; but they cancel: q6_K
// rows times activations around 1 were 5.0e-7 off 64 bits, so 1.0e-7, and an
// infinite activation gave NaN where its row's sum is infinite.)
//
// Bound: the memory round trip at one expert's few rows, the weight stream
// beyond.  Against one lane per block and byte loads into a dequantized
// array in scratch memory (8 of 64 lanes busy on a 2048-column K-quant row),
// 30B-A3B layer: gate q4_K 183 -> 6, up q5_K 178 -> 6, down q6_K 382 -> 8,
// q q8_0 24 -> 8 us.
struct MmvRef {
    const uint8_t *A;
    const float *B;
    float *D;
    const int32_t *ids;  // null for the plain matvec
    int type;
    uint32_t ncols, stride_a, stride_b, stride_d, batch_stride_a, batch_stride_b, batch_stride_d;
    uint32_t ne11, expert_i1, nbi1, nrows;
    int64_t n_mat;  // matrices readable from A (ids at or past it are skipped)
    int G;          // lanes per row (a power of two)
    int passes;     // rows per lane group
};

constexpr int MMV_WG = 256;

// 16 bytes at a 2-byte aligned address (34- and 210-byte blocks).
__device__ __forceinline__ styx_u4 ld16u(const uint8_t *p)
{
    struct __attribute__((packed, aligned(2))) U { uint32_t w[4]; };
    const U *u = (const U *)p;
    return styx_u4{u->w[0], u->w[1], u->w[2], u->w[3]};
}
__device__ __forceinline__ styx_u4 ld16(const uint8_t *p) { return *(const styx_u4 *)p; }

template <int N> __device__ __forceinline__ float ubyte(uint32_t v) { return (float)((v >> (8 * N)) & 255u); }

template <int N> __device__ __forceinline__ float sbyte(uint32_t v) { return (float)(int8_t)(v >> (8 * N)); }

// sum of y(byte) x over 16 bytes (signed if S) and x[0..16), y the byte's weight
template <bool S = false, typename Y> __device__ __forceinline__ float dot16(const styx_u4 q, const float *x, Y y)
{
    auto b = [&](auto n, int i) { return y(S ? sbyte<decltype(n)::value>(q[i]) : ubyte<decltype(n)::value>(q[i])); };
    using std::integral_constant;
    const integral_constant<int, 0> n0;
    const integral_constant<int, 1> n1;
    const integral_constant<int, 2> n2;
    const integral_constant<int, 3> n3;
    float s[4];
#pragma unroll
    for (int i = 0; i < 4; i++)
        s[i] = fmaf(b(n0, i), x[4 * i], b(n1, i) * x[4 * i + 1]) + fmaf(b(n2, i), x[4 * i + 2], b(n3, i) * x[4 * i + 3]);
    return (s[0] + s[1]) + (s[2] + s[3]);
}

// One unit's activations: two runs of 16 values.
struct MX {
    float x[32];
    __device__ __forceinline__ void load(const float *b, int lo, int hi)
    {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const f4 u = ld4(b + lo + 4 * i), v = ld4(b + hi + 4 * i);
#pragma unroll
            for (int j = 0; j < 4; j++) x[4 * i + j] = u[j], x[16 + 4 * i + j] = v[j];
        }
    }
};

// Unit u of a row: its block, the first value of its two runs, its loads
// and its share of the dot product.
template <int T> struct MU;
template <> struct MU<T_Q8_0> {
    styx_u4 q0, q1;
    uint32_t d;
    static __device__ __forceinline__ void runs(int u, int &lo, int &hi) { lo = 32 * u, hi = lo + 16; }
    __device__ __forceinline__ void load(const uint8_t *row, int u)
    {
        const uint8_t *b = row + 34 * (int64_t)u;
        d = *(const uint16_t *)b;
        q0 = ld16u(b + 2);
        q1 = ld16u(b + 18);
    }
    __device__ __forceinline__ float dot(const MX &x, int) const
    {
        const float df = f16f(d);
        auto y = [=](float v) { return df * v; };
        return dot16<true>(q0, x.x, y) + dot16<true>(q1, x.x + 16, y);
    }
};
// q4_K / q5_K: part p = u & 7 reads quant bytes [16 p, +16): run h = p & 1
// of quarter c = p >> 1.
template <int T> struct MUK {
    styx_u4 q, hd, qh;
    static __device__ __forceinline__ void runs(int u, int &lo, int &hi)
    {
        lo = 256 * (u >> 3) + 64 * ((u >> 1) & 3) + 16 * (u & 1);
        hi = lo + 32;
    }
    __device__ __forceinline__ void load(const uint8_t *row, int u)
    {
        const uint8_t *b = row + (T == T_Q4_K ? 144 : 176) * (int64_t)(u >> 3);
        hd = ld16(b);
        q = ld16(b + (T == T_Q4_K ? 16 : 48) + 16 * (u & 7));
        if (T == T_Q5_K) qh = ld16(b + 16 + 16 * (u & 1));
    }
    __device__ __forceinline__ float dot(const MX &x, int u) const
    {
        const int c = (u >> 1) & 3;
        styx_u4 lo = q & 0x0F0F0F0Fu, hi = (q >> 4) & 0x0F0F0F0Fu;
        if (T == T_Q5_K) {
            const styx_u4 h = qh >> (uint32_t)(2 * c);
            lo |= (h & 0x01010101u) << 4;
            hi |= (h & 0x02020202u) << 3;
        }
        float s0, s1, m0, m1;
        k4_scales(make_uint4(hd.x, hd.y, hd.z, hd.w), 16 * (c & 1), c >> 1, s0, s1, m0, m1);
        const float d = f16f(hd.x), dm = f16f(hd.x >> 16);
        s0 *= d, s1 *= d, m0 *= dm, m1 *= dm;
        return dot16(lo, x.x, [=](float u) { return fmaf(s0, u, -m0); }) +
               dot16(hi, x.x + 16, [=](float u) { return fmaf(s1, u, -m1); });
    }
};
template <> struct MU<T_Q4_K> : MUK<T_Q4_K> {};
template <> struct MU<T_Q5_K> : MUK<T_Q5_K> {};
// q6_K: part p = u & 7 reads low bits [16 p, +16): half n = p >> 2, run
// j = (p >> 1) & 1, piece h = p & 1.
template <> struct MU<T_Q6_K> {
    styx_u4 q, qh;
    uint32_t sc, d;  // the two runs' scales, bytes 0 and 2
    static __device__ __forceinline__ void runs(int u, int &lo, int &hi)
    {
        const int p = u & 7;
        lo = 256 * (u >> 3) + 128 * (p >> 2) + 32 * ((p >> 1) & 1) + 16 * (p & 1);
        hi = lo + 64;
    }
    __device__ __forceinline__ void load(const uint8_t *row, int u)
    {
        const int p = u & 7, n = p >> 2;
        const uint8_t *b = row + 210 * (int64_t)(u >> 3);
        q = ld16u(b + 16 * p);
        qh = ld16u(b + 128 + 32 * n + 16 * (p & 1));
        const uint8_t *s = b + 192 + 8 * n + (p & 3);
        sc = (uint32_t)s[0] | (uint32_t)s[4] << 16;
        d = *(const uint16_t *)(b + 208);
    }
    __device__ __forceinline__ float dot(const MX &x, int u) const
    {
        const uint32_t j2 = 2 * ((u >> 1) & 1);
        const styx_u4 lo = (q & 0x0F0F0F0Fu) | (((qh >> j2) & 0x03030303u) << 4);
        const styx_u4 hi = ((q >> 4) & 0x0F0F0F0Fu) | (((qh >> (j2 + 4u)) & 0x03030303u) << 4);
        const float s0 = f16f(d) * (float)(int8_t)sc, s1 = f16f(d) * (float)(int8_t)(sc >> 16);
        // s (u - 32) in one rounding: s u and 32 s are exact
        return dot16(lo, x.x, [=](float u) { return fmaf(s0, u, -32.0f * s0); }) +
               dot16(hi, x.x + 16, [=](float u) { return fmaf(s1, u, -32.0f * s1); });
    }
};

// UPL: units per lane whose activations stay in registers (1 or 2; rows of
// up to 64 or 128 units); 0: any length, activations read again per row.
template <int T, int UPL> __global__ void __launch_bounds__(MMV_WG) kr_mmv(MmvRef p)
{
    constexpr int bb = T == T_Q8_0 ? 34 : T == T_Q4_K ? 144 : T == T_Q5_K ? 176 : 210;
    constexpr int be = T == T_Q8_0 ? 32 : 256;
    const uint32_t slot = blockIdx.y;
    const uint8_t *A = p.A;
    int64_t b_off = 0, d_off = 0;
    if (p.ids) {
        // get_offsets() of mul_mat_vec_base (crates/vk-backend/tests/kernels.rs:124-131)
        const uint32_t e = (uint32_t)p.ids[slot + p.expert_i1 * p.nbi1];
        if (e == SKIP || (int64_t)e >= p.n_mat) return;
        A += (int64_t)e * (p.batch_stride_a / be) * bb;
        b_off = (int64_t)(slot % p.ne11) * p.stride_b + (int64_t)p.expert_i1 * p.batch_stride_b;
        d_off = (int64_t)slot * p.stride_d + (int64_t)p.expert_i1 * p.batch_stride_d;
    }
    const int lg = __builtin_ctz((unsigned)p.G);
    const int lane = threadIdx.x & 63, gl = lane & (p.G - 1), ngrp = MMV_WG >> lg;
    const int64_t first = (int64_t)blockIdx.x * ngrp * p.passes + (threadIdx.x >> lg);
    const int nu = (int)(p.ncols / 32);
    const float *B = p.B + b_off;
    const int64_t rb = (int64_t)p.stride_a * bb;
    auto row_at = [&](int i) {
        return A + rb * min(first + (int64_t)i * ngrp, (int64_t)p.nrows - 1);
    };
    auto put = [&](int i, float v) {
        v = group_sum(v, gl, p.G);
        const int64_t r = first + (int64_t)i * ngrp;
        if (gl == 0 && r < p.nrows) p.D[d_off + r] = v;
    };
    if constexpr (UPL > 0) {
        MX x[UPL];
        MU<T> w[UPL];
        // a lane past the row's units works on unit 0 and adds nothing
        int un[UPL];
        bool on[UPL];
#pragma unroll
        for (int j = 0; j < UPL; j++) {
            on[j] = gl + j * p.G < nu;
            un[j] = on[j] ? gl + j * p.G : 0;
            w[j].load(row_at(0), un[j]);
        }
#pragma unroll
        for (int j = 0; j < UPL; j++) {
            int lo, hi;
            MU<T>::runs(un[j], lo, hi);
            x[j].load(B, lo, hi);
        }
        for (int i = 0; i < p.passes; i++) {
            MU<T> c[UPL];
#pragma unroll
            for (int j = 0; j < UPL; j++) {
                c[j] = w[j];
                if (i + 1 < p.passes) w[j].load(row_at(i + 1), un[j]);
            }
            float v = 0.0f;
#pragma unroll
            for (int j = 0; j < UPL; j++) {
                const float t = c[j].dot(x[j], un[j]);
                if (on[j]) v += t;
            }
            put(i, v);
        }
    } else {
        for (int i = 0; i < p.passes; i++) {
            const uint8_t *row = row_at(i);
            float v = 0.0f;
            for (int u = gl; u < nu; u += p.G) {
                MU<T> w;
                MX x;
                int lo, hi;
                w.load(row, u);
                MU<T>::runs(u, lo, hi);
                x.load(B, lo, hi);
                v += w.dot(x, u);
            }
            put(i, v);
        }
    }
}

template <int T> static void mmv_go(hipStream_t st, MmvRef &p, uint32_t slots)
{
    const uint32_t nu = p.ncols / 32;
    p.G = 1;
    while (p.G < 64 && (uint32_t)p.G < nu) p.G *= 2;
    // about 4096 waves over all slots' rows, at least one row per lane group
    const uint64_t ngrp = MMV_WG / p.G, groups = 4096ull * 64 / p.G;
    p.passes = (int)std::max<uint64_t>(1, ((uint64_t)p.nrows * slots + groups - 1) / groups);
    const uint64_t per = ngrp * p.passes;
    const dim3 grid((unsigned)((p.nrows + per - 1) / per), slots);
    if (nu <= 64)
        hipLaunchKernelGGL((kr_mmv<T, 1>), grid, dim3(MMV_WG), 0, st, p);
    else if (nu <= 128)
        hipLaunchKernelGGL((kr_mmv<T, 2>), grid, dim3(MMV_WG), 0, st, p);
    else
        hipLaunchKernelGGL((kr_mmv<T, 0>), grid, dim3(MMV_WG), 0, st, p);
}

// topk_softmax_f32 with the shader's bindings (remap/pmap required).
__global__ void __launch_bounds__(64) kr_topk(const float *logits, float *w, int32_t *ids,
                                              const uint32_t *remap, const uint32_t *pmap,
                                              uint32_t n, uint32_t k, uint32_t renorm)
{
    topk_wave(logits, (int)n, (int)k, (int)renorm, remap, pmap, 0, 0, w, ids);
}

// rope_neox_f32 with the RopePush of crates/vk-backend/src/ops.rs:385-439
// for the mode the engine uses (NEOX, no frequency factors, no YaRN:
// ext_factor 0, freq_scale 1, attn_factor 1): row r = (i3, i2, i1) of
// (ne01, ne02) rows, pair i < ne00/2 of this thread; pairs (i, i + n/2) of
// the first n_dims values rotate by pos[i2] * base^(-2i/n_dims), the angle
// and its sine and cosine in f64 (the reference test's CPU formula,
// crates/vk-backend/tests/ops2.rs:426-442); values past n_dims are copied.
struct RopeArgs {
    const float *src;
    const int32_t *pos;
    float *dst;
    uint32_t nrows, n_dims, ne00, ne01, ne02;
    uint32_t nb01, nb02, nb03, nb11, nb12, nb13, a_off, d_off;
    double theta_scale;
};

__global__ void __launch_bounds__(256) kr_rope_neox(RopeArgs a)
{
    const uint32_t r = blockIdx.x, i = blockIdx.y * 256 + threadIdx.x;
    if (r >= a.nrows || 2 * i >= a.ne00) return;
    const uint32_t i1 = r % a.ne01, i2 = (r / a.ne01) % a.ne02, i3 = r / (a.ne01 * a.ne02);
    const int64_t s0 = a.a_off + (int64_t)i3 * a.nb03 + (int64_t)i2 * a.nb02 + (int64_t)i1 * a.nb01;
    const int64_t d0 = a.d_off + (int64_t)i3 * a.nb13 + (int64_t)i2 * a.nb12 + (int64_t)i1 * a.nb11;
    if (2 * i >= a.n_dims) {  // past the rotated dims: copied through
        a.dst[d0 + 2 * i] = a.src[s0 + 2 * i];
        a.dst[d0 + 2 * i + 1] = a.src[s0 + 2 * i + 1];
        return;
    }
    const uint32_t half = a.n_dims / 2;
    const double th = (double)a.pos[i2] * pow(a.theta_scale, (double)i);
    double sn, cs;
    sincos(th, &sn, &cs);
    const double x0 = a.src[s0 + i], x1 = a.src[s0 + i + half];
    a.dst[d0 + i] = (float)(x0 * cs - x1 * sn);
    a.dst[d0 + i + half] = (float)(x0 * sn + x1 * cs);
}

// cpy_f32_f32 with the UnaryPush of ops.rs:253-323: element j < ne of the
// source, at its 4-d index in src0's extents and strides (plus the
// misalignment offset's high half), goes to the same running index in dst's
// extents and strides (plus the low half).  512 elements per workgroup
// (the engine's grid, crates/model/src/moe.rs:1935-1943).
struct CpyArgs {
    const float *src;
    float *dst;
    uint32_t ne;
    uint32_t sne[4], snb[4], dne[4], dnb[4];
    uint32_t a_off, d_off;
};

__device__ __forceinline__ int64_t elem_at(uint32_t j, const uint32_t *ne, const uint32_t *nb)
{
    const uint32_t i0 = j % ne[0], i1 = (j / ne[0]) % ne[1], i2 = (j / (ne[0] * ne[1])) % ne[2],
                   i3 = j / (ne[0] * ne[1] * ne[2]);
    return (int64_t)i3 * nb[3] + (int64_t)i2 * nb[2] + (int64_t)i1 * nb[1] + (int64_t)i0 * nb[0];
}

__global__ void __launch_bounds__(256) kr_cpy(CpyArgs a)
{
    const uint64_t wg = ((uint64_t)blockIdx.z * gridDim.y + blockIdx.y) * gridDim.x + blockIdx.x;
    for (uint32_t t = threadIdx.x; t < 512; t += 256) {
        const uint64_t j = wg * 512 + t;
        if (j >= a.ne) return;
        a.dst[a.d_off + elem_at((uint32_t)j, a.dne, a.dnb)] = a.src[a.a_off + elem_at((uint32_t)j, a.sne, a.snb)];
    }
}

// Whether n elements of `bytes_each` bytes fit in a binding of `size` bytes
// (n may be 0).
static bool fits(uint64_t size, uint64_t n, uint64_t bytes_each)
{
    return n == 0 || (bytes_each != 0 && n <= size / bytes_each);
}

hipError_t refk_launch(hipStream_t st, int kid, void *const *ptr, const uint64_t *size,
                       const void *push, uint32_t gx, uint32_t gy, uint32_t gz,
                       const uint32_t *spec, int n_spec, const RefScratch *scratch)
{
    const uint32_t *pc = (const uint32_t *)push;
    const hipError_t bad = hipErrorInvalidValue;
    switch (kid) {
    case RK_MOE_REDUCE: {
        // push: ne, k
        const uint64_t ne = pc[0], k = pc[1];
        if (!fits(size[0], k * ne, 4) || !fits(size[1], k, 4) || !fits(size[2], ne, 4)) return bad;
        hipLaunchKernelGGL(kr_moe_reduce, dim3(gx), dim3(256), 0, st, (const float *)ptr[0],
                           (const float *)ptr[1], (float *)ptr[2], pc[0], pc[1]);
        break;
    }
    case RK_ADD:
        if (!fits(size[0], pc[0], 4) || !fits(size[1], pc[0], 4) || !fits(size[2], pc[0], 4)) return bad;
        hipLaunchKernelGGL(kr_add, dim3(gx), dim3(256), 0, st, (const float *)ptr[0],
                           (const float *)ptr[1], (float *)ptr[2], pc[0]);
        break;
    case RK_AXPY_SIG:
        if (!fits(size[0], pc[0], 4) || !fits(size[1], 1, 4) || !fits(size[2], pc[0], 4)) return bad;
        hipLaunchKernelGGL(kr_axpy_sig, dim3(gx), dim3(256), 0, st, (const float *)ptr[0],
                           (const float *)ptr[1], (float *)ptr[2], pc[0]);
        break;
    case RK_MATVEC_STRIDED: {
        // push: ncols, stride; one row per workgroup
        const uint64_t nc = pc[0], stride = pc[1];
        if (!fits(size[0], (uint64_t)(gx - 1) * stride + nc, 4) || !fits(size[1], nc, 4) ||
            !fits(size[2], gx, 4))
            return bad;
        hipLaunchKernelGGL(kr_matvec_strided, dim3(gx), dim3(64), 0, st, (const float *)ptr[0],
                           (const float *)ptr[1], (float *)ptr[2], pc[0], pc[1]);
        break;
    }
    case RK_ATTN: {
        // push: n_t, hd, kv_dim, gqa, scale; one query head per workgroup
        float scale;
        std::memcpy(&scale, pc + 4, 4);
        const uint64_t n_t = pc[0], hd = pc[1], kvd = pc[2], gqa = pc[3];
        if (hd == 0 || hd > 256 || gqa == 0) return bad;
        const uint64_t kv_need = n_t ? (n_t - 1) * kvd + ((gx - 1) / gqa) * hd + hd : 0;
        if (!fits(size[0], (uint64_t)gx * hd, 4) || !fits(size[1], kv_need, 4) ||
            !fits(size[2], kv_need, 4) || !fits(size[3], (uint64_t)gx * hd, 4))
            return bad;
        // A block of 32 keys costs the matrix-core kernel the same however few
        // it has, so up to hd / 32 keys one workgroup per head is faster.  us
        // per head dimension, general and matrix-core kernel: 64, 2 and 3
        // keys: 5.8 and 7.4, 6.7 and 7.0; 128, 4 and 5: 7.7 and 9.3, 8.5 and
        // 9.0; 256, 8 and 9: 12.7 and 14.7, 13.7 and 14.4, 1: 5.6 and 14.5.
        if (n_t > hd / 32 && (hd == 64 || hd == 128 || hd == 256)) {
            AttnRef a{};
            a.Q = (const float *)ptr[0];
            a.K = (const float *)ptr[1];
            a.V = (const float *)ptr[2];
            a.O = (float *)ptr[3];
            a.n_t = pc[0];
            a.kv_dim = pc[2];
            a.gqa = (uint32_t)std::min<uint64_t>(gqa, gx);
            a.nh = gx;
            a.scale = scale;
            const hipError_t e = attn_go(st, a, pc[1], scratch);
            if (e != hipErrorNotSupported) return e;
        }
        hipLaunchKernelGGL(kr_attn_decode, dim3(gx), dim3(128), 0, st, (const float *)ptr[0],
                           (const float *)ptr[1], (const float *)ptr[2], (float *)ptr[3], pc[0],
                           pc[1], pc[2], pc[3], scale);
        break;
    }
    case RK_SWIGLU:
        // GluPush: n is the first field
        if (!fits(size[0], pc[0], 4) || !fits(size[1], pc[0], 4) || !fits(size[2], pc[0], 4)) return bad;
        hipLaunchKernelGGL(kr_swiglu, dim3((pc[0] + 255) / 256), dim3(256), 0, st,
                           (const float *)ptr[0], (const float *)ptr[1], (float *)ptr[2], pc[0]);
        break;
    case RK_RMS_NORM: {
        // BinaryPush: ne, src0[8] (ne00..ne03, nb00..nb03), src1[8], dst[8], misalign, param1
        float eps;
        std::memcpy(&eps, pc + 26, 4);
        int mul = 1;
        for (int i = 0; i + 1 < 2 * n_spec; i += 2)
            if (spec[i] == 1) mul = spec[i + 1] != 0;
        const uint64_t nc = pc[1], arow = pc[6], drow = pc[22];
        if (!fits(size[0], (uint64_t)(gx - 1) * arow + nc, 4) || (mul && !fits(size[1], nc, 4)) ||
            !fits(size[2], (uint64_t)(gx - 1) * drow + nc, 4))
            return bad;
        hipLaunchKernelGGL(kr_rms_norm, dim3(gx), dim3(256), 0, st, (const float *)ptr[0],
                           (const float *)ptr[1], (float *)ptr[2], pc[1], pc[6], pc[22], eps, mul);
        break;
    }
    case RK_ROPE_NEOX: {
        float f[29];
        std::memcpy(f, pc, sizeof(f));
        RopeArgs a{};
        a.nrows = pc[1];
        a.n_dims = pc[2];
        const float freq_scale = f[3], freq_base = f[4], ext_factor = f[5], attn_factor = f[6];
        a.ne00 = pc[18], a.ne01 = pc[19], a.ne02 = pc[20];
        a.nb01 = pc[21], a.nb02 = pc[22], a.nb03 = pc[23];
        a.nb11 = pc[24], a.nb12 = pc[25], a.nb13 = pc[26];
        a.a_off = pc[27], a.d_off = pc[28];
        // the supported mode: NEOX (2), no frequency factors, no YaRN, not
        // the backward pass, no set_rows, rotation within each row
        if (pc[0] != 2 || freq_scale != 1.0f || ext_factor != 0.0f || attn_factor != 1.0f ||
            pc[10] != 0 || pc[15] != 0 || pc[16] != 0 || pc[17] != 0 || a.n_dims == 0 ||
            a.n_dims % 2 || a.n_dims > a.ne00 || a.ne00 % 2 || a.ne01 == 0 || a.ne02 == 0 ||
            !(freq_base > 0.0f) || gx < a.nrows || (uint64_t)gy * 256 < a.ne00 / 2)
            return bad;
        const uint64_t n3 = ((uint64_t)a.nrows + a.ne01 * a.ne02 - 1) / ((uint64_t)a.ne01 * a.ne02);
        const uint64_t src_need = a.a_off + (n3 - 1) * a.nb03 + (uint64_t)(a.ne02 - 1) * a.nb02 +
                                  (uint64_t)(a.ne01 - 1) * a.nb01 + a.ne00;
        const uint64_t dst_need = a.d_off + (n3 - 1) * a.nb13 + (uint64_t)(a.ne02 - 1) * a.nb12 +
                                  (uint64_t)(a.ne01 - 1) * a.nb11 + a.ne00;
        if (!fits(size[0], src_need, 4) || !fits(size[1], a.ne02, 4) || !fits(size[3], dst_need, 4))
            return bad;
        a.src = (const float *)ptr[0];
        a.pos = (const int32_t *)ptr[1];
        a.dst = (float *)ptr[3];
        a.theta_scale = std::pow((double)freq_base, -2.0 / (double)a.n_dims);
        hipLaunchKernelGGL(kr_rope_neox, dim3(a.nrows, (a.ne00 / 2 + 255) / 256), dim3(256), 0, st,
                           a);
        break;
    }
    case RK_CPY: {
        CpyArgs a{};
        a.ne = pc[0];
        for (int i = 0; i < 4; i++) {
            a.sne[i] = pc[1 + i];
            a.snb[i] = pc[5 + i];
            a.dne[i] = pc[9 + i];
            a.dnb[i] = pc[13 + i];
        }
        a.a_off = pc[17] >> 16;
        a.d_off = pc[17] & 0xFFFF;
        uint64_t sn = 1, dn = 1, s_need = a.a_off + 1, d_need = a.d_off + 1;
        for (int i = 0; i < 4; i++) {
            if (a.sne[i] == 0 || a.dne[i] == 0) return bad;
            sn *= a.sne[i];
            dn *= a.dne[i];
            s_need += (uint64_t)(a.sne[i] - 1) * a.snb[i];
            d_need += (uint64_t)(a.dne[i] - 1) * a.dnb[i];
        }
        if (a.ne == 0 || sn < a.ne || dn < a.ne || sn > 0xFFFFFFFFull || dn > 0xFFFFFFFFull ||
            (uint64_t)gx * gy * gz * 512 < a.ne || !fits(size[0], s_need, 4) ||
            !fits(size[1], d_need, 4))
            return bad;
        a.src = (const float *)ptr[0];
        a.dst = (float *)ptr[1];
        hipLaunchKernelGGL(kr_cpy, dim3(gx, gy, gz), dim3(256), 0, st, a);
        break;
    }
    case RK_TOPK:
        // push: n, k, renorm; writes the 64-entry id row
        if (pc[0] < 1 || pc[0] > MAX_EXPERTS || pc[1] < 1 || pc[1] > MAX_TOPK)
            return bad;
        if (!fits(size[0], pc[0], 4) || !fits(size[1], pc[1], 4) || !fits(size[2], IDS_ROW, 4) ||
            !fits(size[3], pc[0], 4) || !fits(size[4], pc[0], 4))
            return bad;
        hipLaunchKernelGGL(kr_topk, dim3(1), dim3(64), 0, st, (const float *)ptr[0],
                           (float *)ptr[1], (int32_t *)ptr[2], (const uint32_t *)ptr[3],
                           (const uint32_t *)ptr[4], pc[0], pc[1], pc[2]);
        break;
    case RK_GATHER: {
        // push: dst_vg, dst_vu, dst_vd, src_vg, src_vu, src_vd, layer, k, canary
        if (pc[8] != 0) return bad;
        const uint8_t *src[3] = {(const uint8_t *)ptr[0], (const uint8_t *)ptr[1],
                                 (const uint8_t *)ptr[2]};
        uint8_t *dst[3] = {(uint8_t *)ptr[3], (uint8_t *)ptr[4], (uint8_t *)ptr[5]};
        const int64_t ss[3] = {16ll * pc[3], 16ll * pc[4], 16ll * pc[5]};
        const int64_t ds[3] = {16ll * pc[0], 16ll * pc[1], 16ll * pc[2]};
        const uint64_t k = pc[7], slots = ((uint64_t)pc[6] + 1) * k;
        if (k < 1 || k > MAX_TOPK || !fits(size[6], k, 4)) return bad;
        int64_t cnt[3];
        for (int t = 0; t < 3; t++) {
            if (ss[t] == 0 || !fits(size[3 + t], slots, (uint64_t)ds[t])) return bad;
            cnt[t] = (int64_t)(size[t] / (uint64_t)ss[t]);
        }
        return launch_gather_list(st, src, ss, dst, ds, (const int32_t *)ptr[6], (int)pc[7],
                                  (int)pc[6], cnt);
    }
    default: {
        if (kid < RK_MMV_BASE || kid >= RK_MMV_BASE + 8) return bad;
        const int ti = (kid - RK_MMV_BASE) % 4;
        const bool with_id = kid >= RK_MMV_BASE + 4;
        static const int types[4] = {T_Q8_0, T_Q4_K, T_Q5_K, T_Q6_K};
        MmvRef p{};
        p.type = types[ti];
        p.A = (const uint8_t *)ptr[0];
        p.B = (const float *)ptr[1];
        p.D = (float *)ptr[2];
        p.ncols = pc[0];
        p.stride_a = pc[1];
        p.stride_b = pc[2];
        p.stride_d = pc[3];
        p.batch_stride_a = pc[4];
        p.batch_stride_b = pc[5];
        p.batch_stride_d = pc[6];
        const uint64_t be = blk_elems(p.type), bb = blk_bytes(p.type), nb = p.ncols / be;
        if (p.ncols == 0 || p.ncols % be || p.stride_a < nb) return bad;
        if (with_id) {
            // MatVecIdPush: ..., fusion_flags, nei0, ne11, expert_i1, nbi1
            p.ids = (const int32_t *)ptr[5];
            p.ne11 = pc[9] ? pc[9] : 1;
            p.expert_i1 = pc[10];
            p.nbi1 = pc[11];
            p.nrows = gx;
            if (p.batch_stride_a % be) return bad;
            // one matrix: nrows rows of stride_a blocks, within the expert stride
            const uint64_t mat_blocks = (uint64_t)p.batch_stride_a / be;
            const uint64_t used_blocks = (uint64_t)(p.nrows - 1) * p.stride_a + nb;
            if (mat_blocks == 0 || used_blocks > mat_blocks) return bad;
            p.n_mat = (int64_t)(size[0] / (mat_blocks * bb));
            const uint64_t nsl = gy, ne11 = p.ne11;
            const uint64_t b_need = (std::min<uint64_t>(nsl, ne11) - 1) * p.stride_b +
                                    (uint64_t)p.expert_i1 * p.batch_stride_b + p.ncols;
            const uint64_t d_need = (nsl - 1) * p.stride_d +
                                    (uint64_t)p.expert_i1 * p.batch_stride_d + p.nrows;
            const uint64_t id_need = (nsl - 1) + (uint64_t)p.expert_i1 * p.nbi1 + 1;
            if (!fits(size[1], b_need, 4) || !fits(size[2], d_need, 4) || !fits(size[5], id_need, 4))
                return bad;
        } else {
            // MatVecPush: stride_d = nrows (MatVecPush::simple); NUM_ROWS spec id 1
            uint64_t num_rows = 1;
            for (int i = 0; i + 1 < 2 * n_spec; i += 2)
                if (spec[i] == 1) num_rows = spec[i + 1] ? spec[i + 1] : 1;
            p.nrows = p.stride_d;
            p.n_mat = 1;
            if (p.nrows == 0 || !fits(size[0], (uint64_t)(p.nrows - 1) * p.stride_a + nb, bb) ||
                !fits(size[1], p.ncols, 4) || !fits(size[2], p.nrows, 4))
                return bad;
            // the rows the grid covers
            p.nrows = (uint32_t)std::min<uint64_t>(p.nrows, num_rows * gx);
        }
        const uint32_t slots = with_id ? gy : 1;
        switch (p.type) {
        case T_Q8_0: mmv_go<T_Q8_0>(st, p, slots); break;
        case T_Q4_K: mmv_go<T_Q4_K>(st, p, slots); break;
        case T_Q5_K: mmv_go<T_Q5_K>(st, p, slots); break;
        default: mmv_go<T_Q6_K>(st, p, slots); break;
        }
        break;
    }
    }
    return hipGetLastError();
}

}  // namespace styx
