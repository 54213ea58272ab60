// attn16.h -- softmax attention of 16 query rows of one kv head by one wave,
// all products f32 on the matrix cores (v_mfma_f32_16x16x4_f32); shared by
// the prompt batch and the reference's attn_decode_f32 pipeline.
//
// Lane (n = lane & 15, g = lane >> 4) holds query row n.  Scores are formed
// transposed (keys x queries): a lane then holds its own query's scores of
// keys 4 g + i of each 16-key tile, so the softmax factors are lane-local,
// and the scores are already laid out as the operand of the value product.
// K and V are read in 16-byte pieces, the head's dimensions permuted alike
// on both sides of each product.
#pragma once

#include <algorithm>

#include "qdot.h"
#include "refk.h"

namespace styx {

typedef float f4 __attribute__((ext_vector_type(4)));

// Four floats at a 4-byte aligned address, as one load.
__device__ __forceinline__ f4 ld4(const float *p)
{
    f4 v;
    __builtin_memcpy(&v, p, 16);
    return v;
}

// Over the four lane groups of each n, every lane getting the result.
__device__ __forceinline__ float groups_max(float v)
{
    const auto x = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = fmaxf(__uint_as_float(x[0]), __uint_as_float(x[1]));
    const auto y = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return fmaxf(__uint_as_float(y[0]), __uint_as_float(y[1]));
}
__device__ __forceinline__ float groups_sum(float v)
{
    const auto x = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = __uint_as_float(x[0]) + __uint_as_float(x[1]);
    const auto y = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(y[0]) + __uint_as_float(y[1]);
}

constexpr int A16_KT = 2, A16_KB = 16 * A16_KT;  // tiles and keys of a block

template <int HD> struct Attn16 {
    static constexpr int NQ = HD / 16, NV = HD / 64;
    f4 q[NQ], o[NV][4];
    float m, l;  // l: this lane group's share of the sum

    __device__ __forceinline__ void init(const float *qp)
    {
        const int g = (threadIdx.x & 63) >> 4;
#pragma unroll
        for (int i = 0; i < NQ; i++) q[i] = ld4(qp + 16 * i + 4 * g);
#pragma unroll
        for (int j = 0; j < NV; j++)
#pragma unroll
            for (int e = 0; e < 4; e++) o[j][e] = f4{0.0f, 0.0f, 0.0f, 0.0f};
        m = -INFINITY;
        l = 0.0f;
    }

    // A block of keys: rows `stride` floats apart at kb / vb, of which rows
    // past lim are not read and those at or past vis are not seen by this
    // lane's query.  Those meet a factor 0 (rows past lim: times row lim
    // again), which a V value that is not finite turns into NaN: the callers
    // see to that.
    __device__ __forceinline__ void block(const float *kb, const float *vb, int64_t stride, int lim,
                                          int vis, float scale)
    {
        const int n = threadIdx.x & 15, g = (threadIdx.x & 63) >> 4;
        const f4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
        float sc[A16_KT][4], mn = m;
#pragma unroll
        for (int b = 0; b < A16_KT; b++) {
            const float *kp = kb + min(16 * b + n, lim) * stride + 4 * g;
            f4 s4[2][4];
#pragma unroll
            for (int i = 0; i < NQ; i++) {
                const f4 kf = ld4(kp + 16 * i);
#pragma unroll
                for (int e = 0; e < 4; e++)
                    s4[i & 1][e] = __builtin_amdgcn_mfma_f32_16x16x4f32(
                        kf[e], q[i][e], i < 2 ? zero : s4[i & 1][e], 0, 0, 0);
            }
            const f4 s = ((s4[0][0] + s4[0][1]) + (s4[0][2] + s4[0][3])) +
                         ((s4[1][0] + s4[1][1]) + (s4[1][2] + s4[1][3]));
#pragma unroll
            for (int i = 0; i < 4; i++) {
                sc[b][i] = 16 * b + 4 * g + i < vis ? s[i] * scale : -INFINITY;
                mn = fmaxf(mn, sc[b][i]);
            }
        }
        mn = groups_max(mn);
        const float mz = mn == -INFINITY ? 0.0f : mn;  // no key of this query yet
        const float corr = expf(m - mz);
        m = mn;
        float lb = 0.0f;
#pragma unroll
        for (int b = 0; b < A16_KT; b++) {
#pragma unroll
            for (int i = 0; i < 4; i++) sc[b][i] = expf(sc[b][i] - mz);
            lb += (sc[b][0] + sc[b][1]) + (sc[b][2] + sc[b][3]);
        }
        l = l * corr + lb;
        // the block's value sum on its own, then added: the running sum is
        // rounded once per block, not once per four keys
        f4 ob[NV][4];
#pragma unroll
        for (int b = 0; b < A16_KT; b++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const float *vp = vb + min(16 * b + 4 * g + i, lim) * stride + 4 * n;
#pragma unroll
                for (int j = 0; j < NV; j++) {
                    const f4 v = ld4(vp + 64 * j);
#pragma unroll
                    for (int e = 0; e < 4; e++)
                        ob[j][e] = __builtin_amdgcn_mfma_f32_16x16x4f32(
                            v[e], sc[b][i], b + i == 0 ? zero : ob[j][e], 0, 0, 0);
                }
            }
#pragma unroll
        for (int j = 0; j < NV; j++)
#pragma unroll
            for (int e = 0; e < 4; e++) o[j][e] = o[j][e] * corr + ob[j][e];
    }
};

// The four waves' results of the 16 rows merged through LDS (s must be the
// workgroup's): emit(row, d, O, L, M) for every row and dimension, O and L
// the sums scaled by exp(-M).  256 threads.
template <int HD> struct Merge16 {
    static constexpr int DR = HD < 128 ? HD : 128;
    float o[4][16][DR + 4], m[4][16], l[4][16];
};
template <int HD, typename Emit>
__device__ __forceinline__ void attn16_merge(const Attn16<HD> &a, Merge16<HD> &s, Emit emit)
{
    constexpr int DR = Merge16<HD>::DR;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, n = lane & 15, g = lane >> 4;
    const float l = groups_sum(a.l);
    if (g == 0) {
        s.m[wave][n] = a.m;
        s.l[wave][n] = l;
    }
#pragma unroll
    for (int d0 = 0; d0 < HD; d0 += DR) {
        __syncthreads();
        // element (j, e), register i: value 64 j + 4 (4 g + i) + e of query n
#pragma unroll
        for (int j = d0 / 64; j < (d0 + DR) / 64; j++)
#pragma unroll
            for (int i = 0; i < 4; i++)
                *(f4 *)&s.o[wave][n][64 * j - d0 + 4 * (4 * g + i)] =
                    f4{a.o[j][0][i], a.o[j][1][i], a.o[j][2][i], a.o[j][3][i]};
        __syncthreads();
        for (int i = threadIdx.x; i < 16 * DR; i += 256) {
            const int r = i / DR, d = i % DR;
            float M = s.m[0][r];
#pragma unroll
            for (int w = 1; w < 4; w++) M = fmaxf(M, s.m[w][r]);
            float L = 0.0f, O = 0.0f;
#pragma unroll
            for (int w = 0; w < 4; w++) {
                const float f = s.m[w][r] == -INFINITY ? 0.0f : expf(s.m[w][r] - M);
                L += s.l[w][r] * f;
                O += s.o[w][r][d] * f;
            }
            emit(r, d0 + d, O, L, M);
        }
    }
}

// Keys per workgroup of a launch of `groups` workgroups (16 query rows of one
// kv head each, `rows` rows in all) over n_t keys: all of them up to 256 (two
// blocks per wave: a merge kernel costs more), else a multiple of 128 (one
// block per wave) that makes at most 512 workgroups, two per CU, whose
// partials [rows][chunks][hd + 2] fit `floats`.
inline uint32_t attn_chunk_keys(uint64_t n_t, uint64_t groups, uint64_t rows, uint64_t hd, uint64_t floats)
{
    if (n_t <= REF_ATTN_WHOLE) return (uint32_t)n_t;
    const uint64_t most = std::min<uint64_t>(512 / std::min<uint64_t>(groups, 512), floats / (rows * (hd + 2)));
    if (most < 2) return (uint32_t)n_t;
    return (uint32_t)std::min<uint64_t>(n_t, (n_t + 128 * most - 1) / (128 * most) * 128);
}

// O[row][hd] from the chunks' partials {m, l, o[hd]}, part [rows][chunks][hd + 2];
// at most 512 chunks.
hipError_t launch_attn_merge(hipStream_t st, const float *part, float *O, int rows, int chunks, int hd);

}  // namespace styx
