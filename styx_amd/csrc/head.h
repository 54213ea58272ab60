// head.h -- per-head RMSNorm and NEOX rope of one q or k head by one wave,
// shared by the decode attention kernels and the prompt kernels so that both
// form a head's values with the same arithmetic.
#pragma once

#include "qdot.h"

namespace styx {

// One head's RMSNorm(hd) * w and NEOX rope at pos, split into a load phase
// (every operand of the head issued at once) and a compute phase, so a wave
// can have all its heads' loads in flight together.  Lane l owns the rope
// pairs (i, i + hd/2) for i = l + 64 j, j < PPL; cs points at the (cos, sin)
// row of the position.
template <int PPL> struct HeadIn {
    float x0[PPL], x1[PPL], w0[PPL], w1[PPL];
};

template <int PPL>
__device__ __forceinline__ void head_load(HeadIn<PPL> &h, const float *src, const float *w, int hd)
{
    const int lane = threadIdx.x & 63, half = hd / 2;
#pragma unroll
    for (int j = 0; j < PPL; j++) {
        const int i = lane + 64 * j;
        const bool ok = i < half;
        h.x0[j] = ok ? src[i] : 0.0f;
        h.x1[j] = ok ? src[i + half] : 0.0f;
        h.w0[j] = (ok && w) ? w[i] : 1.0f;
        h.w1[j] = (ok && w) ? w[i + half] : 1.0f;
    }
}

// head_load for head_dim 128 with one pair per lane: every load issued
// unconditionally (without norm weights, the weights' loads read the head
// itself and are replaced by 1)
template <int PPL>
__device__ __forceinline__ void head_load_all(HeadIn<PPL> &h, const float *src, const float *w, int hd)
{
    static_assert(PPL == 1, "one rope pair per lane");
    const int lane = threadIdx.x & 63, half = hd / 2;
    const float *ws = w ? w : src;
    h.x0[0] = src[lane];
    h.x1[0] = src[lane + half];
    const float w0 = ws[lane], w1 = ws[lane + half];
    h.w0[0] = w ? w0 : 1.0f;
    h.w1[0] = w ? w1 : 1.0f;
}

template <int PPL>
__device__ __forceinline__ void cs_load(double2 *cs, const double2 *row, int hd)
{
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int j = 0; j < PPL; j++) {
        const int i = lane + 64 * j;
        cs[j] = i < hd / 2 ? row[i] : make_double2(1.0, 0.0);
    }
}

template <int PPL>
__device__ __forceinline__ void head_finish(const HeadIn<PPL> &h, const double2 *cs, bool norm,
                                            float eps, int hd, float *dst)
{
    const int lane = threadIdx.x & 63, half = hd / 2;
    float ss = 0.0f;
#pragma unroll
    for (int j = 0; j < PPL; j++) ss += h.x0[j] * h.x0[j] + h.x1[j] * h.x1[j];
    ss = wave_sum(ss);
    const float scale = norm ? 1.0f / sqrtf(ss / (float)hd + eps) : 1.0f;
#pragma unroll
    for (int j = 0; j < PPL; j++) {
        const int i = lane + 64 * j;
        if (i >= half) continue;
        float x0 = h.x0[j], x1 = h.x1[j];
        if (norm) {
            x0 = (x0 * scale) * h.w0[j];
            x1 = (x1 * scale) * h.w1[j];
        }
        const double c = cs[j].x, sn = cs[j].y;
        dst[i] = (float)((double)x0 * c - (double)x1 * sn);
        dst[i + half] = (float)((double)x0 * sn + (double)x1 * c);
    }
}

}  // namespace styx
