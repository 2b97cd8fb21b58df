// The positive maps of the Gaussian exponents and the merging of their statistics.
#pragma once
#include "cf_common.h"

namespace cf {

__device__ __forceinline__ float positive_map(float x, int func, float beta, float lb)
{
    // models/indexed_lattice_multi_head_attention_cuda.py:675-692
    if (func == 0) {            // elu
        const float t = x * (beta / (1.0f - lb));
        return (1.0f - lb) * (t > 0.f ? t : expf(t) - 1.0f) + 1.0f;
    }
    if (func == 1) return (1.0f - lb) * fabsf(x) + lb;           // abs
    return (1.0f - lb) * expf(x * (beta / (1.0f - lb))) + lb;   // exp
}

__device__ __forceinline__ float positive_map_slope(float x, int func, float beta, float lb)
{
    if (func == 0) {            // elu
        const float t = x * (beta / (1.0f - lb));
        return (t > 0.f ? 1.0f : expf(t)) * beta;
    }
    if (func == 1) return (x > 0.f ? 1.0f : (x < 0.f ? -1.0f : 0.f)) * (1.0f - lb);   // abs
    return expf(x * (beta / (1.0f - lb))) * beta;                                      // exp
}

// Chan's pairwise update of (count, mean, M2).
__device__ __forceinline__ void stat_merge(float &n, float &mean, float &m2, float nb, float meanb, float m2b)
{
    const float nt = n + nb;
    if (nt == 0.f) return;
    const float delta = meanb - mean;
    mean += delta * (nb / nt);
    m2 += m2b + delta * delta * (n * nb / nt);
    n = nt;
}

// (count, mean, M2) of all blocks, three floats each (`part(i)` is the i-th), by one wavefront in one fixed order;
// the same in every lane.
template <class Part>
__device__ __forceinline__ void merge_statistics_of(Part part, int blocks, int lane, float &n, float &mean, float &m2)
{
    n = mean = m2 = 0.f;
    for (int b = lane; b < blocks; b += WAVE) stat_merge(n, mean, m2, part(3 * b), part(3 * b + 1), part(3 * b + 2));
#pragma unroll
    for (int off = 1; off < WAVE; off <<= 1) {
        const float nb = __shfl_xor(n, off, WAVE), mb = __shfl_xor(mean, off, WAVE),
                    qb = __shfl_xor(m2, off, WAVE);
        // lower lane first on both sides so partners agree bit for bit
        float n0 = (lane & off) ? nb : n, m0 = (lane & off) ? mb : mean, q0 = (lane & off) ? qb : m2;
        const float n1 = (lane & off) ? n : nb, m1 = (lane & off) ? mean : mb, q1 = (lane & off) ? m2 : qb;
        stat_merge(n0, m0, q0, n1, m1, q1);
        n = n0; mean = m0; m2 = q0;
    }
}

__device__ __forceinline__ void merge_statistics(const float *part, int blocks, int lane, float &n, float &mean, float &m2)
{
    merge_statistics_of([=](int i) { return part[i]; }, blocks, lane, n, mean, m2);
}

}  // namespace cf
