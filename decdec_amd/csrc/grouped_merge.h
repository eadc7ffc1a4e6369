// Grouped attention of one token: how the sequence is shared, and the merge of the shares, which runs in a launch of its own or beside a
// recurrence that reads the same projections.
#pragma once
#include "mixers.h"

namespace decdec {

// Keys of a workgroup's pass; why 128: k_attention.hip.
constexpr uint32_t kGroupedUnit = 128;
// Shares of the earlier keys, a workgroup's pass at a time; max_splits workgroups at most, one at least (it holds
// the new token).
struct GroupedSplit { uint32_t splits, span; };
__host__ __device__ inline GroupedSplit grouped_split(uint32_t keys, uint32_t max_splits) {
    const uint32_t tiles = (keys + kGroupedUnit - 1u) / kGroupedUnit, per = tiles == 0u ? 1u : (tiles + max_splits - 1u) / max_splits;
    return {tiles == 0u ? 1u : (tiles + per - 1u) / per, per * kGroupedUnit};
}
constexpr uint32_t kGroupedSplits = 128;

// Merge of one head's shares, sink and gate, by 1024 threads: `groups` ranges of the shares, Vp threads each.
template <int DT>
__device__ __forceinline__ void grouped_merge(const GroupedMerge& p, const uint32_t h, float (&share)[1024], float (&ws)[kGroupedSplits]) {
    using E = Elem<DT>;
    const uint32_t tid = threadIdx.x, lane = tid & 63u, V = p.vdim;
    const long long pos = *p.pos;
    if (pos < 0 || pos >= (long long)p.max_seq) return;
    const uint32_t n = grouped_split((uint32_t)pos, p.max_splits).splits;
    const float* ph = p.parts + (size_t)h * (V + 2u);
    const size_t ps = (size_t)p.heads * (V + 2u);
    const uint32_t Vp = (V + 63u) & ~63u, groups = 1024u / Vp, g = tid / Vp, d = tid - g * Vp;
    if (tid < 64u) {
        const float sink = p.sink * kLog2e;
        float m[2], l[2], M = sink;
#pragma unroll
        for (uint32_t e = 0; e < 2u; ++e) {
            const uint32_t i = lane + 64u * e;
            m[e] = i < n ? ph[i * ps + V] : -__builtin_inff();
            l[e] = i < n ? ph[i * ps + V + 1u] : 0.f;
            M = fmaxf(M, m[e]);
        }
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) M = fmaxf(M, __shfl_xor(M, off, 64));
#pragma unroll
        for (int e = 0; e < 2; ++e) m[e] = __builtin_amdgcn_exp2f(m[e] - M);
        const float L = wave_sum(m[0] * l[0] + m[1] * l[1]) + __builtin_amdgcn_exp2f(sink - M);
        const float r = p.out_scale * (p.gates ? sigmoid_f(E::load(p.gates, p.off_g + h)) : 1.f) / L;
        ws[lane] = m[0] * r;
        ws[lane + 64u] = m[1] * r;
    }
    __syncthreads();
    float t = 0.f;
    if (g < groups && d < V) {
        for (uint32_t s = g; s < n; s += 4u * groups) {
            float x[4];
#pragma unroll
            for (uint32_t e = 0; e < 4u; ++e) x[e] = s + e * groups < n ? ph[(s + e * groups) * ps + d] : 0.f;
#pragma unroll
            for (uint32_t e = 0; e < 4u; ++e) t = __builtin_fmaf(s + e * groups < n ? ws[s + e * groups] : 0.f, x[e], t);
        }
    }
    share[tid] = t;
    __syncthreads();
    if (tid < V) {
        float a = 0.f;
        for (uint32_t k = 0; k < groups; ++k) a += share[k * Vp + tid];
        E::store(p.out, h * V + tid, a);
    }
}

}  // namespace decdec
