// RMS norm of a row by one workgroup, as the row kernel and a product that norms its own input have it: the bits of one are those of the other.  A thread takes
// four neighbouring elements of each pass; statistics in fp32.
#pragma once
#include "anyprec_role.h"

namespace decdec {

template <int DT>
__device__ __forceinline__ u32x2 norm_pack(const float (&v)[4]) {
    using E = Elem<DT>;
    return u32x2{E::to_raw(v[0]) | (E::to_raw(v[1]) << 16), E::to_raw(v[2]) | (E::to_raw(v[3]) << 16)};
}

// v = x + y, rounded as storing it would, or x; 0 past the row's end.  Its squares go to `squares`.
template <int DT>
__device__ __forceinline__ void norm_add(u32x2 x, u32x2 y, bool have_y, bool in, float (&v)[4], float& squares) {
    using E = Elem<DT>;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const uint32_t sh = (e & 1) ? 16u : 0u;
        float a = E::from_raw((x[e >> 1] >> sh) & 0xFFFFu);
        if (have_y) a = E::from_raw(E::to_raw(a + E::from_raw((y[e >> 1] >> sh) & 0xFFFFu)));
        v[e] = in ? a : 0.f;
        squares += v[e] * v[e];
    }
}

// 1 / rms of the row whose squares the threads of `waves` waves hold; sums: a float a wave.
__device__ __forceinline__ float norm_factor(float squares, float* sums, uint32_t waves, uint32_t n, float eps) {
    const float s = wave_sum_dpp(squares);                  // total in lane 63
    if ((threadIdx.x & 63u) == 63u) sums[threadIdx.x >> 6] = s;
    __syncthreads();
    float all = 0.f;
    for (uint32_t w = 0; w < waves; ++w) all += sums[w];
    return __builtin_amdgcn_rsqf(all / (float)n + eps);
}

template <int DT>
__device__ __forceinline__ u32x2 norm_scaled(const float (&v)[4], float factor, u32x2 weight) {
    float o[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = v[e] * factor * Elem<DT>::from_raw((weight[e >> 1] >> ((e & 1) ? 16u : 0u)) & 0xFFFFu);
    return norm_pack<DT>(o);
}

}  // namespace decdec
