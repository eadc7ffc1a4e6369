// fp32 numbers as three bf16 pieces (k_rowgemm.hip says what they hold), shared by the kernels that multiply them.
#pragma once
#include "mma.h"

namespace decdec {

// Eight elements as bf16 pieces; most: the largest size so far.
__device__ __forceinline__ void pieces_of(const Frag<kFP32>& f, u32x4 (&p)[3], float& most) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float x = f.v[2 * i], y = f.v[2 * i + 1];
        const uint32_t a = pack_bf16(x, y);
        const float u = x - __uint_as_float(a << 16), v = y - __uint_as_float(a & 0xFFFF0000u);
        const uint32_t b = pack_bf16(u, v);
        p[0][i] = a;
        p[1][i] = b;
        p[2][i] = pack_bf16(u - __uint_as_float(b << 16), v - __uint_as_float(b & 0xFFFF0000u));
        most = fmaxf(most, fmaxf(fabsf(x), fabsf(y)));
    }
}

// acc(i) += a[i] . b without the three products below 2^-24 of the largest: one product of all outputs after the other, the small ones first.
template <int TN, typename F>
__device__ __forceinline__ void six_products(const u32x4 (&a)[TN][3], const u32x4 (&b)[3], F acc) {
    constexpr int of_a[6] = {2, 0, 1, 1, 0, 0}, of_b[6] = {0, 2, 1, 0, 1, 0};
#pragma unroll
    for (int s = 0; s < 6; ++s)
#pragma unroll
        for (int i = 0; i < TN; ++i) {
            Frag<kBF16> f, x;
            f.v = a[i][of_a[s]];
            x.v = b[of_b[s]];
            mma(f, x, acc(i));
        }
}

// Whether three pieces hold the numbers of a row that the four lanes apart by s and t have seen, `most` the largest size of a lane's.
__device__ __forceinline__ bool in_three_pieces(float most, int s, int t) {
    most = fmaxf(most, __shfl_xor(most, s, 64));
    most = fmaxf(most, __shfl_xor(most, t, 64));
    return !(most > 3.3e38f || (most > 0.f && most < 1.2621774e-29f));
}

}  // namespace decdec
