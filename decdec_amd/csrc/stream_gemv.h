// One-token products with a dense row-major weight: a stream of the weight.
//
// A workgroup of four waves owns two rows and its waves a quarter of their columns each: a lane requests 16 bytes of both rows per
// step (never reused, hence non-temporal; x comes through the vector cache), the next step before it uses the present one, and
// the quarters meet in LDS.  Bound by the read of the weight.  Quartered rows keep the requests of a compute unit inside few rows
// at a time and let a row of 14336 end four times as early as a wave of its own would; more rows or more steps per wave leave
// fewer waves for the same bytes.  us a launch (bf16; before: a wave owned four, two or one rows by their number, and converted
// its bf16 pairs one by one instead of v_dot2): 128256 x 4096 161 -> 150 (7.0 TB/s), 20480 x 4096 30.1 -> 26.6, 4096 x 14336 27.6 ->
// 20.7, 4096 x 4096 9.5 -> 7.6, 2048 x 7168 12.2 -> 7.1, 32000 x 2048 24.2 -> 21.1, 2048 x 2048 5.6 -> 3.8.
// v_dot2 in bf16 is no less exact than two fp32 multiply-adds (numbers below the normal ones and infinities included): over the shapes
// above the results differ from 64 bits by the same norm to six digits, and as many are not the rounded 64-bit sum (at most 5 in
// 10000); with multiply-adds 128256 x 4096 takes 149 us for 143.
#pragma once
#include "common.h"

namespace decdec {

constexpr uint32_t kStreamRows = 2, kStreamWaves = 4;

template <int DT>
__device__ __forceinline__ float stream_dot(const u32x4& w, const u32x4& x, float acc) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const uint32_t a = w[j], b = x[j];
        if constexpr (DT == kFP32) {
            acc = __builtin_fmaf(__uint_as_float(a), __uint_as_float(b), acc);
        } else if constexpr (DT == kFP16) {
            half2_t u, v;
            __builtin_memcpy(&u, &a, 4);
            __builtin_memcpy(&v, &b, 4);
            acc = __builtin_amdgcn_fdot2(u, v, acc, false);
        } else {
            bf16x2_t u, v;
            __builtin_memcpy(&u, &a, 4);
            __builtin_memcpy(&v, &b, 4);
            acc = __builtin_amdgcn_fdot2_f32_bf16(u, v, acc, false);
        }
    }
    return acc;
}

// finish(row, sum), by one lane per row; all four waves of the workgroup call this.  K a multiple of the elements in 16 bytes,
// weight and x 16-byte aligned.
template <int DT, typename F>
__device__ __forceinline__ void stream_gemv(const void* __restrict__ weight, const void* __restrict__ x, const uint32_t N,
                                            const uint32_t K, F finish) {
    constexpr uint32_t PE = 16u / Elem<DT>::bytes;
    __shared__ float parts[kStreamWaves][kStreamRows];
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6, row0 = blockIdx.x * kStreamRows;
    const unsigned char* wr[kStreamRows];
#pragma unroll
    for (uint32_t r = 0; r < kStreamRows; ++r) {
        const uint32_t rr = row0 + r < N ? row0 + r : N - 1u;              // rows past the end re-read the last one; not stored
        wr[r] = (const unsigned char*)weight + (size_t)rr * K * Elem<DT>::bytes;
    }
    const uint32_t steps = (K + 64u * PE - 1u) / (64u * PE), per = (steps + kStreamWaves - 1u) / kStreamWaves;
    const uint32_t s0 = wave * per, s1 = s0 + per < steps ? s0 + per : steps;
    u32x4 wv[2][kStreamRows], xv[2];
    float acc[kStreamRows] = {};
    auto request = [&](int b, uint32_t s) {
        const uint32_t col = (s * 64u + lane) * PE;
        const size_t c = (size_t)(col < K ? col : 0u) * Elem<DT>::bytes;
        xv[b] = *(const u32x4*)((const unsigned char*)x + c);
#pragma unroll
        for (uint32_t r = 0; r < kStreamRows; ++r) wv[b][r] = __builtin_nontemporal_load((const u32x4*)(wr[r] + c));
    };
    auto use = [&](int b, uint32_t s) {
        if ((s + 1u) * 64u * PE > K && (s * 64u + lane) * PE >= K) {       // lanes past the end of a row's last step
            xv[b] = u32x4{0u, 0u, 0u, 0u};
#pragma unroll
            for (uint32_t r = 0; r < kStreamRows; ++r) wv[b][r] = u32x4{0u, 0u, 0u, 0u};
        }
#pragma unroll
        for (uint32_t r = 0; r < kStreamRows; ++r) acc[r] = stream_dot<DT>(wv[b][r], xv[b], acc[r]);
    };
    if (s0 < s1) request(0, s0);
    uint32_t s = s0;
    for (; s + 1u < s1; s += 2u) {
        request(1, s + 1u);
        use(0, s);
        if (s + 2u < s1) request(0, s + 2u);
        use(1, s + 1u);
    }
    if (s < s1) use(0, s);
#pragma unroll
    for (uint32_t r = 0; r < kStreamRows; ++r) acc[r] = wave_sum(acc[r]);
    if (lane == 0u)
#pragma unroll
        for (uint32_t r = 0; r < kStreamRows; ++r) parts[wave][r] = acc[r];
    __syncthreads();
    if (threadIdx.x < kStreamRows && row0 + threadIdx.x < N) {
        float v = 0.f;
#pragma unroll
        for (uint32_t w = 0; w < kStreamWaves; ++w) v += parts[w][threadIdx.x];
        finish(row0 + threadIdx.x, v);
    }
}

}  // namespace decdec
