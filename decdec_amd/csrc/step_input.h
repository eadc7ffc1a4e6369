// What a one-token product multiplies, made by the product itself out of what the launches before it left: the residual stream and its norm, or a
// gate and what it gates.  Every workgroup (1024 threads) makes the activations of its own channels, in LDS, while its first weights are on their way.
#pragma once
#include "norm_row.h"

namespace decdec {

enum { kPlainInput = 0, kNormInput = 1, kGateInput = 2 };

// norm: activations = rms_norm(a + y) * weight (y null: of a), as add_rmsnorm_kernel has them; the first workgroup leaves a + y in h_out.
// gate: a [2 K], activations = silu(the first half) * the second.
struct StepInput {
    const void* a;
    const void* y;
    const void* weight;
    void* h_out;
    float eps;
};

constexpr uint32_t kStepSumsBytes = 16u * 4u;              // LDS of a norm's sums of squares, beside the dynamic part

// Between `request` and `finish` are the loads' round trips; `finish` leaves channels k0 .. k1 - 1 in `xl`, two a dword, for use behind a barrier.
// A thread takes four neighbouring channels of a norm in each of PASSES.
template <int DT, int KIND, int PASSES>
struct StepActivations {
    using E = Elem<DT>;
    u32x2 xr[PASSES], yr[PASSES], wr[PASSES];
    uint32_t g, u;

    __device__ __forceinline__ void request(const StepInput& in, uint32_t K, uint32_t k0, uint32_t k1) {
        const uint32_t tid = threadIdx.x;
        if constexpr (KIND == kNormInput) {
#pragma unroll
            for (int k = 0; k < PASSES; ++k) {
                const uint32_t i = 4u * (tid + (uint32_t)k * 1024u), ic = i + 4u <= K ? i : 0u;      // past the end: read, never used
                xr[k] = *(const u32x2*)((const uint16_t*)in.a + ic);
                yr[k] = in.y != nullptr ? *(const u32x2*)((const uint16_t*)in.y + ic) : u32x2{0u, 0u};
                wr[k] = *(const u32x2*)((const uint16_t*)in.weight + ic);
            }
        } else {
            const uint32_t t = 2u * tid < k1 - k0 ? tid : 0u;
            g = ((const uint32_t*)in.a)[(k0 >> 1) + t];
            u = ((const uint32_t*)in.a)[((K + k0) >> 1) + t];
        }
    }

    __device__ __forceinline__ void finish(const StepInput& in, uint32_t K, uint32_t k0, uint32_t k1, uint32_t* xl) {
        const uint32_t tid = threadIdx.x;
        if constexpr (KIND == kNormInput) {
            __shared__ float wsum[kStepSumsBytes / 4u];
            const bool have_y = in.y != nullptr;
            float v[PASSES][4], ss = 0.f;
#pragma unroll
            for (int k = 0; k < PASSES; ++k) {
                const uint32_t i = 4u * (tid + (uint32_t)k * 1024u);
                const bool ok = i + 4u <= K;
                norm_add<DT>(xr[k], yr[k], have_y, ok, v[k], ss);
                if (ok && have_y && blockIdx.x == 0u) *(u32x2*)((uint16_t*)in.h_out + i) = norm_pack<DT>(v[k]);
            }
            const float r = norm_factor(ss, wsum, 16u, K, in.eps);
#pragma unroll
            for (int k = 0; k < PASSES; ++k) {
                const uint32_t i = 4u * (tid + (uint32_t)k * 1024u);
                if (i < k0 || i >= k1) continue;            // ranges are multiples of 32 channels
                *(u32x2*)(xl + ((i - k0) >> 1)) = norm_scaled<DT>(v[k], r, wr[k]);
            }
        } else {
            for (uint32_t t = tid; 2u * t < k1 - k0; t += 1024u) {
                if (t != tid) {
                    g = ((const uint32_t*)in.a)[(k0 >> 1) + t];
                    u = ((const uint32_t*)in.a)[((K + k0) >> 1) + t];
                }
                uint32_t out = 0u;
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    const float a = E::from_raw((g >> (16 * e)) & 0xFFFFu), b = E::from_raw((u >> (16 * e)) & 0xFFFFu);
                    out |= E::to_raw(a / (1.f + __expf(-a)) * b) << (16 * e);
                }
                xl[t] = out;
            }
        }
    }
};

}  // namespace decdec
