// Dense weights [N][K] of packed layers, for products over many tokens.
//
// SqueezeLLM and LUT-GEMM keep neighbouring outputs next to each other and the product wants neighbouring channels, so a workgroup turns
// tiles of 64 outputs x 128 channels around in LDS: a lane owns an output and a wave 32 channels of it (the packed words of a
// wave are whole 256-byte rows), the tile leaves in 16-byte pieces, 256 bytes of an output's row at a time.  What is left is
// the write of the dense weight.  SqueezeLLM: the outputs' tables lie in LDS as [value][lane] (no bank conflicts), read once
// per tile; LUT-GEMM: the binary codes are summed in fp32, plane by plane, then the bias, and rounded once -- for 3 and 4 bits
// and groups of a multiple of 32 channels, the group's 8 or 16 values by that rule and the weights looked up (packed.h).
// Any-precision rows need no turning: a thread owns a word per plane, whose pieces of eight channels leave as they are.
//
// Measured (fp16, 4096 -> 28672, 235 MB dense): SqueezeLLM 4 bits 58 us (5.1 TB/s of packed reads and dense writes, a large
// copy's rate), LUT-GEMM 3 bits, group 128 59 us (sums for every weight: 109 us), any-precision 3 bits 43 us (values looked up one by
// one in memory: 82 us); torch operations on 64-bit indices took 2.3 and 20 ms for the first two.
#include "launch.h"
#include "packed.h"

namespace decdec {

constexpr uint32_t kTileN = 64, kTileK = 128;

// A lane's 32 dense channels, as 16-byte pieces, into the tile and the tile into the dense weight.
template <int DT>
struct DequantTile {
    using T = typename LaneOf<DT>::t;
    static constexpr uint32_t ROW = kTileK + 16u / sizeof(T);
    T v[kTileN * ROW];

    __device__ __forceinline__ void put(uint32_t wave, uint32_t lane, const T (&w)[32]) {
        u32x4 piece;
#pragma unroll
        for (uint32_t i = 0; i < 32u * sizeof(T) / 16u; ++i) {
            __builtin_memcpy(&piece, w + i * (16u / sizeof(T)), 16);
            *(u32x4*)(v + lane * ROW + 32u * wave + i * (16u / sizeof(T))) = piece;
        }
    }
    // K is a multiple of 32, so a piece lies inside a row or outside it
    __device__ __forceinline__ void leave(T* weight, uint32_t n0, uint32_t k0, uint32_t N, uint32_t K) const {
        constexpr uint32_t per = 16u / sizeof(T), pieces = kTileK / per;
        for (uint32_t i = threadIdx.x; i < kTileN * pieces; i += 256u) {
            const uint32_t n = i / pieces, c = i % pieces * per;
            if (n0 + n < N && k0 + c < K) *(u32x4*)(weight + (size_t)(n0 + n) * K + k0 + c) = *(const u32x4*)(v + n * ROW + c);
        }
    }
};

// grid (outputs / 64, shares of the tiles along K)
template <int DT, int BITS>
__global__ __launch_bounds__(256) void sqllm_dequant_kernel(const uint32_t* __restrict__ q, const void* __restrict__ lut,
                                                            void* __restrict__ weight, const uint32_t N, const uint32_t K) {
    using T = typename LaneOf<DT>::t;
    constexpr uint32_t V = 1u << BITS;
    __shared__ __align__(16) DequantTile<DT> tile;
    __shared__ uint32_t table[V][kTileN];
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6, n0 = blockIdx.x * kTileN;
    for (uint32_t i = threadIdx.x; i < V * kTileN; i += 256u) {
        const uint32_t n = n0 + i / V < N ? n0 + i / V : N - 1u;
        table[i % V][i / V] = Elem<DT>::load_raw(lut, (size_t)n * V + i % V);
    }
    const uint32_t col = n0 + lane < N ? n0 + lane : N - 1u, units = K / 32u;
    for (uint32_t k0 = blockIdx.y * kTileK; k0 < K; k0 += gridDim.y * kTileK) {
        const uint32_t u = k0 / 32u + wave;
        uint32_t w[BITS];
#pragma unroll
        for (uint32_t i = 0; i < (uint32_t)BITS; ++i) w[i] = q[(size_t)((u < units ? u : units - 1u) * BITS + i) * N + col];
        __syncthreads();                                   // the table is written, the tile before has left
        T out[32];
#pragma unroll
        for (uint32_t c = 0; c < 32u; ++c) {
            const uint32_t bit = c * BITS, word = bit / 32u, off = bit % 32u;
            uint32_t idx = w[word] >> off;
            if (off + BITS > 32u) idx |= w[word + 1u < (uint32_t)BITS ? word + 1u : word] << (32u - off);
            const uint32_t raw = table[idx & (V - 1u)][lane];
            __builtin_memcpy(&out[c], &raw, sizeof(T));
        }
        tile.put(wave, lane, out);
        __syncthreads();
        tile.leave((T*)weight, n0, k0, N, K);
    }
}

template <int DT, int BITS>
__global__ __launch_bounds__(256) void lutgemm_dequant_kernel(const uint32_t* __restrict__ q, const void* __restrict__ alpha,
                                                              const void* __restrict__ q_bias, void* __restrict__ weight,
                                                              const uint32_t N, const uint32_t K, const uint32_t group) {
    using T = typename LaneOf<DT>::t;
    using E = Elem<DT>;
    __shared__ __align__(16) DequantTile<DT> tile;
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6, n0 = blockIdx.x * kTileN;
    const uint32_t col = n0 + lane < N ? n0 + lane : N - 1u, units = K / 32u;
    for (uint32_t k0 = blockIdx.y * kTileK; k0 < K; k0 += gridDim.y * kTileK) {
        const uint32_t u = k0 / 32u + wave < units ? k0 / 32u + wave : units - 1u;
        uint32_t w[BITS];
#pragma unroll
        for (uint32_t p = 0; p < (uint32_t)BITS; ++p) w[p] = q[((size_t)u * BITS + p) * N + col];
        float a[BITS], b = 0.f;
        T out[32];
        uint32_t g = ~0u;
#pragma unroll
        for (uint32_t c = 0; c < 32u; ++c) {
            const uint32_t gc = (32u * u + c) / group;
            if (gc != g) {                                 // the same for the whole wave; once where groups are multiples of 32
                g = gc;
#pragma unroll
                for (uint32_t p = 0; p < (uint32_t)BITS; ++p) a[p] = E::load(alpha, ((size_t)g * BITS + p) * N + col);
                b = E::load(q_bias, (size_t)g * N + col);
            }
            float v = 0.f;
#pragma unroll
            for (uint32_t p = 0; p < (uint32_t)BITS; ++p) {
                const float s = __uint_as_float(__float_as_uint(a[p]) ^ (~(w[p] << (31u - c)) & 0x80000000u));   // bit 1: plus
                v = p == 0u ? s : v + s;
            }
            const uint32_t raw = E::to_raw(v + b);
            __builtin_memcpy(&out[c], &raw, sizeof(T));
        }
        __syncthreads();                                   // the tile before has left
        tile.put(wave, lane, out);
        __syncthreads();
        tile.leave((T*)weight, n0, k0, N, K);
    }
}

// 3 and 4 bits, 16-bit types, groups of a multiple of 32 channels.
template <int DT, int BITS>
__global__ __launch_bounds__(256) void lutgemm_lookup_kernel(const uint32_t* __restrict__ q, const void* __restrict__ alpha,
                                                             const void* __restrict__ q_bias, uint16_t* __restrict__ weight,
                                                             const uint32_t N, const uint32_t K, const uint32_t group) {
    using E = Elem<DT>;
    __shared__ __align__(16) DequantTile<DT> tile;
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6, n0 = blockIdx.x * kTileN;
    const uint32_t col = n0 + lane < N ? n0 + lane : N - 1u, units = K / 32u;
    for (uint32_t k0 = blockIdx.y * kTileK; k0 < K; k0 += gridDim.y * kTileK) {
        const uint32_t u = k0 / 32u + wave < units ? k0 / 32u + wave : units - 1u;
        const size_t g = 32u * u / group;
        uint32_t w[BITS];
        float a[BITS + 1];
#pragma unroll
        for (uint32_t p = 0; p < (uint32_t)BITS; ++p) {
            w[p] = q[((size_t)u * BITS + p) * N + col];
            a[p] = E::load(alpha, (g * BITS + p) * N + col);
        }
        a[BITS] = E::load(q_bias, g * N + col);
        u32x4 r[4];
        decode<kLutgemm, BITS>(w, group_tables<DT, BITS>(a), r);
        __syncthreads();                                   // the tile before has left
#pragma unroll
        for (uint32_t j = 0; j < 4u; ++j) *(u32x4*)(tile.v + lane * tile.ROW + 32u * wave + 8u * j) = r[j];
        __syncthreads();
        tile.leave(weight, n0, k0, N, K);
    }
}

// A thread per word of a row; 16-bit entries, moved bit for bit.
template <int BITS>
__global__ __launch_bounds__(256) void anyprec_lookup_kernel(const uint32_t* __restrict__ q, const uint16_t* __restrict__ lut,
                                                             uint16_t* __restrict__ weight, const uint32_t N, const uint32_t K) {
    const uint32_t W = K / 32u;
    const size_t id = (size_t)blockIdx.x * 256u + threadIdx.x;
    if (id >= (size_t)N * W) return;
    const uint32_t n = (uint32_t)(id / W), wi = (uint32_t)(id - (size_t)n * W), i = wi >> 5, t = wi & 31u;
    const uint32_t eff = (i == K / 1024u) ? (K % 1024u) / 32u : 32u;
    uint32_t w[BITS], e[1 << (BITS - 1)];
#pragma unroll
    for (int p = 0; p < BITS; ++p) w[p] = q[((size_t)p * N + n) * W + wi];
    const u32x4* row = (const u32x4*)(lut + (size_t)n * (1u << BITS));
#pragma unroll
    for (int k = 0; k < (1 << (BITS - 3)); ++k) {
        const u32x4 v = row[k];
#pragma unroll
        for (int j = 0; j < 4; ++j) e[4 * k + j] = v[j];
    }
    u32x4 r[4];
    decode<kAnyprec, BITS>(w, tables_of<BITS>(e), r);
    uint16_t* dst = weight + (size_t)n * K + 1024u * i + 8u * t;
#pragma unroll
    for (uint32_t j = 0; j < 4u; ++j) *(u32x4*)(dst + 8u * eff * j) = r[j];
}

// Enough workgroups for every compute unit's eight (a dense tile is 17 KB of LDS), each with as many tiles as that leaves.
static dim3 dequant_grid(uint32_t N, uint32_t K) {
    const uint32_t cols = (N + kTileN - 1u) / kTileN, tiles = (K + kTileK - 1u) / kTileK;
    uint32_t share = (2048u + cols - 1u) / cols;
    return dim3(cols, share < tiles ? share : tiles);
}

template <int DT>
static hipError_t sqllm_dt(int bits, const uint32_t* q, const void* lut, void* weight, uint32_t N, uint32_t K, hipStream_t s) {
    if (bits == 3) hipLaunchKernelGGL((sqllm_dequant_kernel<DT, 3>), dequant_grid(N, K), dim3(256), 0, s, q, lut, weight, N, K);
    else hipLaunchKernelGGL((sqllm_dequant_kernel<DT, 4>), dequant_grid(N, K), dim3(256), 0, s, q, lut, weight, N, K);
    return hipGetLastError();
}

hipError_t launch_sqllm_dequant(int dt, int bits, const uint32_t* q, const void* lut, void* weight, uint32_t N, uint32_t K, hipStream_t s) {
    if (dt == kFP32) return sqllm_dt<kFP32>(bits, q, lut, weight, N, K, s);
    return sqllm_dt<kFP16>(bits, q, lut, weight, N, K, s);   // 16-bit entries are copied bit for bit: one instance for both types
}

template <int DT>
static hipError_t lutgemm_dt(int bits, const uint32_t* q, const void* alpha, const void* q_bias, void* weight, uint32_t N, uint32_t K,
                             uint32_t group, hipStream_t s) {
    if constexpr (DT != kFP32) {
        if ((bits == 3 || bits == 4) && group % 32u == 0) {
            if (bits == 3) hipLaunchKernelGGL((lutgemm_lookup_kernel<DT, 3>), dequant_grid(N, K), dim3(256), 0, s, q, alpha, q_bias, (uint16_t*)weight, N, K, group);
            else hipLaunchKernelGGL((lutgemm_lookup_kernel<DT, 4>), dequant_grid(N, K), dim3(256), 0, s, q, alpha, q_bias, (uint16_t*)weight, N, K, group);
            return hipGetLastError();
        }
    }
#define DD_CASE(B) case B: hipLaunchKernelGGL((lutgemm_dequant_kernel<DT, B>), dequant_grid(N, K), dim3(256), 0, s, q, alpha, q_bias, weight, N, K, group); break
    switch (bits) { DD_CASE(1); DD_CASE(2); DD_CASE(3); DD_CASE(4); DD_CASE(5); DD_CASE(6); DD_CASE(7); DD_CASE(8); default: return hipErrorInvalidValue; }
#undef DD_CASE
    return hipGetLastError();
}

hipError_t launch_lutgemm_dequant(int dt, int bits, const uint32_t* q, const void* alpha, const void* q_bias, void* weight, uint32_t N,
                                  uint32_t K, uint32_t group, hipStream_t s) {
    if (dt == kFP32) return lutgemm_dt<kFP32>(bits, q, alpha, q_bias, weight, N, K, group, s);
    if (dt == kFP16) return lutgemm_dt<kFP16>(bits, q, alpha, q_bias, weight, N, K, group, s);
    return lutgemm_dt<kBF16>(bits, q, alpha, q_bias, weight, N, K, group, s);
}

hipError_t launch_anyprec_lookup(int bits, const uint32_t* q, const void* lut, void* weight, uint32_t N, uint32_t K, hipStream_t s) {
    const size_t words = (size_t)N * (K / 32u);
    const dim3 grid((uint32_t)((words + 255u) / 256u));
    if (bits == 3) hipLaunchKernelGGL((anyprec_lookup_kernel<3>), grid, dim3(256), 0, s, q, (const uint16_t*)lut, (uint16_t*)weight, N, K);
    else hipLaunchKernelGGL((anyprec_lookup_kernel<4>), grid, dim3(256), 0, s, q, (const uint16_t*)lut, (uint16_t*)weight, N, K);
    return hipGetLastError();
}

}  // namespace decdec
