// What the kernels of products with packed weights share.
#pragma once
#include "launch.h"
#include "packed.h"

namespace decdec {

struct QgemmParams {
    const void* x;                 // [M][K]
    const uint32_t* q;
    const void* lut;               // tables [N][2^bits], or the scales [K / group][bits][N] of LUT-GEMM
    const void* q_bias;            // [K / group][N]
    void* out;                     // [M][N]
    float* part;                   // [split tile][ks][wave column][16-token tile][its two 16-output fragments][lane][4]
    uint32_t M, N, K, group;
    uint32_t groups, z;            // column groups and token tiles
    uint32_t wk, whole, ks;        // ranges of channels inside a workgroup; tiles with one workgroup; workgroups of a tile behind them
    uint32_t blocks, ks_blocks;    // blocks of 16 units in a range: of a whole tile, of a split one
    uint32_t wide;                 // whole pieces of results may be stored at once
    // 0, or N / 2 (a multiple of 8): columns are gates and, `half` further, what they gate, and out [M][half] is silu(gate) * up of both rounded.  A
    // wave's two fragments of sixteen outputs are then sixteen gates and their sixteen partners, so that a lane has both.  4096 -> 28672, 512 tokens,
    // SqueezeLLM 4 bits: 121 us (traced; half as much is stored), 127 and 10 for the gates by a kernel of their own; 5120 -> 35840, 77 tokens, LUT-GEMM 3 bits: 51
    // and, for the sums of shares, 5, that kernel's 5 saved.
    uint32_t half;
    // With `half`: the wave columns that hold gates and partners, all (~0) where all columns are dealt the same way.  Of tiles with one workgroup and tiles with
    // several beside each other a column stays with its kind, so that its sum has the order, and the bits, of the product alone: pairs where gate and partner are of
    // whole tiles, then, up to wave column `wholes`, 32 gates each, stored rounded, whose partners are behind in split tiles, and meet them where the shares are added.
    uint32_t pairs, wholes;
};

// Unit of lane group g in packet i of a block.  LUT-GEMM: a lane stays in one group of 128 channels for a block, and builds its table once.
template <int FMT>
__device__ __forceinline__ uint32_t unit_of(uint32_t block, uint32_t i, uint32_t g) {
    return 16u * block + (FMT == kAnyprec ? 8u * (i >> 1) + 2u * g + (i & 1u) : FMT == kLutgemm ? 4u * g + i : 4u * i + g);
}

// A wave's columns n0 .. end and the lane's two past `nb`; columns past the end repeat the last one and are not stored.
struct QgemmColumns { bool gated; uint32_t n0, end, nb, col[2]; };
__device__ __forceinline__ QgemmColumns qgemm_columns(const QgemmParams& p, uint32_t wave_column, uint32_t l16) {
    QgemmColumns c;
    c.gated = wave_column < p.pairs;
    const bool gates = !c.gated && wave_column < p.wholes;
    c.n0 = c.gated ? 16u * wave_column : 32u * wave_column - (gates ? 16u * p.pairs : 0u);
    c.end = c.gated || gates ? p.half : p.N;
    c.nb = c.n0 < c.end ? c.n0 : c.end - 1u;
#pragma unroll
    for (uint32_t b = 0; b < 2u; ++b) {
        const uint32_t n = c.n0 + l16 + (c.gated ? 0u : 16u * b);
        c.col[b] = (n < c.end ? n : c.end - 1u) - c.nb + (c.gated ? b * p.half : 0u);
    }
    return c;
}

// silu(gate) * up of numbers that are rounded first, as storing them and reading them back would; storage bits of two neighbours.  fp16: the last product
// is rounded once, by the instruction that the kernel of gates alone (silu_mul_rows_kernel) has there; left to itself the compiler rounds to 32 bits first in some places.
template <int DT>
__device__ __forceinline__ uint32_t gated2(float g0, float u0, float g1, float u1) {
    using E = Elem<DT>;
    const float a0 = E::from_raw(E::to_raw(g0)), a1 = E::from_raw(E::to_raw(g1));
    const float s0 = a0 / (1.f + __expf(-a0)), s1 = a1 / (1.f + __expf(-a1));
    const uint32_t b0 = E::to_raw(u0), b1 = E::to_raw(u1);
    if constexpr (DT == kFP16) {
        uint32_t d = 0u;
        asm("v_fma_mixlo_f16 %0, %1, %2, 0 op_sel_hi:[0,1,0]" : "+v"(d) : "v"(s0), "v"(b0));
        asm("v_fma_mixhi_f16 %0, %1, %2, 0 op_sel_hi:[0,1,0]" : "+v"(d) : "v"(s1), "v"(b1));
        return d;
    } else {
        return E::to_raw(s0 * E::from_raw(b0)) | (E::to_raw(s1 * E::from_raw(b1)) << 16);
    }
}

// A wave's pairs, gated: its MT x 16 tokens from m0 on.
template <int DT, int MT>
__device__ __forceinline__ void store_gated(const QgemmParams& p, const QgemmColumns& c, const f32x4 (&acc)[MT][2], uint32_t m0, uint32_t l16, uint32_t lg) {
#pragma unroll
    for (int m = 0; m < MT; ++m) {
        const uint32_t row = m0 + 16u * m + l16, n = c.n0 + 4u * lg;
        if (row >= p.M || n >= c.end) continue;
        const f32x4 g = acc[m][0], u = acc[m][1];
        *(u32x2*)((uint16_t*)p.out + (size_t)row * p.half + n) = u32x2{gated2<DT>(g[0], u[0], g[1], u[1]), gated2<DT>(g[2], u[2], g[3], u[3])};
    }
}

constexpr uint32_t kXRow = 256u;                                                       // bytes of a staged token: four units

// Tiles of 256 tokens x 256 outputs (k_qgemm_wide.hip): whether a product takes them, and its launch.
bool qgemm_goes_wide(int fmt, int bits, uint32_t M, uint32_t N, uint32_t K, uint32_t group);
hipError_t launch_qgemm_wide(int fmt, int dt, int bits, QgemmParams p, hipStream_t s);

}  // namespace decdec
