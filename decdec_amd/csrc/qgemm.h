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
};

// Unit of lane group g in packet i of a block.  LUT-GEMM: a lane stays in one group of 128 channels for a block, and builds its table once.
template <int FMT>
__device__ __forceinline__ uint32_t unit_of(uint32_t block, uint32_t i, uint32_t g) {
    return 16u * block + (FMT == kAnyprec ? 8u * (i >> 1) + 2u * g + (i & 1u) : FMT == kLutgemm ? 4u * g + i : 4u * i + g);
}

constexpr uint32_t kXRow = 256u;                                                       // bytes of a staged token: four units

// Tiles of 256 tokens x 256 outputs (k_qgemm_wide.hip): whether a product takes them, and its launch.
bool qgemm_goes_wide(int fmt, int bits, uint32_t M, uint32_t N, uint32_t K, uint32_t group);
hipError_t launch_qgemm_wide(int fmt, int dt, int bits, QgemmParams p, hipStream_t s);

}  // namespace decdec
