// Products of 129 and more tokens with a packed weight (SqueezeLLM, 3-bit LUT-GEMM), for layers whose tiles of 256 tokens x 256 outputs fill
// the compute units: a weight is decoded once for up to 256 tokens, where the tiles of qgemm_tile.h decode it for 128.
//
// Eight waves, 32 outputs each; fragments, units and packets as in qgemm_tile.h.  A packet of all tokens (64 KB for 256) comes to LDS by copies
// that pass no register, while the one before it is multiplied; sums take 128 registers of a lane.  There are as many blocks of 512
// channels as the layer has: no remainders, no ranges of channels.  The two waves of a SIMD take turns: one decodes a packet while the other
// multiplies.
//
// What bounds it: products (1.13 PFLOP/s at 512 tokens of bf16, and what normal numbers let the matrix units reach is about 1.3,
// k_splitgemm.hip): counted, 4096 of a packet's 5800 cycles, beside vector instructions on 53 % of the cycles and reads of their operands on 35 % of LDS's.  us, 4096 -> 28672, fp16, beside all waves in step
// (and tiles of 128 tokens): SqueezeLLM 4 bits 260 tokens 83 / 88, 384 91 / 98, 448 99 / 113, 512 110 / 128 (bf16 106 / 125); 3 bits 76 / 83, 85 / 92 and, at 512,
// 106 / 122; LUT-GEMM 3 bits 78 / 85, 88 / 94, 99 / 106.  Waves in step decode at the same time, and a SIMD's matrix unit waits for both.
// Copies of the first waves ahead of their products: 1 % more; wave priorities: the same.
//
// Registers: words of two packets, not four, and addresses that stay a scalar and 32 bits of a lane make room for a packet decoded ahead of its
// products with 16 tiles of tokens.  LUT-GEMM's 16 tiles stay narrow.
#include "qgemm.h"

namespace decdec {

template <int FMT, int BITS, int DT, int MT>
__global__ __attribute__((amdgpu_flat_work_group_size(512, 512), amdgpu_waves_per_eu(2, 2))) void qgemm_wide_kernel(const QgemmParams p) {
    constexpr uint32_t ROWS = 16u * MT, BUFFER = ROWS * kXRow, ROUNDS = ROWS / 32u;                // MT is even
    extern __shared__ __align__(1024) unsigned char smem[];      // [2][token][256]
    const uint32_t lane = threadIdx.x & 63u, wn = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l16 = lane & 15u, lg = lane >> 4;
    const bool second = wn >= 4u;                          // of the two waves of a SIMD
    const uint32_t N = p.N, tile = blockIdx.x;
    // token tiles of the same columns follow each other on one die
    const uint32_t cg = p.z == 1u ? tile : tile / (8u * p.z) * 8u + tile % 8u, zt = p.z == 1u ? 0u : tile / 8u % p.z;
    if (cg >= p.groups) return;
    const uint32_t m0 = zt * ROWS, blocks = p.K / 512u;
    const QgemmColumns columns = qgemm_columns(p, cg * 8u + wn, l16);
    const uint32_t n0 = columns.n0, nb = columns.nb;
    const uint32_t (&col)[2] = columns.col;
    Tables<BITS> tab[2];
    if constexpr (FMT != kLutgemm) {
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            uint32_t e[1 << (BITS - 1)];
            const u32x4* row = (const u32x4*)((const uint16_t*)p.lut + (size_t)(nb + col[b]) * (1u << BITS));
#pragma unroll
            for (int i = 0; i < (1 << (BITS - 3)); ++i) {
                const u32x4 v = row[i];
#pragma unroll
                for (int k = 0; k < 4; ++k) e[4 * i + k] = v[k];
            }
            tab[b] = tables_of<BITS>(e);
        }
    }
    // words of two packets, [packet][word][column]: one is requested as soon as the one before the last is decoded
    uint32_t w[2][BITS][2];
    auto request = [&](uint32_t block, uint32_t i) {
        const uint32_t step = FMT == kLutgemm ? 4u : 1u;
        asm volatile("" : "+s"(block));                    // addresses stay a scalar and a lane's 32 bits: carried from block to block in 64 they fill the registers
        const uint32_t* row = p.q + (size_t)unit_of<FMT>(block, i, 0u) * BITS * N + nb;
#pragma unroll
        for (uint32_t k = 0; k < (uint32_t)BITS; ++k, row += N)
#pragma unroll
            for (int b = 0; b < 2; ++b) w[i & 1u][k][b] = *(const uint32_t*)((const char*)row + 4u * (step * lg * (uint32_t)BITS * N + col[b]));
    };
    uint32_t sc[BITS + 1][2];
    auto request_scales = [&](uint32_t block) {
        if constexpr (FMT == kLutgemm) {
            const size_t gr = unit_of<FMT>(block, 0u, lg) / (p.group / 32u);
#pragma unroll
            for (uint32_t k = 0; k <= (uint32_t)BITS; ++k) {
                const uint16_t* row = (k < (uint32_t)BITS ? (const uint16_t*)p.lut + (gr * BITS + k) * N : (const uint16_t*)p.q_bias + gr * N) + nb;
#pragma unroll
                for (int b = 0; b < 2; ++b) sc[k][b] = row[col[b]];
            }
        }
    };
    // A copy is 4 tokens x 256 bytes; piece q of token m lies at q ^ (m - 4), so that a lane copies the piece that belongs where it writes.
    // Tokens past the end repeat the last one and are not stored.
    const uint32_t sub = lane >> 4, xq = l16 ^ ((4u * (wn & 3u) + sub + 12u) & 15u);
    uint32_t xoff[ROUNDS];
#pragma unroll
    for (uint32_t t = 0; t < ROUNDS; ++t) {
        const uint32_t m = 32u * t + 4u * wn + sub;
        xoff[t] = (m0 + m < p.M ? m : p.M - 1u - m0) * p.K * 2u + 64u * unit_of<FMT>(0u, 0u, xq >> 2) + 16u * (xq & 3u);
    }
    const unsigned char* xb = (const unsigned char*)p.x + (size_t)m0 * p.K * 2u;
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)smem;
    auto request_x = [&](uint32_t block, uint32_t i, uint32_t buf) {
        const unsigned char* from = xb + (size_t)64u * unit_of<FMT>(block, i, 0u);
#pragma unroll
        for (uint32_t t = 0; t < ROUNDS; ++t) {
            const uint32_t to = lds0 + buf * BUFFER + (32u * t + 4u * wn) * kXRow;
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                         : : "s"(__builtin_amdgcn_readfirstlane(to)), "v"(xoff[t]), "s"(from) : "memory");
        }
    };
    f32x4 acc[MT][2];
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[m][0] = acc[m][1] = f32x4{0.f, 0.f, 0.f, 0.f};
    const uint32_t frag_at = l16 * kXRow + (((4u * lg) ^ ((l16 + 12u) & 15u)) << 4);
    // Behind the last products: they may stand behind the barrier, but their operands have to be there before it, where the other waves go on to
    // copy to the buffer.
    auto turn = [&] {
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    };
    request_scales(0u);
    request_x(0u, 0u, 0u);
    request(0u, 0u);
    __builtin_amdgcn_sched_barrier(0);                     // requests in this order: a wait counts what is behind the one that is waited for
    request(0u, 1u);
    if (second) {                                          // half a packet behind the first
        asm volatile("s_waitcnt vmcnt(%0)" : : "n"(4 * BITS) : "memory");
        turn();
    }
    for (uint32_t block = 0; block < blocks; ++block) {
        const uint32_t next = block + 1u < blocks ? block + 1u : block;     // what is requested past the last packet is not used
#pragma unroll
        for (uint32_t i = 0; i < 4u; ++i) {
            const unsigned char* xs = smem + (i & 1u) * BUFFER;
            // The next packet's copies go to the buffer of the packet before, which all waves are done with when the second come to decode
            // and the first to multiply.
            if (second) request_x(i < 3u ? block : next, (i + 1u) & 3u, (i + 1u) & 1u);
            if constexpr (FMT == kLutgemm) {
                if (i == 0u) {
#pragma unroll
                    for (int b = 0; b < 2; ++b) {
                        float a[BITS + 1];
#pragma unroll
                        for (int k = 0; k <= BITS; ++k) a[k] = Elem<DT>::from_raw(sc[k][b]);
                        tab[b] = group_tables<DT, BITS>(a);
                    }
                    request_scales(next);
                }
            }
            uint32_t u[2][BITS];
#pragma unroll
            for (int b = 0; b < 2; ++b)
#pragma unroll
                for (int k = 0; k < BITS; ++k)             // an instruction of its own: left to itself the compiler copies where the loop ends, and waits there
                    asm volatile("v_mov_b32 %0, %1" : "=&v"(u[b][k]) : "v"(w[i & 1u][k][b]));
            request(i < 2u ? block : next, (i + 2u) & 3u);
            u32x4 f[2][4];
#pragma unroll
            for (int b = 0; b < 2; ++b) {
                decode<FMT, BITS>(u[b], tab[b], f[b]);
#pragma unroll
                for (int j = 0; j < 4; ++j) asm volatile("" : "+v"(f[b][j]));              // here, and not where it is used
            }
            // this packet's copies of the first waves, requested behind their last products and ahead of 2 BITS words
            if (!second) asm volatile("s_waitcnt vmcnt(%0)" : : "n"(2 * BITS) : "memory");
            turn();
#pragma unroll
            for (uint32_t j = 0; j < 4u; ++j)
#pragma unroll
                for (int m = 0; m < MT; ++m) {
                    Frag<DT> xf;
                    xf.v = *(const u32x4*)(xs + (frag_at ^ (j << 4)) + 16u * m * kXRow);
#pragma unroll
                    for (int b = 0; b < 2; ++b) {
                        Frag<DT> wf;
                        wf.v = f[b][j];
                        mma(wf, xf, acc[m][b]);
                    }
                }
            __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
#pragma unroll
            for (int k = 0; k < 4 * MT; ++k) {
                __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
                if (k + 4 < 4 * MT) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
            // the next packet's copies: of the first waves behind their products, of the second waves, requested ahead of 2 BITS words, there by now
            if (!second) request_x(i < 3u ? block : next, (i + 1u) & 3u, (i + 1u) & 1u);
            else asm volatile("s_waitcnt vmcnt(%0)" : : "n"(2 * BITS) : "memory");
            turn();
        }
    }
    if (!second) turn();
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");       // copies into LDS end before the workgroup does
    if (p.half != 0u) {
        store_gated<DT, MT>(p, columns, acc, m0, l16, lg);
        return;
    }
#pragma unroll
    for (int m = 0; m < MT; ++m) {
        const uint32_t row = m0 + 16u * m + l16;
#pragma unroll
        for (uint32_t b = 0; b < 2u; ++b) {
            const uint32_t n = n0 + 16u * b + 4u * lg;
            if (row >= p.M || n >= N) continue;
            if (p.wide) {
                *(u32x2*)((uint16_t*)p.out + (size_t)row * N + n) = u32x2{pack16<DT>(acc[m][b][0], acc[m][b][1]), pack16<DT>(acc[m][b][2], acc[m][b][3])};
            } else {
#pragma unroll
                for (uint32_t e = 0; e < 4u; ++e) if (n + e < N) Elem<DT>::store(p.out, (size_t)row * N + n + e, acc[m][b][e]);
            }
        }
    }
}

template <int FMT, int BITS, int DT, int MT>
static hipError_t wide_mt(const QgemmParams& p, uint32_t tiles, hipStream_t s) {
    constexpr size_t lds = 2u * 16u * MT * kXRow;
    if (hipError_t e = allow_lds<qgemm_wide_kernel<FMT, BITS, DT, MT>>(lds); e != hipSuccess) return e;
    hipLaunchKernelGGL((qgemm_wide_kernel<FMT, BITS, DT, MT>), dim3(tiles), dim3(512), lds, s, p);
    return hipGetLastError();
}

template <int FMT, int BITS, int DT>
static hipError_t wide_dt(const QgemmParams& p, uint32_t mt, uint32_t tiles, hipStream_t s) {
    switch (mt) {
        case 10u: return wide_mt<FMT, BITS, DT, 10>(p, tiles, s);
        case 12u: return wide_mt<FMT, BITS, DT, 12>(p, tiles, s);
        case 14u: return wide_mt<FMT, BITS, DT, 14>(p, tiles, s);
        default: break;
    }
    if constexpr (FMT == kSqllm) return wide_mt<FMT, BITS, DT, 16>(p, tiles, s);
    else return hipErrorInvalidValue;                      // qgemm_goes_wide
}

// 16-token tiles of a workgroup (an even number), token tiles, workgroups.
struct WidePlan { uint32_t mt, z, tiles; };
static WidePlan wide_plan(uint32_t M, uint32_t N) {
    const uint32_t z = (M + 255u) / 256u, mt = ((M + z - 1u) / z + 31u) / 32u * 2u, groups = (N + 255u) / 256u;
    return {mt, z, (z == 1u ? groups : (groups + 7u) / 8u * 8u) * z};
}

// Where one or two turns of the compute units are three quarters full.  (4096 -> 28672: 224 workgroups for 257 - 512 tokens; 112 for up to
// 256, 134 us for 98; 4096 -> 4096 at 512 tokens, in eight ranges of channels, 43 for 33.)  Of one block of channels alone filling and storing are
// the larger part: one turn, and of more than 12 tiles of tokens one that is seven eighths full.  Times over those of tiles of 128 tokens, 129 - 1999
// tokens x 6144 - 49160 outputs, all three formats: 1024 - 14336 channels 0.59 - 0.90; 512 channels, taken 0.79 - 0.975, left 0.94 - 1.21.
bool qgemm_goes_wide(int fmt, int bits, uint32_t M, uint32_t N, uint32_t K, uint32_t group) {
    if ((fmt != kSqllm && !(fmt == kLutgemm && bits == 3 && group % 128u == 0u)) || M <= 128u || K % 512u != 0u || K >= 1u << 22 || N >= 1u << 24) return false;
    const WidePlan g = wide_plan(M, N);
    const uint32_t turns = (g.tiles + 255u) / 256u;
    if (g.mt < 10u || (g.mt > 14u && fmt != kSqllm) || turns > 2u || 4u * g.tiles < 3u * 256u * turns) return false;
    return K >= 1024u || (turns == 1u && (g.mt <= 12u || 8u * g.tiles >= 7u * 256u));
}

hipError_t launch_qgemm_wide(int fmt, int dt, int bits, QgemmParams p, hipStream_t s) {
    const WidePlan g = wide_plan(p.M, p.N);
    p.z = g.z;
    p.groups = (p.N + 255u) / 256u;
    if (fmt == kLutgemm) return dt == kFP16 ? wide_dt<kLutgemm, 3, kFP16>(p, g.mt, g.tiles, s) : wide_dt<kLutgemm, 3, kBF16>(p, g.mt, g.tiles, s);
    if (bits == 3) return dt == kFP16 ? wide_dt<kSqllm, 3, kFP16>(p, g.mt, g.tiles, s) : wide_dt<kSqllm, 3, kBF16>(p, g.mt, g.tiles, s);
    return dt == kFP16 ? wide_dt<kSqllm, 4, kFP16>(p, g.mt, g.tiles, s) : wide_dt<kSqllm, 4, kBF16>(p, g.mt, g.tiles, s);
}

}  // namespace decdec
