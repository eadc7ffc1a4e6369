// Products of several tokens with a packed weight: out[m][n] = sum_c x[m][c] W[n][c], the weight decoded on the way into the
// matrix cores (any-precision, LUT-GEMM, SqueezeLLM, 3 and 4 bits, fp16 / bf16).  The weight is read once, packed; a dense one
// would be written and read, sixteen bits a weight, before a product of a few tokens that needs neither.
//
// A unit is 32 channels of one output, which is what a lane decodes at once: the byte-permute look-ups of the batch-1 kernels
// (16-bit table entries as byte tables in registers; LUT-GEMM builds the table of a group's 8 or 16 values from its scales)
// leave its 32 weights as four fragments of eight.  Weights are the left operand (a lane's row is an output), so neither they
// nor the sums pass LDS.  Which eight channels a fragment holds is up to the look-up -- the contraction may visit channels in
// any order as long as both operands do -- so the activations are arranged to match when they are staged in LDS, once per
// workgroup.  A wave owns 32 outputs (lane row r: 2 r and 2 r + 1) and all 16 MT tokens; the eight waves of a workgroup are WN
// such columns x WK ranges of channels, whose sums meet in LDS; ranges of different workgroups meet in a workspace, summed in
// order by a second kernel.  K advances in blocks of 16 units, four packets of four units (one per lane group): any-precision
// rows give a lane two neighbouring words per plane that way, the other formats' words are neighbours over the outputs.
//
// Bound by the decoding instructions (2 to 3.5 a weight) and, from about 100 tokens, by the matrix cores; both grow with the
// number of 128-token tiles, which a dense weight's expansion does not: beyond a few hundred tokens that is faster.
// Measured, 4096 -> 28672, fp16, us, beside expansion and library product: SqueezeLLM 4 bits 2 tokens 28 / 113, 77 46 / 109, 256
// 103 / 135; any-precision 3 bits 29 / 109, 44 / 103, 107 / 130; LUT-GEMM 3 bits 26 / 109, 44 / 108, 105 / 140.
#include "launch.h"
#include "packed.h"

namespace decdec {

struct QgemmParams {
    const void* x;                 // [M][K]
    const uint32_t* q;
    const void* lut;               // tables [N][2^bits], or the scales [K / group][bits][N] of LUT-GEMM
    const void* q_bias;            // [K / group][N]
    void* out;                     // [M][N]
    float* part;                   // [ks][M][N] where ks > 1
    uint32_t M, N, K, group, ks, blocks;   // blocks of 16 units per range of channels
    uint32_t pairs;                // two neighbouring words (and scales) may be read at once: of a row, or of two outputs
    uint32_t wide;                 // eight neighbouring results may be stored at once
};

template <int FMT>
__device__ __forceinline__ uint32_t unit_of(uint32_t block, uint32_t i, uint32_t g) {
    return 16u * block + (FMT == kAnyprec ? 8u * (i >> 1) + 2u * g + (i & 1u) : 4u * i + g);
}

// More tokens: more columns share the staged ones (four tiles with two columns: 50 us for 39 above).
constexpr uint32_t qgemm_wn(int mt) { return mt >= 4 ? 4u : 2u; }
constexpr uint32_t kXRow = 4u * 64u + 16u;                                             // bytes of a staged token: four units, a pad
constexpr size_t qgemm_lds(int mt) { return 2u * (8u / qgemm_wn(mt)) * 16u * mt * kXRow; }

template <int FMT, int BITS, int DT, int MT>
__global__ __launch_bounds__(512, MT == 1 && (BITS == 3 || FMT == kSqllm) ? 4 : 2) void qgemm_kernel(const QgemmParams p) {
    constexpr uint32_t WN = qgemm_wn(MT), WK = 8u / WN, TASKS = (16u * MT * 4u + 64u * WN - 1u) / (64u * WN);
    extern __shared__ __align__(16) unsigned char smem[];
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6, l16 = lane & 15u, lg = lane >> 4;
    const uint32_t wn = wave % WN, wk = wave / WN, units = p.K / 32u, N = p.N;
    const uint32_t n0 = (blockIdx.x * WN + wn) * 32u, m0 = blockIdx.z * 16u * MT;
    const uint32_t range = blockIdx.y * WK + wk;
    // two columns of a lane; columns past the end repeat the last ones and are not stored
    uint32_t col[2];
    col[0] = n0 + 2u * l16;
    if (FMT != kAnyprec && p.pairs && col[0] + 2u > N) col[0] = N - 2u;
    col[0] = col[0] < N ? col[0] : N - 1u;
    col[1] = col[0] + 1u < N ? col[0] + 1u : N - 1u;
    Tables<BITS> tab[FMT == kLutgemm ? 1 : 2];
    if constexpr (FMT != kLutgemm) {
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            uint32_t e[1 << (BITS - 1)];
            const u32x4* row = (const u32x4*)((const uint16_t*)p.lut + (size_t)col[b] * (1u << BITS));
#pragma unroll
            for (int i = 0; i < (1 << (BITS - 3)); ++i) {
                const u32x4 v = row[i];
#pragma unroll
                for (int k = 0; k < 4; ++k) e[4 * i + k] = v[k];
            }
            tab[b] = tables_of<BITS>(e);
        }
    }
    // words of a block, [packet][word][column], and the scales of its units (two columns in a word); a packet is requested again,
    // for the next block, as soon as it is decoded (any-precision: two packets at once, two neighbouring words of a row)
    uint32_t w[4][BITS][2], sc[FMT == kLutgemm ? 4 : 1][BITS + 1];
    auto request = [&](uint32_t block, uint32_t i) {
        if constexpr (FMT == kAnyprec) {
            const uint32_t u = unit_of<FMT>(block, i, lg);
#pragma unroll
            for (int k = 0; k < BITS; ++k)
#pragma unroll
                for (int b = 0; b < 2; ++b) {
                    const uint32_t* row = p.q + ((size_t)k * N + col[b]) * units;
                    if (p.pairs) {
                        const u32x2 v = *(const u32x2*)(row + (u + 2u <= units ? u : units - 2u));
                        w[i][k][b] = v[0]; w[i + 1][k][b] = v[1];
                    } else {
                        w[i][k][b] = row[u < units ? u : units - 1u];
                        w[i + 1][k][b] = row[u + 1u < units ? u + 1u : units - 1u];
                    }
                }
        } else {
            uint32_t u = unit_of<FMT>(block, i, lg);
            u = u < units ? u : units - 1u;
#pragma unroll
            for (uint32_t k = 0; k < (uint32_t)BITS; ++k) {
                const uint32_t* row = p.q + ((size_t)u * BITS + k) * N;
                if (p.pairs) {
                    const u32x2 v = *(const u32x2*)(row + col[0]);
                    w[i][k][0] = v[0]; w[i][k][1] = v[1];
                } else {
                    w[i][k][0] = row[col[0]]; w[i][k][1] = row[col[1]];
                }
            }
            if constexpr (FMT == kLutgemm) {
                const size_t gr = 32u * u / p.group;
#pragma unroll
                for (uint32_t k = 0; k <= (uint32_t)BITS; ++k) {
                    const uint16_t* row = k < (uint32_t)BITS ? (const uint16_t*)p.lut + (gr * BITS + k) * N : (const uint16_t*)p.q_bias + gr * N;
                    sc[i][k] = p.pairs ? *(const uint32_t*)(row + col[0]) : row[col[0]] | ((uint32_t)row[col[1]] << 16);
                }
            }
        }
    };
    // activations of a packet, a unit of a token per task
    u32x4 xr[TASKS][4];
    const uint32_t ttid = wn * 64u + lane;
    auto request_x = [&](uint32_t block, uint32_t i) {
#pragma unroll
        for (uint32_t t = 0; t < TASKS; ++t) {
            const uint32_t task = ttid + t * 64u * WN, m = m0 + task / 4u, u = unit_of<FMT>(block, i, task & 3u);
            const bool ok = task < 16u * MT * 4u && m < p.M && u < units;
            const uint32_t uc = ok ? u : 0u;
            uint32_t c = 32u * uc, step = 8u;
            if constexpr (FMT == kAnyprec) {
                step = uc / 32u == p.K / 1024u ? 8u * (p.K % 1024u / 32u) : 256u;
                c = 1024u * (uc / 32u) + 8u * (uc & 31u);
            }
            const uint16_t* src = (const uint16_t*)p.x + (size_t)(ok ? m : 0u) * p.K + c;
#pragma unroll
            for (uint32_t j = 0; j < 4u; ++j) xr[t][j] = ok ? *(const u32x4*)(src + j * step) : u32x4{0u, 0u, 0u, 0u};
        }
    };
    f32x4 acc[MT][2];
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[m][0] = acc[m][1] = f32x4{0.f, 0.f, 0.f, 0.f};
    const uint32_t all = (units + 15u) / 16u, first = range * p.blocks;
    const auto at = [&](uint32_t blk) { return first + blk < all ? first + blk : all; };   // `all`: a block with no units
#pragma unroll
    for (uint32_t i = 0; i < 4u; i += FMT == kAnyprec ? 2u : 1u) request(at(0u), i);
    request_x(at(0u), 0u);
    uint32_t turn = 0u;
    for (uint32_t blk = 0; blk < p.blocks; ++blk) {
        const uint32_t block = at(blk);
        const bool tail = 16u * block + 16u > units;
        const uint32_t next = blk + 1u < p.blocks ? at(blk + 1u) : all;
#pragma unroll
        for (uint32_t i = 0; i < 4u; ++i, turn ^= 1u) {
            unsigned char* xs = smem + (turn * WK + wk) * (16u * MT * kXRow);
#pragma unroll
            for (uint32_t t = 0; t < TASKS; ++t) {
                const uint32_t task = ttid + t * 64u * WN;
                u32x4 f[4];
                arrange<FMT, BITS>(xr[t], f);
                if (task < 16u * MT * 4u) {
                    u32x4* dst = (u32x4*)(xs + (task / 4u) * kXRow + (task & 3u) * 64u);
#pragma unroll
                    for (int j = 0; j < 4; ++j) dst[j] = f[j];
                }
            }
            __syncthreads();                               // one a packet: the other buffer's readers passed it before
            if (i < 3u) request_x(block, i + 1u);
            else if (blk + 1u < p.blocks) request_x(next, 0u);
            // few tokens: one column at a time, for its fragments' registers; more: both, for one read of the activations
            constexpr int B = MT <= 2 ? 1 : 2;
#pragma unroll
            for (int b0 = 0; b0 < 2; b0 += B) {
                Frag<DT> wf[B][4];
#pragma unroll
                for (int b = 0; b < B; ++b) {
                    uint32_t u[BITS];
                    u32x4 f[4];
#pragma unroll
                    for (int k = 0; k < BITS; ++k) u[k] = w[i][k][b0 + b];
                    if constexpr (FMT == kLutgemm) {
                        float a[BITS + 1];
#pragma unroll
                        for (int k = 0; k <= BITS; ++k) a[k] = Elem<DT>::from_raw(b0 + b ? sc[i][k] >> 16 : sc[i][k] & 0xFFFFu);
                        decode<FMT, BITS>(u, group_tables<DT, BITS>(a), f);
                    } else {
                        decode<FMT, BITS>(u, tab[b0 + b], f);
                    }
                    // units past the end: their activations are zero, their weights have to be finite
                    const uint32_t mask = !tail || unit_of<FMT>(block, i, lg) < units ? ~0u : 0u;
#pragma unroll
                    for (int j = 0; j < 4; ++j) wf[b][j].v = tail ? f[j] & u32x4{mask, mask, mask, mask} : f[j];
                }
#pragma unroll
                for (int j = 0; j < 4; ++j)
#pragma unroll
                    for (int m = 0; m < MT; ++m) {
                        Frag<DT> xf;
                        xf.v = *(const u32x4*)(xs + (16u * m + l16) * kXRow + lg * 64u + j * 16u);
#pragma unroll
                        for (int b = 0; b < B; ++b) mma(wf[b][j], xf, acc[m][b0 + b]);
                    }
            }
            if (next < all) {
                if (FMT != kAnyprec) request(next, i);
                else if (i & 1u) request(next, i - 1u);
            }
        }
    }
    // the ranges of channels of a workgroup meet in LDS
    __syncthreads();
    f32x4* red = (f32x4*)smem;
    static_assert((WK - 1u) * WN * MT * 2u * 64u * 16u <= qgemm_lds(MT), "sums fit where the activations were");
    if (wk > 0u) {
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int b = 0; b < 2; ++b) red[((((wk - 1u) * WN + wn) * MT + m) * 2u + b) * 64u + lane] = acc[m][b];
    }
    __syncthreads();
    if (wk > 0u) return;
    for (uint32_t r = 0; r + 1u < WK; ++r)
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int b = 0; b < 2; ++b) acc[m][b] += red[(((r * WN + wn) * MT + m) * 2u + b) * 64u + lane];
    // register v of column b: output n0 + 8 (lane / 16) + 2 v + b of token lane % 16
    const uint32_t n = n0 + 8u * lg;
#pragma unroll
    for (int m = 0; m < MT; ++m) {
        const uint32_t row = m0 + 16u * m + l16;
        if (row >= p.M || n >= N) continue;
        float v[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = acc[m][e & 1][e >> 1];
        if (p.ks > 1u) {
            float* dst = p.part + ((size_t)blockIdx.y * p.M + row) * N + n;
            if (p.wide) {
                *(f32x4*)dst = f32x4{v[0], v[1], v[2], v[3]};
                *(f32x4*)(dst + 4) = f32x4{v[4], v[5], v[6], v[7]};
            } else {
#pragma unroll
                for (uint32_t e = 0; e < 8u; ++e) if (n + e < N) dst[e] = v[e];
            }
        } else if (p.wide) {
            Frag<DT> f = frag_of(v, Frag<DT>{});
            *(u32x4*)((uint16_t*)p.out + (size_t)row * N + n) = f.v;
        } else {
#pragma unroll
            for (uint32_t e = 0; e < 8u; ++e) if (n + e < N) Elem<DT>::store(p.out, (size_t)row * N + n + e, v[e]);
        }
    }
}

// Sums of the ranges, in order: eight neighbouring results a thread, moved at once where they are whole and aligned (vec).
template <int DT>
__global__ __launch_bounds__(256) void qgemm_sum_kernel(const float* __restrict__ part, void* __restrict__ out, const uint32_t ks, const size_t count,
                                                        const bool vec) {
    const size_t i = ((size_t)blockIdx.x * 256u + threadIdx.x) * 8u;
    if (i >= count) return;
    float v[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    if (vec) {
        for (uint32_t k = 0; k < ks; ++k) {
            const f32x4 a = *(const f32x4*)(part + k * count + i), b = *(const f32x4*)(part + k * count + i + 4);
#pragma unroll
            for (int e = 0; e < 4; ++e) { v[e] += a[e]; v[4 + e] += b[e]; }
        }
        const Frag<DT> f = frag_of(v, Frag<DT>{});
        *(u32x4*)((uint16_t*)out + i) = f.v;
    } else {
        for (uint32_t e = 0; e < 8u && i + e < count; ++e) {
            float s = 0.f;
            for (uint32_t k = 0; k < ks; ++k) s += part[k * count + i + e];
            Elem<DT>::store(out, i + e, s);
        }
    }
}

// 16-token tiles of a workgroup for M tokens: whole 128-token tiles, evened out.  Every number of them has its instance: tiles of
// padding cost as much as tokens (4096 -> 28672, SqueezeLLM 4 bits, us, with 1, 2, 3, 5 and 8 tiles only / now: 64 tokens 44 / 39, 96
// 52 / 47, 112 54 / 51, 190 98 / 90).
static int qgemm_mt(uint32_t M) {
    const uint32_t tiles = (M + 127u) / 128u;
    return (int)(((M + tiles - 1u) / tiles + 15u) / 16u);
}

// Ranges of channels in different workgroups: as many as bring two workgroups (three tiles or more: one) to every compute unit,
// with at least one block of channels for every wave.
static uint32_t qgemm_ks(uint32_t M, uint32_t N, uint32_t K) {
    const int mt = qgemm_mt(M);
    const uint32_t wn = qgemm_wn(mt), groups = (N + 32u * wn - 1u) / (32u * wn) * ((M + 16u * mt - 1u) / (16u * mt));
    const uint32_t want = mt <= 2 ? 512u : 256u, most = (K + 511u) / 512u / (8u / wn);
    uint32_t ks = want / groups;
    ks = ks < most ? ks : most;
    return ks > 1u ? ks : 1u;
}

size_t qgemm_workspace(uint32_t M, uint32_t N, uint32_t K) {
    const uint32_t ks = qgemm_ks(M, N, K);
    return ks > 1u ? (size_t)ks * M * N * sizeof(float) : 0;
}

template <int FMT, int BITS, int DT>
static hipError_t qgemm_mt_launch(const QgemmParams& p, int mt, hipStream_t s) {
    const uint32_t wn = qgemm_wn(mt);
    const dim3 grid((p.N + 32u * wn - 1u) / (32u * wn), p.ks, (p.M + 16u * mt - 1u) / (16u * mt));
#define DD_MT(m) case m: \
        if (hipError_t e = allow_lds<qgemm_kernel<FMT, BITS, DT, m>>(qgemm_lds(m)); e != hipSuccess) return e; \
        hipLaunchKernelGGL((qgemm_kernel<FMT, BITS, DT, m>), grid, dim3(512), qgemm_lds(m), s, p); break
    switch (mt) { DD_MT(1); DD_MT(2); DD_MT(3); DD_MT(4); DD_MT(5); DD_MT(6); DD_MT(7); default: DD_MT(8); }
#undef DD_MT
    return hipGetLastError();
}

template <int DT>
static hipError_t qgemm_dt(int fmt, int bits, const QgemmParams& p, int mt, hipStream_t s) {
    hipError_t e;
    if (fmt == kAnyprec) e = bits == 3 ? qgemm_mt_launch<kAnyprec, 3, DT>(p, mt, s) : qgemm_mt_launch<kAnyprec, 4, DT>(p, mt, s);
    else if (fmt == kLutgemm) e = bits == 3 ? qgemm_mt_launch<kLutgemm, 3, DT>(p, mt, s) : qgemm_mt_launch<kLutgemm, 4, DT>(p, mt, s);
    else e = bits == 3 ? qgemm_mt_launch<kSqllm, 3, DT>(p, mt, s) : qgemm_mt_launch<kSqllm, 4, DT>(p, mt, s);
    if (e != hipSuccess || p.ks == 1u) return e;
    const size_t count = (size_t)p.M * p.N;
    hipLaunchKernelGGL((qgemm_sum_kernel<DT>), dim3((uint32_t)((count + 2047u) / 2048u)), dim3(256), 0, s, p.part, p.out, p.ks, count,
                       count % 8u == 0 && (((uintptr_t)p.out | (uintptr_t)p.part) % 16u) == 0);
    return hipGetLastError();
}

hipError_t launch_qgemm(int fmt, int dt, int bits, const void* x, const uint32_t* q, const void* lut, const void* q_bias, void* out,
                        void* workspace, uint32_t M, uint32_t N, uint32_t K, uint32_t group, hipStream_t s) {
    const int mt = qgemm_mt(M);
    QgemmParams p{};
    p.x = x; p.q = q; p.lut = lut; p.q_bias = q_bias; p.out = out; p.part = (float*)workspace;
    p.M = M; p.N = N; p.K = K; p.group = group;
    p.ks = qgemm_ks(M, N, K);
    const uint32_t ranges = p.ks * (8u / qgemm_wn(mt)), all = (K + 511u) / 512u;
    p.blocks = (all + ranges - 1u) / ranges;
    p.pairs = (fmt == kAnyprec ? K % 64u : N % 2u) == 0 && ((uintptr_t)q % 8u) == 0 && (((uintptr_t)lut | (uintptr_t)q_bias) % 4u) == 0;
    p.wide = N % 8u == 0 && (((uintptr_t)out | (uintptr_t)workspace) % 16u) == 0;
    return dt == kFP16 ? qgemm_dt<kFP16>(fmt, bits, p, mt, s) : qgemm_dt<kBF16>(fmt, bits, p, mt, s);
}

}  // namespace decdec
