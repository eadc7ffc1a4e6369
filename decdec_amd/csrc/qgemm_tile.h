// Products of several tokens with a packed weight: out[m][n] = sum_c x[m][c] W[n][c], the weight decoded on the way into the
// matrix cores (any-precision, LUT-GEMM, SqueezeLLM, 3 and 4 bits, fp16 / bf16).  The weight is read once, packed; a dense one
// would be written and read, sixteen bits a weight, before a product of a few tokens that needs neither.
//
// A unit is 32 channels of one output, which is what a lane decodes at once: the byte-permute look-ups of the batch-1 kernels
// (16-bit table entries as byte tables in registers; LUT-GEMM builds the table of a group's 8 or 16 values from its scales, once for four
// units where groups are a multiple of 128 channels) leave its 32 weights as four fragments of eight neighbouring channels.  Weights are
// the left operand (a lane's row is an output), so neither they nor the sums pass LDS; the activations do, as they are in memory, by copies that
// pass no register.
// A wave owns 32 outputs (lane row r: r and r + 16) and all 16 MT tokens; the waves of a workgroup are WN such columns x WK ranges of
// channels, whose sums meet in LDS.  K advances in blocks of 16 units, four packets of four units (one per lane group): any-precision
// rows give a lane two neighbouring words per plane that way, the other formats' words are neighbours over the outputs.
//
// Tiles of outputs and tokens that fill the compute units go to one workgroup each; what is left after the last full turn is split along
// the channels, its sums meet in a workspace and a second kernel adds them in order (5120 -> 35840 are 280 tiles on 256 units: two turns
// before, 1.2 now).
//
// What bounds it: vector instructions of the decoding (2.2 to 4 a weight) and matrix products, which take turns in the waves of a SIMD (below), and
// what a launch costs whatever it does.  Counted, vector instructions take 49 % of the SIMDs' cycles and products 31 % at 77 tokens of LUT-GEMM 3 bits, 52 and 40 % in
// tiles of 128 of SqueezeLLM 4 bits, reads of the activations 16 and 21 % of LDS's; no bank conflicts.  Before, activations passed registers (1100 of a
// packet's 5500 cycles at 128 tokens), both ranges of channels decoded at the same time and waited for each other (2000), and a wave waited for all
// its requests once a block, where the compiler copied their registers.  us, fp16, graphs of four layers in turn, 16, 77 and 128 tokens, before -> now: SqueezeLLM 4 bits
// 4096 -> 28672 28.4, 39.7, 52.6 -> 26.2, 37.6, 43.6; 14336 -> 4096 21.5, 27.2, 34.9 -> 20.2, 26.9, 31.0 (256 and 512 tokens 53, 85 -> 47.5, 73); any-precision 3 bits
// 4096 -> 28672 28.1, 38.8, 52.5 -> 26.8, 37.0, 44.6; LUT-GEMM 3 bits 24.3, 35.8, 48.7 -> 21.6, 33.0, 40.2.
// Tried: tiles of 32 x 32 (a third of the vector issue of 16 x 16 for the same products; fewer cycles at a lower clock, 45 for 42 us of one layer at 128 tokens,
// and 39.5 for 34 at 77, of which 96 are multiplied), copies requested ahead of the products, between them or behind them instead of ahead of the decoding (41 to
// 44), priorities for waves that multiply (the same), results added and stored by both ranges (43.5).
// Beside expansion and library product, 4096 -> 28672: SqueezeLLM 4 bits 16 tokens 26 / 129, 77 37 / 116; any-precision 3 bits 28 / 125, 38 / 114; LUT-GEMM
// 3 bits 22 / 125, 33 / 114.
// Where tiles of 256 tokens and outputs fill the compute units they are taken instead, k_qgemm_wide.hip.  How tiles are dealt, and their sums: k_qgemm.hip.
#pragma once
#include <type_traits>
#include "qgemm.h"

namespace decdec {


// More tokens: more columns share the staged ones.
constexpr uint32_t qgemm_wn(int mt) { return mt >= 3 ? 4u : 2u; }
// Waves a SIMD for which registers are dealt out, and no more: left to itself the compiler goes for three where they nearly fit and shortens the
// way from a load to its use (64 tokens 4096 -> 28672, any-precision 3 bits, 41.0 us with three and 34.6 with two).  One tile: four; LUT-GEMM 4 bits
// would keep 12 bytes a lane in scratch then (with 48, 16 tokens 14336 -> 4096 27.3 us, with two waves 22.3; the other formats 28 us at 4096 -> 28672 and 31 with two).
constexpr int qgemm_waves(int fmt, int bits, int mt) { return mt == 1 && !(fmt == kLutgemm && bits == 4) ? 4 : 2; }
// Packets of activations in LDS or on their way there: three, as long as there is room.
constexpr uint32_t qgemm_stages(int mt) { return mt <= 6 ? 3u : 2u; }
constexpr size_t qgemm_lds(int mt, uint32_t wk) { return (size_t)qgemm_stages(mt) * wk * 16u * mt * kXRow; }

// At most N of this wave's requests to memory are still out, and none to LDS.
template <uint32_t N>
__device__ __forceinline__ void wait_copies() { asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" : : "n"(N) : "memory"); }

// FLAG: any-precision: two neighbouring words of a row may be read at once.  The others: fewer than 2^24 outputs, so that offsets among a
// block's units have 32 bits (4 % of the time), and, LUT-GEMM, groups of a multiple of 128 channels.
template <int FMT, int BITS, int DT, int MT, bool FLAG>
__global__ __attribute__((amdgpu_flat_work_group_size(64, 512), amdgpu_waves_per_eu(qgemm_waves(FMT, BITS, MT), qgemm_waves(FMT, BITS, MT))))
void qgemm_kernel(const QgemmParams p) {
    constexpr uint32_t WN = qgemm_wn(MT), TASKS = 4u * MT / WN, BN = 32u * WN, S = qgemm_stages(MT);
    constexpr bool PAIRS = FLAG, once = FMT == kLutgemm && FLAG;
    extern __shared__ __align__(16) unsigned char smem[];
    const uint32_t lane = threadIdx.x & 63u, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l16 = lane & 15u, lg = lane >> 4;
    const uint32_t wn = wave % WN, wk = wave / WN, units = p.K / 32u, N = p.N;
    // the workgroup's tile and its share of the channels
    const bool split = blockIdx.x >= p.whole;
    const uint32_t rest = blockIdx.x - p.whole, tile = split ? p.whole + rest / p.ks : blockIdx.x, share = split ? rest % p.ks : 0u;
    // token tiles of the same columns follow each other on one die
    const uint32_t cg = p.z == 1u ? tile : tile / (8u * p.z) * 8u + tile % 8u, zt = p.z == 1u ? 0u : tile / 8u % p.z;
    if (cg >= p.groups) return;
    const uint32_t m0 = zt * 16u * MT;
    const uint32_t blocks = split ? p.ks_blocks : p.blocks, first = (share * p.wk + wk) * blocks;
    const QgemmColumns columns = qgemm_columns(p, cg * WN + wn, l16);
    const uint32_t n0 = columns.n0, nb = columns.nb;
    const uint32_t (&col)[2] = columns.col;
    Tables<BITS> tab[2];
    u32x4 lut[2][1 << (BITS - 3)];                         // rows of the table
    if constexpr (FMT != kLutgemm) {
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            const u32x4* row = (const u32x4*)((const uint16_t*)p.lut + (size_t)(nb + col[b]) * (1u << BITS));
#pragma unroll
            for (int i = 0; i < (1 << (BITS - 3)); ++i) lut[b][i] = row[i];
        }
    }
    __builtin_amdgcn_sched_barrier(0);                     // requests in this order: a wait counts what is behind the one that is waited for
    // Words of a block, [packet][word][column]; a packet's are requested for the next block as soon as it is decoded (any-precision:
    // two packets' at once, neighbouring words of a row).  Loads return in order: a wait for a packet's activations, requested S - 1 packets ago, waits for the words that
    // were asked for before them and leaves those behind them, which it counts; words have a block, four packets, to arrive.
    uint32_t w[4][BITS][2];
    auto request = [&](uint32_t block, uint32_t i) {
        if constexpr (FMT == kAnyprec) {
            const uint32_t ub = 16u * block + 8u * (i >> 1), u0 = ub < units ? ub : (PAIRS ? units - 2u : units - 1u), room = units - u0;
            const uint32_t l0 = 2u * lg < room ? 2u * lg : (PAIRS ? room - 2u : room - 1u), l1 = 2u * lg + 1u < room ? 2u * lg + 1u : room - 1u;
#pragma unroll
            for (int k = 0; k < BITS; ++k) {
                const uint32_t* row = p.q + ((size_t)k * N + nb) * units + u0;
#pragma unroll
                for (int b = 0; b < 2; ++b) {
                    if constexpr (PAIRS) {
                        const u32x2 v = *(const u32x2*)(row + ((size_t)col[b] * units + l0));
                        w[i][k][b] = v[0]; w[i + 1][k][b] = v[1];
                    } else {
                        w[i][k][b] = row[(size_t)col[b] * units + l0];
                        w[i + 1][k][b] = row[(size_t)col[b] * units + l1];
                    }
                }
            }
        } else {
            const uint32_t step = FMT == kLutgemm ? 4u : 1u, ub = unit_of<FMT>(block, i, 0u), u0 = ub < units ? ub : units - 1u;
            const uint32_t l = step * lg < units - u0 ? step * lg : units - 1u - u0, at = l * (uint32_t)BITS;
            const uint32_t* row = p.q + (size_t)u0 * BITS * N + nb;
#pragma unroll
            for (uint32_t k = 0; k < (uint32_t)BITS; ++k, row += N)
#pragma unroll
                for (int b = 0; b < 2; ++b)
                    w[i][k][b] = FLAG ? *(const uint32_t*)((const char*)row + 4u * (at * N + col[b])) : row[(size_t)at * N + col[b]];
        }
    };
    // scales of a unit; groups of a multiple of 128 channels: of a block's four units
    uint32_t sc[BITS + 1][2];
    auto request_scales = [&](uint32_t block, uint32_t i) {
        if constexpr (FMT == kLutgemm) {
            uint32_t u = unit_of<FMT>(block, i, lg);
            u = u < units ? u : units - 1u;
            const size_t gr = u / (p.group / 32u);
#pragma unroll
            for (uint32_t k = 0; k <= (uint32_t)BITS; ++k) {
                const uint16_t* row = (k < (uint32_t)BITS ? (const uint16_t*)p.lut + (gr * BITS + k) * N : (const uint16_t*)p.q_bias + gr * N) + nb;
#pragma unroll
                for (int b = 0; b < 2; ++b) sc[k][b] = row[col[b]];
            }
        }
    };
    // Activations of a packet go to LDS by copies that pass no register, four tokens of 256 bytes each.  Piece q of row m lies at
    // q ^ (m - 4): the sixteen lanes of a phase of a 16-byte LDS read are rows 0-3 and 12-15 with one lane group and rows 4-11 with its
    // neighbour.  A lane copies the piece that belongs where it writes; piece: 4 unit + j, any-precision 4 j + unit, whose four units lie in one
    // line of memory.  Tokens past the end repeat the last one and are not stored.
    const char* xb = (const char*)p.x + (size_t)m0 * p.K * 2u;
    uint32_t xrow[TASKS];
#pragma unroll
    for (uint32_t t = 0; t < TASKS; ++t) {
        const uint32_t m = t * 4u * WN + 4u * wn + lg;
        xrow[t] = (m0 + m < p.M ? m : p.M - 1u - m0) * p.K * 2u;
    }
    auto piece = [&](uint32_t t) { return l16 ^ ((t * 4u * WN + 4u * wn + lg + 12u) & 15u); };      // the same for every t, or for every other one
    auto unit_in = [&](uint32_t t) { return FMT == kAnyprec ? piece(t) & 3u : piece(t) >> 2; };
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)smem;
    auto place = [&](uint32_t buf) { return (buf * p.wk + wk) * (16u * MT * kXRow); };
    auto request_x = [&](uint32_t block, uint32_t i, uint32_t buf) {
        uint32_t at[2];
#pragma unroll
        for (uint32_t t = 0; t < (WN == 4u ? 1u : 2u); ++t) {
            uint32_t u = unit_of<FMT>(block, i, unit_in(t));
            u = u < units ? u : units - 1u;
            const uint32_t j = FMT == kAnyprec ? piece(t) >> 2 : piece(t) & 3u;
            at[t] = 64u * u + 16u * j;
            if constexpr (FMT == kAnyprec) {               // pieces of a word's 32 channels are 256 apart, closer in a last, shorter chunk
                const uint32_t step = u / 32u == p.K / 1024u ? 16u * (p.K % 1024u / 32u) : 512u;
                at[t] = 2048u * (u / 32u) + 16u * (u & 31u) + step * j;
            }
        }
        const uint32_t to = lds0 + place(buf) + 4u * wn * kXRow;
#pragma unroll
        for (uint32_t t = 0; t < TASKS; ++t)
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                         : : "s"(__builtin_amdgcn_readfirstlane(to + t * 4u * WN * kXRow)), "v"(xrow[t] + at[WN == 4u ? 0u : t & 1u]), "s"(xb) : "memory");
    };
    f32x4 acc[MT][2];
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[m][0] = acc[m][1] = f32x4{0.f, 0.f, 0.f, 0.f};
    const uint32_t all = (units + 15u) / 16u;
    const auto at = [&](uint32_t blk) { return first + blk < all ? first + blk : all; };   // `all`: a block with no units
    request_x(at(0u), 0u, 0u);
    if constexpr (FMT == kLutgemm) request_scales(at(0u), 0u);
    if constexpr (S == 3u) request_x(at(0u), 1u, 1u);
#pragma unroll
    for (uint32_t i = 0; i < 4u; i += FMT == kAnyprec ? 2u : 1u) {
        __builtin_amdgcn_sched_barrier(0);
        request(at(0u), i);
    }
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (FMT != kLutgemm) {
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            uint32_t e[1 << (BITS - 1)];
#pragma unroll
            for (int i = 0; i < (1 << (BITS - 1)); ++i) e[i] = lut[b][i >> 2][i & 3];
            tab[b] = tables_of<BITS>(e);
        }
    }
    const uint32_t frag_at = l16 * kXRow + (((FMT == kAnyprec ? lg : 4u * lg) ^ ((l16 + 12u) & 15u)) << 4);
    constexpr uint32_t frag_j = FMT == kAnyprec ? 64u : 16u;
    // Waves of two ranges of channels share a SIMD and take turns: one range decodes while the other multiplies.  Left to themselves both come
    // to either at the same time, and the vector instructions of the older one keep the matrix units from the other.
    const bool turns = MT >= 3 && p.wk == 2u;
    auto turn = [&] {
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    };
    uint32_t buf = 0u;
    // Packet I of a block; MORE: the block is not the last one, whose waves would ask for twice as much as they use.  (Where a loop may or may not
    // request, a wait behind it counts on none.)
    auto packet = [&](auto more_blocks, auto number, const uint32_t blk) {
        constexpr bool MORE = decltype(more_blocks)::value;
        constexpr uint32_t I = decltype(number)::value;
        const uint32_t block = at(blk), next = at(blk + 1u);
        const bool tail = 16u * block + 16u > units;
        unsigned char* xs = smem + place(buf);
        // This packet's copies, requested S - 1 packets ago.  Behind them: words of the packets since (any-precision: of a pair, in its second
        // packet) and later packets' copies.  And what this wave reads of the buffer that is copied to next.
        constexpr uint32_t W = FMT == kAnyprec ? (PAIRS ? 2u : 4u) * BITS : 2u * BITS, ALL = FMT == kAnyprec ? 2u * W : 4u * W;
        constexpr uint32_t back1 = (!MORE && I > 0u) || (FMT == kAnyprec && (I & 1u)) ? 0u : W;            // words requested a packet ago
        constexpr uint32_t back2 = (!MORE && I > 1u) || (FMT == kAnyprec && !(I & 1u)) ? 0u : W;
        if constexpr (S == 2u) {
            if (I == 0u && blk == 0u) wait_copies<ALL>();
            else wait_copies<back1>();
        } else {
            if (I < 2u && blk == 0u) wait_copies<TASKS + ALL>();
            else wait_copies<back2 + (MORE || I < 3u ? TASKS : 0u) + back1>();
        }
        if (tail) {                                        // units past the end: zero
#pragma unroll
            for (uint32_t t = 0; t < TASKS; ++t)
                if (unit_of<FMT>(block, I, unit_in(t)) >= units) *(u32x4*)(xs + (t * 4u * WN + 4u * wn) * kXRow + lane * 16u) = u32x4{0u, 0u, 0u, 0u};
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        }
        turn();                                            // everybody's copies are there, and nobody reads what is copied to next
        if constexpr (I + S - 1u < 4u || MORE) request_x(I + S - 1u < 4u ? block : next, (I + S - 1u) & 3u, buf + S - 1u < S ? buf + S - 1u : buf - 1u);
        if constexpr (FMT == kLutgemm) {
            if constexpr (I == 0u || !once) {
#pragma unroll
                for (int b = 0; b < 2; ++b) {
                    float a[BITS + 1];
#pragma unroll
                    for (int k = 0; k <= BITS; ++k) a[k] = Elem<DT>::from_raw(sc[k][b]);
                    tab[b] = group_tables<DT, BITS>(a);
                }
                if constexpr (MORE || !(once || I == 3u)) request_scales(once || I == 3u ? next : block, once ? 0u : (I + 1u) & 3u);
            }
        }
        uint32_t u[2][BITS];
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int k = 0; k < BITS; ++k) {
                // A copy here, in an instruction of its own: left to itself the compiler copies where the loop ends, and waits for every
                // request there.
                if constexpr (MORE) asm volatile("v_mov_b32 %0, %1" : "=&v"(u[b][k]) : "v"(w[I][k][b]));
                else u[b][k] = w[I][k][b];
            }
        if constexpr (FMT != kAnyprec && MORE) request(next, I);
        // few tokens: one column at a time, for its fragments' registers; more: both, for one read of the activations
        constexpr int B = MT <= 2 ? 1 : 2;
#pragma unroll
        for (int b0 = 0; b0 < 2; b0 += B) {
            Frag<DT> wf[B][4];
#pragma unroll
            for (int b = 0; b < B; ++b) {
                u32x4 f[4];
                decode<FMT, BITS>(u[b0 + b], tab[b0 + b], f);
#pragma unroll
                for (int j = 0; j < 4; ++j) wf[b][j].v = f[j];
                if (tail) {                                // units past the end: their activations are zero, their weights have to be finite
                    const uint32_t mask = unit_of<FMT>(block, I, lg) < units ? ~0u : 0u;
#pragma unroll
                    for (int j = 0; j < 4; ++j) wf[b][j].v &= u32x4{mask, mask, mask, mask};
                }
            }
            if (turns) turn();
#pragma unroll
            for (uint32_t j = 0; j < 4u; ++j)
#pragma unroll
                for (int m = 0; m < MT; ++m) {
                    Frag<DT> xf;
                    xf.v = *(const u32x4*)(xs + (frag_at ^ (j * frag_j)) + 16u * m * kXRow);
#pragma unroll
                    for (int b = 0; b < B; ++b) mma(wf[b][j], xf, acc[m][b0 + b]);
                }
            if constexpr (MT >= 3) {                       // activations six reads ahead of their products
                constexpr int AHEAD = 6;
                __builtin_amdgcn_sched_group_barrier(0x100, AHEAD, 0);
#pragma unroll
                for (int k = 0; k < 4 * MT; ++k) {
                    __builtin_amdgcn_sched_group_barrier(0x008, B, 0);
                    if (k + AHEAD < 4 * MT) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                }
            }
        }
        if constexpr (FMT == kAnyprec && (I & 1u) && MORE) request(next, I - 1u);
        buf = buf + 1u < S ? buf + 1u : 0u;
    };
    auto step = [&](auto more_blocks, const uint32_t blk) {
        packet(more_blocks, std::integral_constant<uint32_t, 0>{}, blk);
        packet(more_blocks, std::integral_constant<uint32_t, 1>{}, blk);
        packet(more_blocks, std::integral_constant<uint32_t, 2>{}, blk);
        packet(more_blocks, std::integral_constant<uint32_t, 3>{}, blk);
    };
    if (turns && wk == 1u) turn();
    for (uint32_t blk = 0; blk + 1u < blocks; ++blk) step(std::true_type{}, blk);
    step(std::false_type{}, blocks - 1u);
    if (turns && wk == 0u) turn();
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");       // copies into LDS end before the workgroup does
    // the ranges of channels of a workgroup meet in LDS
    f32x4* red = (f32x4*)smem;
    if (p.wk > 1u) {
        __syncthreads();
        if (wk > 0u) {
#pragma unroll
            for (int m = 0; m < MT; ++m)
#pragma unroll
                for (int b = 0; b < 2; ++b) red[((((wk - 1u) * WN + wn) * MT + m) * 2u + b) * 64u + lane] = acc[m][b];
        }
        __syncthreads();
        if (wk > 0u) return;
        for (uint32_t r = 0; r + 1u < p.wk; ++r)
#pragma unroll
            for (int m = 0; m < MT; ++m)
#pragma unroll
                for (int b = 0; b < 2; ++b) acc[m][b] += red[(((r * WN + wn) * MT + m) * 2u + b) * 64u + lane];
    }
    // register v of column b: output n0 + 16 b + 4 (lane / 16) + v of token lane % 16
    if (columns.gated && !(split && p.ks > 1u)) {
        store_gated<DT, MT>(p, columns, acc, m0, l16, lg);
        return;
    }
    const uint32_t ld = p.half != 0u ? p.half : N;
#pragma unroll
    for (int m = 0; m < MT; ++m) {
        const uint32_t row = m0 + 16u * m + l16;
#pragma unroll
        for (uint32_t b = 0; b < 2u; ++b) {
            const uint32_t c = 16u * b + 4u * lg, n = n0 + c;
            if (split && p.ks > 1u) {
                *(f32x4*)(p.part + (size_t)rest * (16u * MT * BN) + ((((wn * MT + m) * 2u + b) * 64u + lane) * 4u)) = acc[m][b];
                continue;
            }
            if (row >= p.M || n >= columns.end) continue;
            if (p.wide) {
                uint32_t v[2];
#pragma unroll
                for (int e = 0; e < 2; ++e) v[e] = pack16<DT>(acc[m][b][2 * e], acc[m][b][2 * e + 1]);
                *(u32x2*)((uint16_t*)p.out + (size_t)row * ld + n) = u32x2{v[0], v[1]};
            } else {
#pragma unroll
                for (uint32_t e = 0; e < 4u; ++e) if (n + e < columns.end) Elem<DT>::store(p.out, (size_t)row * ld + n + e, acc[m][b][e]);
            }
        }
    }
}

// How a product is dealt to workgroups.
struct QgemmPlan {
    int mt;
    uint32_t wn, wk, groups, z, whole, tiles, ks, blocks, ks_blocks;
};

template <int FMT, int BITS, int DT, bool FLAG>
static hipError_t qgemm_mt_launch(const QgemmParams& p, const QgemmPlan& g, hipStream_t s) {
    const dim3 grid(g.whole + (g.tiles - g.whole) * g.ks), block(64u * g.wn * g.wk);
    const size_t lds = qgemm_lds(g.mt, g.wk);
#define DD_MT(m) case m: \
        if (hipError_t e = allow_lds<qgemm_kernel<FMT, BITS, DT, m, FLAG>>(qgemm_lds(m, 8u / qgemm_wn(m))); e != hipSuccess) return e; \
        hipLaunchKernelGGL((qgemm_kernel<FMT, BITS, DT, m, FLAG>), grid, block, lds, s, p); break
    switch (g.mt) { DD_MT(1); DD_MT(2); DD_MT(3); DD_MT(4); DD_MT(5); DD_MT(6); DD_MT(7); default: DD_MT(8); }
#undef DD_MT
    return hipGetLastError();
}

template <int FMT, int DT>
static hipError_t qgemm_bits(int bits, bool flag, const QgemmParams& p, const QgemmPlan& g, hipStream_t s) {
    if (flag) return bits == 3 ? qgemm_mt_launch<FMT, 3, DT, true>(p, g, s) : qgemm_mt_launch<FMT, 4, DT, true>(p, g, s);
    return bits == 3 ? qgemm_mt_launch<FMT, 3, DT, false>(p, g, s) : qgemm_mt_launch<FMT, 4, DT, false>(p, g, s);
}

// All instances of a format, in a translation unit of its own: all of them in one take the compiler three times as long as anything else here.
template <int FMT>
static hipError_t qgemm_tiles(int dt, int bits, bool flag, const QgemmParams& p, const QgemmPlan& g, hipStream_t s) {
    return dt == kFP16 ? qgemm_bits<FMT, kFP16>(bits, flag, p, g, s) : qgemm_bits<FMT, kBF16>(bits, flag, p, g, s);
}

hipError_t launch_qgemm_anyprec(int dt, int bits, bool flag, const QgemmParams& p, const QgemmPlan& g, hipStream_t s);
hipError_t launch_qgemm_lutgemm(int dt, int bits, bool flag, const QgemmParams& p, const QgemmPlan& g, hipStream_t s);
hipError_t launch_qgemm_sqllm(int dt, int bits, bool flag, const QgemmParams& p, const QgemmPlan& g, hipStream_t s);

}  // namespace decdec
