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
// Where tiles of 256 tokens and outputs fill the compute units they are taken instead, k_qgemm_wide.hip.
#include <type_traits>
#include "qgemm.h"

namespace decdec {

// More tokens: more columns share the staged ones.
constexpr uint32_t qgemm_wn(int mt) { return mt >= 3 ? 4u : 2u; }
// Waves a SIMD for which registers are dealt out, and no more: left to itself the compiler goes for three where they nearly fit and shortens the
// way from a load to its use (64 tokens 4096 -> 28672, any-precision 3 bits, 41.0 us with three and 34.6 with two).  One tile: four; LUT-GEMM 4 bits
// would keep 48 bytes a lane in scratch then (16 tokens 14336 -> 4096 27.3 us, with two waves 22.3; the other formats 28 us at 4096 -> 28672 and 31 with two).
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

// Sums of the split tiles' shares, in order: eight neighbouring results of a token a thread.  A share lies as its lanes hold it, a kilobyte a
// fragment, so that whole lines are written and read (in rows of a tile, pieces of 64 bytes, 128 tokens 4096 -> 4096, SqueezeLLM 4 bits, took
// 25.4 us, now 21.9).  grid (rows of a tile x its pieces / 256, split tiles)
template <int DT>
__global__ __launch_bounds__(256) void qgemm_sum_kernel(const QgemmParams p, const uint32_t rows, const uint32_t cols) {
    // a fragment: 16 tokens, 16 outputs; a thread takes those of two neighbouring lane groups, with gates those of their partners too
    const bool pairs = p.half != 0u && p.whole == 0u;
    const uint32_t id = blockIdx.x * 256u + threadIdx.x, l16 = id & 15u, half = id >> 4 & 1u, mt = rows / 16u, frag = pairs ? id >> 5 << 1 : id >> 5;
    const uint32_t m = frag / 2u % mt * 16u + l16, wave = frag / 2u / mt, c = wave * (pairs ? 16u : 32u) + (frag & 1u) * 16u + half * 8u;
    const uint32_t tile = p.whole + blockIdx.y, width = pairs ? cols / 2u : cols, N = pairs ? p.half : p.N;
    const uint32_t cg = p.z == 1u ? tile : tile / (8u * p.z) * 8u + tile % 8u, zt = p.z == 1u ? 0u : tile / 8u % p.z;
    const uint32_t row = zt * rows + m, n = cg * width + c;
    if (c >= width || row >= p.M || n >= N) return;
    const float* part = p.part + (size_t)blockIdx.y * p.ks * (rows * cols) + (frag * 64u + half * 32u + l16) * 4u;
    float v[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f}, u[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    for (uint32_t k = 0; k < p.ks; ++k, part += rows * cols) {
        const f32x4 a = *(const f32x4*)part, b = *(const f32x4*)(part + 64);
#pragma unroll
        for (int e = 0; e < 4; ++e) { v[e] += a[e]; v[4 + e] += b[e]; }
        if (pairs) {
            const f32x4 g = *(const f32x4*)(part + 256), h = *(const f32x4*)(part + 320);
#pragma unroll
            for (int e = 0; e < 4; ++e) { u[e] += g[e]; u[4 + e] += h[e]; }
        }
    }
    if (pairs) {
        u32x4 r;
#pragma unroll
        for (int e = 0; e < 4; ++e) r[e] = gated2<DT>(v[2 * e], u[2 * e], v[2 * e + 1], u[2 * e + 1]);
        *(u32x4*)((uint16_t*)p.out + (size_t)row * N + n) = r;
        return;
    }
    if (p.half != 0u) {                                    // partners of gates that whole tiles have stored
        u32x4* at = (u32x4*)((uint16_t*)p.out + (size_t)row * p.half + (n - p.half));
        const u32x4 g = *at;
        u32x4 r;
#pragma unroll
        for (int e = 0; e < 4; ++e)
            r[e] = gated2<DT>(Elem<DT>::from_raw(g[e] & 0xFFFFu), v[2 * e], Elem<DT>::from_raw(g[e] >> 16), v[2 * e + 1]);
        *at = r;
        return;
    }
    if (p.wide) {
        const Frag<DT> f = frag_of(v, Frag<DT>{});
        *(u32x4*)((uint16_t*)p.out + (size_t)row * N + n) = f.v;
    } else {
#pragma unroll
        for (uint32_t e = 0; e < 8u; ++e) if (n + e < N) Elem<DT>::store(p.out, (size_t)row * N + n + e, v[e]);
    }
}

// 16-token tiles of a workgroup for M tokens: whole 128-token tiles, evened out.  Every number of them has its instance: tiles of
// padding cost as much as tokens (4096 -> 28672, SqueezeLLM 4 bits, us, with 1, 2, 3, 5 and 8 tiles only / all: 64 tokens 44 / 39, 96
// 52 / 47, 112 54 / 51, 190 98 / 90).
static int qgemm_mt(uint32_t M, uint32_t K) {
    if (K >= 1u << 24) return 1;                           // offsets of a tile's tokens have 32 bits
    const uint32_t tiles = (M + 127u) / 128u;
    return (int)(((M + tiles - 1u) / tiles + 15u) / 16u);
}

// How a product is dealt to workgroups.
struct QgemmPlan {
    int mt;
    uint32_t wn, wk, groups, z, whole, tiles, ks, blocks, ks_blocks;
};
static QgemmPlan qgemm_plan(uint32_t M, uint32_t N, uint32_t K) {
    QgemmPlan g{};
    g.mt = qgemm_mt(M, K);
    g.wn = qgemm_wn(g.mt);
    g.z = (M + 16u * g.mt - 1u) / (16u * g.mt);
    g.groups = (N + 32u * g.wn - 1u) / (32u * g.wn);
    g.tiles = (g.z == 1u ? g.groups : (g.groups + 7u) / 8u * 8u) * g.z;
    const uint32_t all = (K + 511u) / 512u, slots = g.mt == 1 ? 512u : 256u;
    g.wk = 8u / g.wn;
    // Smaller workgroups, where that brings every slot one; not where half the units (three quarters, up to two tiles of tokens) have one already
    // whose waves take one block each and are eight a unit at most: fewer shares to write and add (SqueezeLLM 4 bits, us, by ranges of a workgroup:
    // 128 tokens 4096 -> 6144 24.9 with one, 23.7 with two (192 workgroups); 24 tokens 4096 -> 6144 14.5 with two, 13.5 with four (192), but 4096 -> 4096
    // 11.7 and 13.4 (128); 16 tokens 4096 -> 6144 13.1 with two, 16.5 with one, 4096 -> 1024 11.9 with four, 10.1 with one, 14336 -> 4096 22.4 and, with two, 20.4).
    while (g.wk > 1u && (uint64_t)g.tiles * (all / g.wk) < slots) {
        const uint32_t shares = g.tiles * (all / g.wk);
        if (shares >= (g.mt >= 3 ? 128u : 192u) && all % g.wk == 0u && shares * g.wn * g.wk <= 2048u) break;
        g.wk /= 2u;
    }
    g.blocks = (all + g.wk - 1u) / g.wk;
    g.whole = g.tiles / slots * slots;
    g.ks = 1u;
    const uint32_t left = g.tiles - g.whole;
    if (left > 0u) {
        // us: a block of every range of a tile takes 2.5 + 1.2 a token tile, sums of shares are written and read at about 4 TB/s, by a kernel more.  Fitted
        // ahead of copies that pass no register and of turns (4096 -> 28672, four blocks, one layer: 77 tokens 37, 128 50; now 34.6 and 42): a block of many tokens takes
        // less now than is said here, so that a split is taken a little more often than it pays
        const double block_us = 2.5 + 1.2 * g.mt, tile_us = 2.0 * 16.0 * g.mt * 32.0 * g.wn * 4.0 / 4e6;
        double best = 0.0;
        for (uint32_t ks = 1u; ks <= 16u && ks * g.wk <= all; ++ks) {
            const uint32_t turns = (left * ks + slots - 1u) / slots, steps = (all + ks * g.wk - 1u) / (ks * g.wk);
            const double us = turns * steps * block_us + (ks > 1u ? 3.0 + left * ks * tile_us : 0.0);
            if (ks == 1u || us < best) { best = us; g.ks = ks; }
        }
    }
    if (g.ks == 1u) g.whole = g.tiles;
    g.ks_blocks = (all + g.ks * g.wk - 1u) / (g.ks * g.wk);
    return g;
}

// Rows so long that the offsets of sixteen do not have 32 bits go one by one.
static bool qgemm_one_by_one(uint32_t M, uint32_t K) { return M > 1u && K >= 1u << 27; }

size_t qgemm_workspace(uint32_t M, uint32_t N, uint32_t K) {
    const QgemmPlan g = qgemm_plan(qgemm_one_by_one(M, K) ? 1u : M, N, K);
    return (size_t)(g.tiles - g.whole) * g.ks * 16u * g.mt * 32u * g.wn * sizeof(float);
}

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

template <int DT>
static hipError_t qgemm_dt(int fmt, int bits, bool flag, const QgemmParams& p, const QgemmPlan& g, hipStream_t s) {
    const hipError_t e = fmt == kAnyprec ? qgemm_bits<kAnyprec, DT>(bits, flag, p, g, s)
                       : fmt == kLutgemm ? qgemm_bits<kLutgemm, DT>(bits, flag, p, g, s) : qgemm_bits<kSqllm, DT>(bits, flag, p, g, s);
    if (e != hipSuccess || g.tiles == g.whole) return e;
    const uint32_t rows = 16u * g.mt, cols = 32u * g.wn;
    const uint32_t threads = rows * cols / (p.half != 0u && p.whole == 0u ? 16u : 8u);
    hipLaunchKernelGGL((qgemm_sum_kernel<DT>), dim3((threads + 255u) / 256u, g.tiles - g.whole), dim3(256), 0, s, p, rows, cols);
    return hipGetLastError();
}

// What stands where in a product that gates (QgemmParams::pairs), or false: a turn of the units ends among the token tiles of a column, whose sums are of both kinds then.
static bool qgemm_pairs(const QgemmPlan& g, uint32_t N, uint32_t* pairs, uint32_t* wholes) {
    *pairs = ~0u;
    *wholes = 0u;
    if (N % 16u != 0u) return false;
    if (g.whole == 0u || g.whole == g.tiles) return true;
    if (N % 32u != 0u || (g.z > 1u && g.whole % (8u * g.z) != 0u)) return false;
    const uint32_t whole = std::min(g.whole / g.z * g.wn, N / 32u);           // wave columns
    if (4u * whole < N / 16u) return false;                // all gates are of whole tiles
    *pairs = 2u * whole - N / 32u;
    *wholes = whole;
    return true;
}

bool qgemm_gates(int fmt, int bits, uint32_t M, uint32_t N, uint32_t K, uint32_t group) {
    uint32_t pairs, wholes;
    return (N % 16u == 0u && qgemm_form(fmt, bits, M, N, K, group) == 1) || qgemm_pairs(qgemm_plan(qgemm_one_by_one(M, K) ? 1u : M, N, K), N, &pairs, &wholes);
}

int qgemm_form(int fmt, int bits, uint32_t M, uint32_t N, uint32_t K, uint32_t group) {
    return qgemm_one_by_one(M, K) ? 2 : qgemm_goes_wide(fmt, bits, M, N, K, group) ? 1 : 0;
}

hipError_t launch_qgemm(int fmt, int dt, int bits, const void* x, const uint32_t* q, const void* lut, const void* q_bias, void* out,
                        void* workspace, uint32_t M, uint32_t N, uint32_t K, uint32_t group, bool gate_up, hipStream_t s) {
    if (gate_up && (!qgemm_gates(fmt, bits, M, N, K, group) || ((uintptr_t)out % 16u) != 0)) return hipErrorInvalidValue;
    if (qgemm_one_by_one(M, K)) {
        for (size_t m = 0; m < M; ++m) {
            const hipError_t e = launch_qgemm(fmt, dt, bits, (const uint16_t*)x + m * K, q, lut, q_bias, (uint16_t*)out + m * (gate_up ? N / 2u : N), workspace, 1u, N, K, group,
                                              gate_up, s);
            if (e != hipSuccess) return e;
        }
        return hipSuccess;
    }
    const QgemmPlan g = qgemm_plan(M, N, K);
    QgemmParams p{};
    p.x = x; p.q = q; p.lut = lut; p.q_bias = q_bias; p.out = out; p.part = (float*)workspace;
    p.M = M; p.N = N; p.K = K; p.group = group;
    p.groups = g.groups; p.z = g.z; p.wk = g.wk; p.whole = g.whole; p.ks = g.ks; p.blocks = g.blocks; p.ks_blocks = g.ks_blocks;
    const bool flag = fmt == kAnyprec ? K % 64u == 0 && ((uintptr_t)q % 8u) == 0 : N < 1u << 24 && (fmt == kSqllm || group % 128u == 0);
    p.half = gate_up ? N / 2u : 0u;
    p.wide = N % 8u == 0 && ((uintptr_t)out % 16u) == 0;
    p.pairs = gate_up ? ~0u : 0u;
    if (qgemm_goes_wide(fmt, bits, M, N, K, group)) return launch_qgemm_wide(fmt, dt, bits, p, s);
    if (gate_up) qgemm_pairs(g, N, &p.pairs, &p.wholes);
    return dt == kFP16 ? qgemm_dt<kFP16>(fmt, bits, flag, p, g, s) : qgemm_dt<kBF16>(fmt, bits, flag, p, g, s);
}

}  // namespace decdec
