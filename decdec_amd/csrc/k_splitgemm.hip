// Products of many tokens with a dense 32-bit weight, out[m][n] = sum_k x[m][k] w[n][k], on the fp16 units of the matrix cores.
//
// A float times a power of two that brings its row near 1 is almost the sum of two fp16 numbers of eleven significant bits each,
// s x = x1 + x2 (s x rounded, and what is left rounded): a quarter of all numbers lose their last bit, none more.  Three products
// x1 w2 + x2 w1 + x1 w1 are added up in fp32; what is left out, x2 w2, is at most 2^-22 of x w.  Per product these errors have a root of
// the mean square of 2^-23.7, and a sum of K products has them as it has K roundings, while the fp32 sums themselves err by more from a
// few hundred terms on, and by less here than in six bf16 products (k_rowgemm.hip), since a half as many are added, in two sums.  Error
// against 64 bits, norm over norm, normal x and w, this / six bf16 products / the fp32 library product: K 128 1.11 / 1.53 / 2.04e-7, 512 1.88 /
// 3.35 / 4.05e-7, 2048 3.59 / 7.00 / 8.12e-7, 7168 6.72 / 13.5 / 15.2e-7; with sizes spread by exp(2 randn) in x and exp(randn) in w 512 1.82 /
// 2.55 / 4.35e-7, 2048 3.37 / 5.54 / 8.21e-7, but 128 1.60 / 0.83 / 1.28e-7: K below 512 is left to six products.
//
// Scales.  The tokens' are by their rows' largest numbers, which a first kernel finds; it leaves the pieces in the order in which the
// product copies them to LDS.  The weight is read once, so its rows' scales are by 32 numbers from all over a row: 2^8 for the largest of
// them, so that numbers 128 times as large still fit.  fp16 ends at 2^-24: what a piece cannot hold is up to 2^-33 of the largest of the 32, in
// tokens 2^-39 of the largest of the row, and no longer 2^-23 of the number.  Where a row's small numbers are what counts (weights spread by
// channel and tokens the other way, a far channel that the other operand does not have), that would be all of the error.  So a workgroup takes six
// products of three bf16 pieces (pieces.h) in place of these, straight from memory, where
//   - numbers of one of its rows are too far apart (kRowLow, kSampleLow), or too large beside the 32 (their products are infinite or NaN then);
//   - a token is one number or nearly (its results are single products, no sum whose roundings are larger), or 32 numbers are zero and the row is not;
//   - a row holds infinities, NaN or nothing above 2^-96; where three pieces do not hold it either, it takes fp32 products.
// The 32 lie elsewhere in every row: a channel far from the others is in some row's.
// Error of 777 x 8448 x 2048, norm over norm, this / six products everywhere / pieces alone, under 2^5: normal numbers 3.6 / 7.0 / 3.6e-7, weights spread by
// exp(2 randn) along the channels and tokens the other way 4.9 / 7.0 / 5.5e-7 (777 x 2048 x 7168 5.1 / 5.5 / 23e-7, exp(2.5 randn) 4.7 / 5.5 / 451e-7), 1e4 in a
// channel in which tokens are zero 4.9 / 7.0 / 31e-7, one-hot tokens 0 / 0 / 0.4e-7.  us: 92 with pieces, 216 with six products, 220 - 295 where a row is
// seen to need them later; k_rowgemm.hip 175 (all without large products ahead).
//
// A workgroup of two groups of four waves owns 16 TM tokens x 256 outputs; the groups take a half of its steps of 32 channels each, and their
// sums meet in LDS.  A wave owns 64 outputs.  It reads their weights as they lie (four lanes to 64 bytes of a row: straight into operands,
// sixteen rows a quarter-wave, every lane is an access of its own, 50 a request, and those alone took longer than the products), splits
// them, and passes them through LDS of its own into operands; the tokens' pieces come to LDS by copies that pass no register, two steps
// ahead.  Splitting the next step's weights lies between this one's products.  A die takes neighbouring row blocks and panels, so that a
// panel of the weight is read by one of them, or two.
//
// What bounds it: products and the power they take.  777 x 14336 x 4096, two turns of the compute units for 1.53 of work: 331 us (827
// TFLOP/s of fp16 products at 2.06 GHz; matrix units busy 38 % of the cycles, waves at barriers and waits 26 %), 294 with all numbers one; a
// loop of nothing but these products of normal numbers reaches 1740 TFLOP/s, of zeros 2170.  Weights read straight into operands: 382;
// one group of four waves and its own ranges of K, 300, but 100 for 87 at 777 x 7168 x 2048, where the ranges' sums pass memory; one wave a
// SIMD with every operand two or four steps ahead, 510.  Measured, us a call with the first kernel and the sums, behind large products (clocks are
// 5 - 10 % higher without), this / six bf16 products / the library: 777 x 8448 x 2048 99 / 196 / 243, 777 x 4096 x 4096 106 / 172 / 220, 777 x 2048 x
// 2048 49 / 64 / 65, 200 x 8448 x 2048 54 / 67 / 71; looking for rows that are no pieces is 1 - 2 us of these.
#include "mixers.h"
#include "pieces.h"

namespace decdec {

struct SplitGemm {
    const float* x;              // [M][ldx]
    const float* w;              // [N][ldw]
    float* out;                  // [M][ldo], or with several ranges of K [range][M][N]
    unsigned char* pieces;       // [row block][step][piece][row][32] fp16
    int* exps;                   // [M]: the power of two that a row's pieces are short of, or kNoPieces
    uint32_t M, N, K, ldx, ldw, ldo, ks, steps, blocks, rows;      // steps of a range, row blocks, rows of one
    uint32_t wide;               // four neighbouring outputs may be stored at once
};

constexpr int kNoPieces = 0x7FFFFFFF;
constexpr int kRowExp = 14, kSampleExp = 8;        // of the largest number of a token's row, of a weight row's sample
// Numbers below 2^-20 of a token's largest one, or 2^-14 of the largest of a weight row's sample, keep 20 bits or fewer.  Rows with more of them than
// chance has in a bell-shaped one are left to six products: a quarter of a token's, six of a sample's 32.
constexpr float kRowLow = 9.5367432e-7f, kSampleLow = 6.1035156e-5f;
constexpr uint32_t kSampleFew = 5u;
constexpr uint32_t kSplitBN = 256, kStages = 3;

// Place of the 16-byte piece g of a row of 32 numbers: the sixteen lanes of a phase of a 16-byte LDS read are rows 0-3 and 12-15 with one
// g and rows 4-11 with its neighbour.  Piece g holds numbers 4 g .. + 3 and 16 + 4 g .. + 3, in x and w alike: four lanes that
// read four numbers each of either half have 64 bytes of memory side by side.
__device__ __forceinline__ uint32_t split_place(uint32_t row, uint32_t g) { return ((row >> 2) & 3u) ^ ((0x2130u >> (4u * g)) & 3u); }
__device__ __forceinline__ void split_load(const float* p, float (&v)[8]) {
    const f32x4 a = *(const f32x4*)p, b = *(const f32x4*)(p + 16);
#pragma unroll
    for (int i = 0; i < 4; ++i) { v[i] = a[i]; v[4 + i] = b[i]; }
}
__device__ __forceinline__ void split_pieces(const float (&v)[8], float scale, u32x4 (&o)[2]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float x = v[2 * i], y = v[2 * i + 1];
        half2_t h = {(_Float16)(x * scale), (_Float16)(y * scale)};
        uint32_t a, b;
        __builtin_memcpy(&a, &h, 4);
        asm("" : "+v"(a));                                 // or each half is rounded once more to be subtracted
        __builtin_memcpy(&h, &a, 4);
        const half2_t r = {(_Float16)__builtin_fmaf(x, scale, -(float)h[0]), (_Float16)__builtin_fmaf(y, scale, -(float)h[1])};
        __builtin_memcpy(&b, &r, 4);
        o[0][i] = a;
        o[1][i] = b;
    }
}
__device__ __forceinline__ float split_most(const float (&v)[8], float most) {
#pragma unroll
    for (int i = 0; i < 8; ++i) most = fmaxf(most, fabsf(v[i]));
    return most;
}
// scale that gives `most` (a normal number) the exponent `to`, and the power of two that it takes away
__device__ __forceinline__ int split_scale(float most, int to, float& scale) {
    const int up = to - ((int)(__float_as_uint(most) >> 23) - 127);
    scale = __uint_as_float((uint32_t)(127 + up) << 23);
    return -up;
}

// Scales and pieces of the tokens, and which of them have none: a workgroup a row.  777 x 2048 6 us, 777 x 7168 10.
__global__ __launch_bounds__(256) void split_rows_kernel(const SplitGemm p) {
    __shared__ float red[4], sizes[4];
    __shared__ uint32_t counts[8];
    const uint32_t m = blockIdx.x, tid = threadIdx.x, units = p.K / 8u, row = m % p.rows;
    const float* x = p.x + (size_t)m * p.ldx;
    float v[2][8], most = 0.f;                             // the row's first 4096 numbers stay in registers
    auto at = [&](uint32_t u) { return x + 32u * (u >> 2) + 4u * (u & 3u); };
#pragma unroll
    for (uint32_t c = 0; c < 2u; ++c)
        if (tid + 256u * c < units) {
            split_load(at(tid + 256u * c), v[c]);
            most = split_most(v[c], most);
        }
    for (uint32_t u = tid + 512u; u < units; u += 256u) {
        float t[8];
        split_load(at(u), t);
        most = split_most(t, most);
    }
#pragma unroll
    for (int s = 1; s < 64; s <<= 1) most = fmaxf(most, __shfl_xor(most, s, 64));
    if ((tid & 63u) == 0u) red[tid >> 6] = most;
    __syncthreads();
    most = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    const bool bad = most > 3.3e38f || (most > 0.f && most < 1.2621774e-29f);
    float scale = 1.f;
    const int e = bad || most == 0.f ? 0 : split_scale(most, kRowExp, scale);
    const float cut = most * kRowLow;
    uint32_t low = 0u, some = 0u;                          // numbers that are small, and any but zero
    float size = 0.f;
    unsigned char* block = p.pieces + (size_t)(m / p.rows) * (p.K / 32u) * (p.rows * 128u) + row * 64u;
    auto put = [&](uint32_t u, const float (&t)[8]) {
        u32x4 o[2];
        split_pieces(t, scale, o);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            low += t[i] != 0.f && fabsf(t[i]) < cut ? 1u : 0u;
            some += t[i] != 0.f ? 1u : 0u;
            size += fabsf(t[i]);
        }
        unsigned char* d = block + (size_t)(u >> 2) * (p.rows * 128u) + 16u * split_place(row, u & 3u);
        *(u32x4*)d = o[0];
        *(u32x4*)(d + p.rows * 64u) = o[1];
    };
#pragma unroll
    for (uint32_t c = 0; c < 2u; ++c)
        if (tid + 256u * c < units) put(tid + 256u * c, v[c]);
    for (uint32_t u = tid + 512u; u < units; u += 256u) {
        float t[8];
        split_load(at(u), t);
        put(u, t);
    }
#pragma unroll
    for (int s = 1; s < 64; s <<= 1) { low += __shfl_xor(low, s, 64); some += __shfl_xor(some, s, 64); size += __shfl_xor(size, s, 64); }
    if ((tid & 63u) == 0u) { counts[tid >> 6] = low; counts[4u + (tid >> 6)] = some; sizes[tid >> 6] = size; }
    __syncthreads();
    if (tid != 0u) return;
    for (uint32_t w = 1; w < 4u; ++w) { low += counts[w]; some += counts[4u + w]; size += sizes[w]; }
    // a row that is one number, or nearly: results are single products, which six of them give in full
    p.exps[m] = bad || low > some / 4u || size < 1.5f * most ? kNoPieces : e;
}

template <int TM>
__global__ __launch_bounds__(512, 2) void split_gemm_kernel(const SplitGemm p) {
    constexpr int TN = 4;
    constexpr uint32_t ROWS = 16u * TM, PIECE = ROWS * 64u, BUFFER = 2u * PIECE, COPIES = BUFFER / 1024u, GROUP = kStages * BUFFER + 4u * TN * 2048u;
    extern __shared__ __align__(1024) unsigned char smem[];      // a group: [stage][piece][row][32] fp16 of x, [wave][tile][piece][16][32] of w
    __shared__ int exp_x[ROWS], exp_w[2][kSplitBN];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = __builtin_amdgcn_readfirstlane(tid >> 6), l16 = lane & 15u, lg = lane >> 4;
    const uint32_t group = wave >> 2, wn = (wave & 3u) * 64u;
    const uint32_t id = (blockIdx.x & 7u) * (gridDim.x >> 3) + (blockIdx.x >> 3), panel = id / p.blocks, cols = (p.N + kSplitBN - 1u) / kSplitBN;
    if (panel >= cols * p.ks) return;
    const uint32_t range = panel / cols, n0 = panel % cols * kSplitBN + wn, mb = id % p.blocks, m0 = mb * ROWS;
    const uint32_t all = p.K / 32u, begin = range * p.steps < all ? range * p.steps : all, end = begin + p.steps < all ? begin + p.steps : all;
    const uint32_t turns = (end - begin + 1u) / 2u, first = begin + group * turns < end ? begin + group * turns : end;
    const uint32_t last = first + turns < end ? first + turns : end;
    bool again = false;
    if (tid < ROWS) {
        const int e = m0 + tid < p.M ? p.exps[m0 + tid] : 0;
        exp_x[tid] = e;
        again = e == kNoPieces;
    }
    again = __syncthreads_or(again);
    // rows past the end repeat the last one and are never stored
    const float* wb = p.w + (size_t)(n0 < p.N ? n0 : 0u) * p.ldw;
    const uint32_t left = n0 < p.N ? p.N - 1u - n0 : p.N - 1u;
    uint32_t wo[TN];
#pragma unroll
    for (uint32_t i = 0; i < (uint32_t)TN; ++i) {
        const uint32_t r = 16u * i + (lane >> 2);
        wo[i] = (r < left ? r : left) * p.ldw + 4u * (lane & 3u);
    }
    f32x4 acc[TN][TM];
    auto clear = [&] {
#pragma unroll
        for (int i = 0; i < TN; ++i)
#pragma unroll
            for (int j = 0; j < TM; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    };
    clear();
    if (!again) {                                          // the same in all waves
        unsigned char* xs = smem + group * GROUP;
        unsigned char* own = xs + kStages * BUFFER + (wave & 3u) * (TN * 2048u);
        const uint32_t src = l16 * 64u + 16u * split_place(l16, lg), put = (lane >> 2) * 64u + 16u * split_place(lane >> 2, lane & 3u);
        float w[TN][8], scale_w[TN];
        auto inside = [&](uint32_t step) { return step < last ? step : (last > begin ? last - 1u : begin < all ? begin : 0u); };   // what is requested past the end is not used
        auto request_w = [&](uint32_t step) {
            const float* y = wb + (size_t)inside(step) * 32u;
#pragma unroll
            for (int i = 0; i < TN; ++i) split_load(y + wo[i], w[i]);
        };
        const unsigned char* image = p.pieces + (size_t)mb * all * BUFFER + 16u * lane;
        // a wave copies every fourth kilobyte
        auto request_x = [&](uint32_t step, uint32_t stage) {
            const unsigned char* from = image + (size_t)inside(step) * BUFFER;
            const uint32_t to = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)xs + stage * BUFFER;
#pragma unroll
            for (uint32_t c = 0; c < (COPIES + 3u) / 4u; ++c) {
                const uint32_t k = (wave & 3u) + 4u * c;
                if (k < COPIES)
                    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off"
                                 : : "s"(__builtin_amdgcn_readfirstlane(to + 1024u * k)), "v"(from + 1024u * k) : "memory");
            }
        };
        auto split = [&] {
#pragma unroll
            for (int i = 0; i < TN; ++i) {
                u32x4 o[2];
                split_pieces(w[i], scale_w[i], o);
                *(u32x4*)(own + 2048u * i + put) = o[0];
                *(u32x4*)(own + 2048u * i + 1024u + put) = o[1];
            }
        };
        request_x(first, 0u);
        request_w(first);
        request_x(first + 1u, 1u);
        {
            const uint32_t count = last > first ? last - first : 1u, base = inside(first);
            bool none[TN];
#pragma unroll
            for (int i = 0; i < TN; ++i) {
                float v[8];
                // elsewhere in every row, so that channels far from the others are in some row's sample
                split_load(wb + wo[i] + (size_t)(base + count * (64u * (lane & 3u) + 16u * (uint32_t)i + (lane >> 2)) / 256u) * 32u, v);
                float most = split_most(v, 0.f);
                most = fmaxf(most, __shfl_xor(most, 1, 64));
                most = fmaxf(most, __shfl_xor(most, 2, 64));
                none[i] = most == 0.f;
                uint32_t low = 0u;
#pragma unroll
                for (int e = 0; e < 8; ++e) low += v[e] != 0.f && fabsf(v[e]) < most * kSampleLow ? 1u : 0u;
                low += __shfl_xor(low, 1, 64);
                low += __shfl_xor(low, 2, 64);
                again |= low > kSampleFew;
                const bool fits = most > 1.2621774e-29f && most < 3.3e38f;
                scale_w[i] = 1.f;
                const int e = fits ? split_scale(most, kSampleExp, scale_w[i]) : 0;
                if ((lane & 3u) == 0u) exp_w[group][wn + 16u * i + (lane >> 2)] = e;
                again |= !fits && !none[i];
            }
#pragma unroll
            for (int i = 0; i < TN; ++i)
                if (__any(none[i]))                        // a row of zeros, or only its sample?
                    for (uint32_t step = first; step < last; ++step) {
                        float v[8];
                        split_load(wb + wo[i] + (size_t)step * 32u, v);
                        again |= none[i] && !(split_most(v, 0.f) == 0.f);
                    }
        }
        split();
        request_w(first + 1u);
        uint32_t stage = 0u;
        const uint32_t count = __syncthreads_or(again) ? 0u : turns;
        // every group takes part in all turns: the barrier is the workgroup's
        for (uint32_t t = 0; t < count; ++t) {
            // What was requested two steps ago is there: the weights requested after it have been waited for (and the pieces written).
            asm volatile("s_waitcnt vmcnt(12) lgkmcnt(0)" ::: "memory");
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
            const uint32_t step = first + t, ahead = stage >= 1u ? stage - 1u : 2u;
            if (step < last) {
                const unsigned char* buf = xs + stage * BUFFER + src;
                u32x4 a[TN][2], b[TM][2];
#pragma unroll
                for (int i = 0; i < TN; ++i)
#pragma unroll
                    for (int k = 0; k < 2; ++k) a[i][k] = *(const u32x4*)(own + 2048u * i + 1024u * k + src);
#pragma unroll
                for (int j = 0; j < TM; ++j)
#pragma unroll
                    for (int k = 0; k < 2; ++k) b[j][k] = *(const u32x4*)(buf + PIECE * k + 1024u * j);
                split();                                   // of the next step; a wave's LDS accesses stay in order
                request_x(step + 2u, ahead);               // read last before this step's barrier
                request_w(step + 2u);
                // the small products first; of the first tile those of one output after another, as its operands arrive
#pragma unroll
                for (int j = 0; j < TM; ++j)
#pragma unroll
                    for (int q = 0; q < 12; ++q) {
                        const int k = j == 0 ? q % 3 : q / 4, i = j == 0 ? q / 3 : q % 4;
                        Frag<kFP16> f, g;
                        f.v = a[i][k == 0];
                        g.v = b[j][k == 1];
                        mma(f, g, acc[i][j]);
                    }
                __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
#pragma unroll
                for (int i = 0; i < TN; ++i) {
                    __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
                    __builtin_amdgcn_sched_group_barrier(0x008, 3, 0);
                }
#pragma unroll
                for (int j = 1; j < TM; ++j)
#pragma unroll
                    for (int k = 0; k < 12; ++k) {
                        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                        __builtin_amdgcn_sched_group_barrier(0x002, 1, 0);
                        if (k % 6 == 5 && j + 1 < TM) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                        if (k == 11 && j > 1) __builtin_amdgcn_sched_group_barrier(0x200, 2, 0);
                    }
            }
            stage = stage + 1u < kStages ? stage + 1u : 0u;
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
        for (int i = 0; i < TN; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int ew = exp_w[group][wn + 16u * i + 4u * lg + (uint32_t)e];
#pragma unroll
                for (int j = 0; j < TM; ++j) {
                    again |= !(fabsf(acc[i][j][e]) < __builtin_inff()) && m0 + 16u * (uint32_t)j + l16 < p.M;      // pieces past the end are what memory held
                    acc[i][j][e] = __builtin_ldexpf(acc[i][j][e], ew + exp_x[16 * j + (int)l16]);
                }
            }
    }
    if (__syncthreads_or(again)) {
        // straight from memory: six products of three bf16 pieces, and where those hold a row as little, fp32 products (as in k_rowgemm.hip)
        auto weights = [&](uint32_t step, uint32_t i) {
            const uint32_t r = 16u * i + l16;
            Frag<kFP32> f;
            split_load(wb + (size_t)(r < left ? r : left) * p.ldw + step * 32u + 4u * lg, f.v);
            return f;
        };
        auto tokens = [&](uint32_t step, uint32_t j) {
            const uint32_t r = m0 + 16u * j + l16;
            Frag<kFP32> f;
            split_load(p.x + (size_t)(r < p.M ? r : p.M - 1u) * p.ldx + step * 32u + 4u * lg, f.v);
            asm volatile("" ::: "memory");                 // one tile's at a time: registers
            return f;
        };
        float most_w[TN] = {}, most_x[TM] = {};
        clear();
        for (uint32_t step = first; step < last; ++step) {
            u32x4 a[TN][3];
#pragma unroll
            for (uint32_t i = 0; i < (uint32_t)TN; ++i) pieces_of(weights(step, i), a[i], most_w[i]);
#pragma unroll
            for (int j = 0; j < TM; ++j) {
                u32x4 b[3];
                pieces_of(tokens(step, (uint32_t)j), b, most_x[j]);
                six_products<TN>(a, b, [&](int i) -> f32x4& { return acc[i][j]; });
            }
        }
        again = false;
#pragma unroll
        for (int i = 0; i < TN; ++i) again |= !in_three_pieces(most_w[i], 16, 32);
#pragma unroll
        for (int j = 0; j < TM; ++j) again |= !in_three_pieces(most_x[j], 16, 32);
        if (__syncthreads_or(again)) {
            clear();
            for (uint32_t step = first; step < last; ++step) {
                Frag<kFP32> f[TN];
#pragma unroll
                for (uint32_t i = 0; i < (uint32_t)TN; ++i) f[i] = weights(step, i);
#pragma unroll
                for (int j = 0; j < TM; ++j) {
                    const Frag<kFP32> x = tokens(step, (uint32_t)j);
#pragma unroll
                    for (int i = 0; i < TN; ++i) mma(f[i], x, acc[i][j]);
                }
            }
        }
        __syncthreads();
    }
    // the second group's sums pass LDS, which nothing else uses any more
    f32x4* sums = (f32x4*)smem + (tid & 255u);
    if (group == 1u) {
#pragma unroll
        for (int i = 0; i < TN; ++i)
#pragma unroll
            for (int j = 0; j < TM; ++j) sums[(i * TM + j) * 256] = acc[i][j];
    }
    __syncthreads();
    if (group == 1u) return;
#pragma unroll
    for (int j = 0; j < TM; ++j) {
        const uint32_t m = m0 + 16u * j + l16;
#pragma unroll
        for (int i = 0; i < TN; ++i) {
            const uint32_t n = n0 + 16u * (uint32_t)i + 4u * lg;
            const f32x4 v = acc[i][j] + sums[(i * TM + j) * 256];
            if (m >= p.M || n >= p.N) continue;
            float* dst = p.out + (p.ks > 1u ? ((size_t)range * p.M + m) * p.N : (size_t)m * p.ldo) + n;
            if (p.wide) *(f32x4*)dst = v;
            else
#pragma unroll
                for (uint32_t e = 0; e < 4u; ++e) if (n + e < p.N) dst[e] = v[e];
        }
    }
}

// Tiles of 16 tokens in a workgroup and ranges of K, by the time that they take.  Fitted to 500 products of 14 shapes, 160 - 800 tokens x 2048 -
// 17408 outputs x 512 - 14336 channels, which it meets within 4 % on average: 7.2 us for the first kernel and the launches, 3.5 and 1.18 +
// 0.15 TM a step for each turn of the compute units, a range's sums through memory.  Its choice is 1.002 times as slow as the best one.
SplitPlan split_plan(uint32_t M, uint32_t N, uint32_t K) {
    const uint32_t all = K / 32u, cols = (N + kSplitBN - 1u) / kSplitBN;
    SplitPlan best{0u, 0u, __builtin_inff()};
    if (K < 512u || K % 32u != 0u) return best;            // the error above, and whole steps
    for (uint32_t tm = 4u; tm <= 7u; ++tm)
        for (uint32_t ks = 1u; ks <= 16u && 4u * ks <= all; ++ks) {
            const uint64_t groups = (uint64_t)((M + 16u * tm - 1u) / (16u * tm)) * cols * ks;
            if (groups > 0x7FFFFFF0u) continue;
            const float turns = (float)((groups + 255u) / 256u), half = (float)(((all + ks - 1u) / ks + 1u) / 2u);
            float us = 7.2f + turns * (3.5f + half * (1.18f + 0.15f * (float)tm));
            if (ks > 1u) us += 3.7f + (float)ks * (float)M * (float)N * 8.f / 3.8e6f;
            if (us < best.us) best = {tm, ks, us};
        }
    return best;
}

// exponents, pieces, the ranges' sums
static size_t split_pieces_at(uint32_t M) { return ((size_t)M * sizeof(int) + 255u) / 256u * 256u; }
static size_t split_sums_at(const SplitPlan& plan, uint32_t M, uint32_t K) {
    const size_t rows = 16u * plan.tm;
    return split_pieces_at(M) + (M + rows - 1u) / rows * rows * K * 4u;
}
size_t split_workspace(const SplitPlan& plan, uint32_t M, uint32_t N, uint32_t K) {
    return split_sums_at(plan, M, K) + (plan.ks > 1u ? (size_t)plan.ks * M * N * sizeof(float) : 0u);
}
float* split_sums(const SplitPlan& plan, void* ws, uint32_t M, uint32_t K) { return (float*)((unsigned char*)ws + split_sums_at(plan, M, K)); }

template <int TM>
static hipError_t split_launch(const SplitGemm& p, hipStream_t s) {
    constexpr size_t lds = 2u * (kStages * 16u * TM * 128u + 4u * 4u * 2048u);
    static_assert(lds >= 4u * TM * 4096u, "the second group's sums");
    if (hipError_t e = allow_lds<split_gemm_kernel<TM>>(lds); e != hipSuccess) return e;
    const uint32_t groups = (p.N + kSplitBN - 1u) / kSplitBN * p.ks * p.blocks;
    hipLaunchKernelGGL((split_gemm_kernel<TM>), dim3((groups + 7u) / 8u * 8u), dim3(512), lds, s, p);
    return hipGetLastError();
}

hipError_t launch_split_gemm(const SplitPlan& plan, const float* x, uint32_t ldx, const float* w, uint32_t ldw, float* out, uint32_t ldo, void* ws,
                             uint32_t M, uint32_t N, uint32_t K, bool wide, hipStream_t s) {
    const uint32_t rows = 16u * plan.tm;
    const SplitGemm p{x, w, plan.ks > 1u ? split_sums(plan, ws, M, K) : out, (unsigned char*)ws + split_pieces_at(M), (int*)ws, M, N, K, ldx, ldw, ldo,
                      plan.ks, (K / 32u + plan.ks - 1u) / plan.ks, (M + rows - 1u) / rows, rows, wide ? 1u : 0u};
    hipLaunchKernelGGL(split_rows_kernel, dim3(M), dim3(256), 0, s, p);
    if (hipError_t e = hipGetLastError(); e != hipSuccess) return e;
    switch (plan.tm) {
        case 4u: return split_launch<4>(p, s);
        case 5u: return split_launch<5>(p, s);
        case 6u: return split_launch<6>(p, s);
        default: return split_launch<7>(p, s);
    }
}

}  // namespace decdec
