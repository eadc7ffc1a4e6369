// Products of several tokens with a dense weight, out[m][n] = sum_k x[m][k] w[n][k], for the shapes in which they are a decoder's
// own: 32-bit storage, and few tokens.
//
// 32-bit operands, where pieces of fp16 (k_splitgemm.hip) are not faster: the matrix cores multiply fp32 at a sixteenth of their bf16 rate.  A
// float is exactly the sum of three numbers (pieces.h) of eight significant bits each, x = x1 + x2 + x3 (x rounded to bf16, the same of what is left, and what is left then), so x w is
// the sum of nine exact bf16 products.  Six of them (x1 w1, x1 w2, x2 w1, x2 w2, x1 w3, x3 w1) are added up in fp32, which rounds
// no more often than fp32 products do (32 terms an instruction instead of four).  x2 is at most 2^-8 of x and x3 2^-17, so that each
// of x2 w3 and x3 w2 may reach 2^-25 of x w and what is left out 2^-24 of it, the rounding of one fp32 product; the root of
// its mean square over all significands is 2^-27.5.  Infinities and numbers that bf16 would round to one have no three pieces, and the
// pieces of numbers below about 2^-110 end where bf16 does: a workgroup that has seen one of the former, or a row (of x or w) whose
// largest number is below 2^-96, starts again with fp32 products.
// Error against 64 bits, norm of the difference over norm of the result: 777 x 264 x 2048 2.1e-7, the fp32 library product 8.1e-7;
// 100 x 257 x 1000 1.6e-7 and 2.9e-7.
//
// A workgroup of four waves owns 16 TM tokens x 128 outputs, a wave 32 of these.  Weights are the left operand and each of them
// meets one wave, so a wave reads its own straight into operands (and splits them); the tokens pass LDS, as bf16 (split on the way
// in), in rows of 32 elements whose 16-byte pieces are dealt so that the lanes that read together hit all banks (with the weights
// in LDS as well, its bandwidth was the bound).  The next step is requested into registers while the present one is multiplied,
// one barrier a step.  A lane ends with four neighbouring outputs of a token.  Where a shape has too few tiles for the GPU, ranges
// of K go to different workgroups and a second kernel adds their sums in order.
//
// Measured, us a call, beside the library: fp32 160 x 2048 x 2048 23 / 21, 777 x 2048 x 128 10 / 9;
// bf16 16 x 2048 x 2048 12 / 20, 16 x 20480 x 4096 42 / 69.
#include "mixers.h"
#include "pieces.h"

namespace decdec {

struct RowGemm {
    const void* x;               // [M][ldx]
    const void* w;               // [N][ldw]
    void* out;                   // [M][ldo]
    float* part;                 // [ks][M][N] where ks > 1
    uint32_t M, N, K, ldx, ldw, ldo, ks, steps;      // steps of a range
    uint32_t wide;               // four neighbouring outputs may be stored at once
};

template <int DT> struct GemmShape;
template <> struct GemmShape<kBF16> { static constexpr int pieces = 1, blocks = 2; };        // blocks of 32 elements a step
template <> struct GemmShape<kFP32> { static constexpr int pieces = 3, blocks = 1; };

// Eight neighbouring elements as bf16 pieces.
__device__ __forceinline__ void pieces_of(const Frag<kBF16>& f, u32x4 (&p)[1], float&) { p[0] = f.v; }

// Place of the 16-byte piece g (elements 8 g ..) of a row of 32: the sixteen lanes of a phase of a 16-byte LDS read are rows 0-3 and
// 12-15 with one g and rows 4-11 with its neighbour.
__device__ __forceinline__ uint32_t piece_at(uint32_t row, uint32_t g) { return ((row >> 2) & 3u) ^ ((0x2130u >> (4u * g)) & 3u); }

constexpr uint32_t kGemmBN = 128;

// Up to seven tiles of fp32 three workgroups share a unit, in 168 registers.  With seven the compiler has to be told: it takes 184,
// and 777 x 2048 x 7168 takes 180 us for 158; told so with fewer, it takes less than it may (six tiles, 777 x 7168 x 2048: 192 for 186).
template <int DT, int TM>
__global__ __launch_bounds__(256, DT == kFP32 && TM == 7 ? 3 : 2) void row_gemm_kernel(const RowGemm p) {
    using T = typename LaneOf<DT>::t;
    constexpr int P = GemmShape<DT>::pieces, KB = GemmShape<DT>::blocks, TN = 2;
    constexpr uint32_t ROWS = 16u * TM, STEP = 32u * KB;
    constexpr uint32_t TASKS = (ROWS * 4u * KB + 255u) / 256u;             // a task: eight elements of x
    constexpr uint32_t BLOCK = ROWS * 64u * P, BUFFER = BLOCK * KB;
    extern __shared__ __align__(16) unsigned char smem[];                  // [2][block][piece][row][32] bf16
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6, l16 = lane & 15u, lg = lane >> 4;
    const uint32_t n0 = blockIdx.x * kGemmBN, m0 = blockIdx.y * ROWS, wn = wave * 16u * TN;
    const uint32_t first = blockIdx.z * p.steps, all = (p.K + STEP - 1u) / STEP;
    const uint32_t last = first + p.steps < all ? first + p.steps : all;
    // task -> row, and piece of eight elements: four rows of a block of 32 elements are neighbours, so that sixteen lanes fill all banks
    auto task_row = [&](uint32_t id) { return KB == 1 ? id >> 2 : (id >> 5) * 4u + ((id >> 2) & 3u); };
    auto task_piece = [&](uint32_t id) { return (id & 3u) + (KB == 1 ? 0u : 4u * ((id >> 4) & 1u)); };
    Frag<DT> held[TASKS], w0[TN][KB], w1[TN][KB];
    float most_x[TASKS] = {}, most_w[TN] = {};              // largest sizes of a row
    auto request_x = [&](uint32_t step) {
#pragma unroll
        for (uint32_t t = 0; t < TASKS; ++t) {
            const uint32_t id = tid + 256u * t, r = m0 + task_row(id), c = step * STEP + 8u * task_piece(id);
            held[t] = frag_load<DT>((const T*)p.x + (size_t)(r < p.M ? r : p.M - 1u) * p.ldx + (c < p.K ? c : 0u));   // K is a multiple of 8
        }
    };
    const T* wrow[TN];
#pragma unroll
    for (uint32_t i = 0; i < (uint32_t)TN; ++i) {
        const uint32_t n = n0 + wn + 16u * i + l16;
        wrow[i] = (const T*)p.w + (size_t)(n < p.N ? n : p.N - 1u) * p.ldw;
    }
    auto request_w = [&](Frag<DT> (&w)[TN][KB], uint32_t step) {
#pragma unroll
        for (int kb = 0; kb < KB; ++kb)
#pragma unroll
            for (int i = 0; i < TN; ++i) {
                const uint32_t c = step * STEP + 32u * (uint32_t)kb + 8u * lg;
                w[i][kb] = frag_load<DT>(wrow[i] + (c < p.K ? c : 0u));
            }
    };
    auto put = [&](unsigned char* buf, uint32_t step) {
        const bool tail = (step + 1u) * STEP > p.K;
#pragma unroll
        for (uint32_t t = 0; t < TASKS; ++t) {
            const uint32_t id = tid + 256u * t, row = task_row(id), k = task_piece(id);
            if (ROWS * 4u * KB % 256u != 0 && row >= ROWS) break;
            if (tail && step * STEP + 8u * k >= p.K) held[t] = Frag<DT>{};
            u32x4 pc[P];
            pieces_of(held[t], pc, most_x[t]);
            unsigned char* dst = buf + (k >> 2) * BLOCK + row * 64u + 16u * piece_at(row, k & 3u);
#pragma unroll
            for (int j = 0; j < P; ++j) *(u32x4*)(dst + (uint32_t)j * ROWS * 64u) = pc[j];
        }
    };
    f32x4 acc[TN][TM];
#pragma unroll
    for (int i = 0; i < TN; ++i)
#pragma unroll
        for (int j = 0; j < TM; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto advance = [&](Frag<DT> (&w)[TN][KB], Frag<DT> (&ahead)[TN][KB], uint32_t step) {
        unsigned char* buf = smem + (step & 1u) * BUFFER;
        put(buf, step);
        __syncthreads();                                   // one a step: the other buffer's readers passed it before
        if (step + 1u < last) {
            request_x(step + 1u);
            request_w(ahead, step + 1u);
        }
#pragma unroll
        for (int kb = 0; kb < KB; ++kb) {
            u32x4 a[TN][P];
#pragma unroll
            for (int i = 0; i < TN; ++i) {
                if ((step + 1u) * STEP > p.K && step * STEP + 32u * (uint32_t)kb + 8u * lg >= p.K) w[i][kb] = Frag<DT>{};
                pieces_of(w[i][kb], a[i], most_w[i]);
            }
#pragma unroll
            for (int j = 0; j < TM; ++j) {
                const uint32_t row = 16u * j + l16;
                u32x4 b[P];
#pragma unroll
                for (int s = 0; s < P; ++s)
                    b[s] = *(const u32x4*)(buf + (uint32_t)kb * BLOCK + (uint32_t)s * ROWS * 64u + row * 64u + 16u * piece_at(row, lg));
                if constexpr (P == 3) six_products<TN>(a, b, [&](int i) -> f32x4& { return acc[i][j]; });
                else
#pragma unroll
                    for (int i = 0; i < TN; ++i) {
                        Frag<kBF16> f, x;
                        f.v = a[i][0];
                        x.v = b[0];
                        mma(f, x, acc[i][j]);
                    }
            }
        }
    };
    if (first < last) {
        request_x(first);
        request_w(w0, first);
    }
    for (uint32_t step = first; step < last; step += 2u) {
        advance(w0, w1, step);
        if (step + 1u < last) advance(w1, w0, step + 1u);
    }
    if constexpr (DT == kFP32) {
        // Numbers that are no three pieces (see above): four neighbouring lanes staged a row of x, lanes l16 + 16 g split one of w.
        bool again = false;
#pragma unroll
        for (uint32_t t = 0; t < TASKS; ++t) again |= !in_three_pieces(most_x[t], 1, 2);
#pragma unroll
        for (int i = 0; i < TN; ++i) again |= !in_three_pieces(most_w[i], 16, 32);
        if (__syncthreads_or(again)) {
#pragma unroll
            for (int i = 0; i < TN; ++i)
#pragma unroll
                for (int j = 0; j < TM; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
            for (uint32_t step = first; step < last; ++step) {
                const uint32_t c = step * STEP + 8u * lg;
                const bool in = c < p.K;
                request_w(w0, step);
#pragma unroll
                for (int j = 0; j < TM; ++j) {
                    const uint32_t r = m0 + 16u * j + l16;
                    Frag<DT> x = frag_load<DT>((const T*)p.x + (size_t)(r < p.M ? r : p.M - 1u) * p.ldx + (in ? c : 0u));
                    if (!in) x = Frag<DT>{};
#pragma unroll
                    for (int i = 0; i < TN; ++i) {
                        if (!in) w0[i][0] = Frag<DT>{};
                        mma(w0[i][0], x, acc[i][j]);
                    }
                }
            }
        }
    }
#pragma unroll
    for (int j = 0; j < TM; ++j) {
        const uint32_t m = m0 + 16u * j + l16;
        if (m >= p.M) continue;
#pragma unroll
        for (int i = 0; i < TN; ++i) {
            const uint32_t n = n0 + wn + 16u * (uint32_t)i + 4u * lg;
            if (n >= p.N) continue;
            const f32x4 v = acc[i][j];
            if (p.ks > 1u) {
                float* dst = p.part + ((size_t)blockIdx.z * p.M + m) * p.N + n;
                if (p.wide) *(f32x4*)dst = v;
                else
#pragma unroll
                    for (uint32_t e = 0; e < 4u; ++e) if (n + e < p.N) dst[e] = v[e];
            } else if (p.wide) {
                if constexpr (DT == kFP32) *(f32x4*)((float*)p.out + (size_t)m * p.ldo + n) = v;
                else *(u32x2*)((uint16_t*)p.out + (size_t)m * p.ldo + n) = u32x2{pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3])};
            } else {
#pragma unroll
                for (uint32_t e = 0; e < 4u; ++e) if (n + e < p.N) Elem<DT>::store(p.out, (size_t)m * p.ldo + n + e, v[e]);
            }
        }
    }
}

// Sums of the ranges of K, in order: four neighbouring outputs a thread where WIDE.
template <int DT, bool WIDE>
__global__ __launch_bounds__(256) void row_gemm_sum_kernel(const RowGemm p) {
    const size_t count = (size_t)p.M * p.N, i = ((size_t)blockIdx.x * 256u + threadIdx.x) * (WIDE ? 4u : 1u);
    if (i >= count) return;
    const size_t m = i / p.N, n = i - m * p.N;
    if constexpr (WIDE) {
        f32x4 v = *(const f32x4*)(p.part + i);
        for (uint32_t k = 1; k < p.ks; ++k) v += *(const f32x4*)(p.part + k * count + i);
        if constexpr (DT == kFP32) *(f32x4*)((float*)p.out + m * p.ldo + n) = v;
        else *(u32x2*)((uint16_t*)p.out + m * p.ldo + n) = u32x2{pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3])};
    } else {
        float v = p.part[i];
        for (uint32_t k = 1; k < p.ks; ++k) v += p.part[k * count + i];
        Elem<DT>::store(p.out, m * p.ldo + n, v);
    }
}

// 16-token tiles of a workgroup, and ranges of K.
struct GemmPlan { uint32_t tm, ks; float us; };
static GemmPlan gemm_plan(int dt, uint32_t M, uint32_t N, uint32_t K) {
    const uint32_t step = dt == kFP32 ? 32u : 64u, steps = (K + step - 1u) / step, most = (steps + 3u) / 4u, cols = (N + kGemmBN - 1u) / kGemmBN;
    if (dt != kFP32) {
        // few tokens, whose steps are short: one or two tiles, and as many ranges as bring four workgroups to every compute unit
        const uint32_t tm = M <= 16u ? 1u : 2u, ks = 1024u / (cols * ((M + 16u * tm - 1u) / (16u * tm)));
        return {tm, ks < 1u ? 1u : (ks < most ? ks : most), 0.f};
    }
    // The least of steps x (0.9 us that a step takes from its requests to its products, and for every workgroup of a compute unit
    // its products and four tiles' worth of splitting the weight, 0.057 us a tile), and the sums of the ranges through memory.
    // Fewer than four tiles split the weight for too few products.
    GemmPlan best{4u, 1u, __builtin_inff()};
    for (uint32_t tm = 4u; tm <= 8u; ++tm)
        for (uint32_t ks = 1u; ks <= 32u && ks <= most; ++ks) {
            const uint32_t turns = ((M + 16u * tm - 1u) / (16u * tm) * cols * ks + 255u) / 256u;
            float t = (float)((steps + ks - 1u) / ks) * (0.9f * (float)((turns + 2u) / 3u) + 0.057f * (float)(turns * (tm + 4u)));
            if (ks > 1u) t += 4.f + (float)ks * (float)M * (float)N * 8.f / 5e6f;
            if (t < best.us) best = {tm, ks, t};
        }
    return best;
}

// Whether the fp16 units take a 32-bit product: where that is faster, by the two estimates, of which that of six products is short by
// 10-30 %.  Over 50 products on pieces, 160-800 x 1024-14336 x 512-7168, they take 0.51 to 1.00 of the time of six.  Pieces / six products, us a call:
// 777 x 8448 x 2048 99 / 196, 777 x 2048 x 2048 49 / 64, 256 x 8448 x 512 31 / 37, 160 x 8448 x 1024 38 / 38; left to six 160 x 2048 x 2048 30 / 23, 256
// x 2048 x 512 22 / 16.  Rows of 2^26 numbers and more: offsets of a wave's 64 rows have 32 bits there.
static bool takes_split(const GemmPlan& six, const SplitPlan& split, uint32_t ldw) { return split.us < 1.12f * six.us && ldw < (1u << 26); }

size_t row_gemm_workspace(int dt, uint32_t M, uint32_t N, uint32_t K) {
    const GemmPlan plan = gemm_plan(dt, M, N, K);
    const size_t need = plan.ks > 1u ? (size_t)plan.ks * M * N * sizeof(float) : 0;
    if (dt != kFP32) return need;
    const SplitPlan split = split_plan(M, N, K);
    const size_t other = takes_split(plan, split, 0u) ? split_workspace(split, M, N, K) : 0;
    return other > need ? other : need;                    // the row stride, which is not known here, decides between them
}

int row_gemm_pieces(int dt, uint32_t M, uint32_t N, uint32_t K, uint32_t ldw) {
    if (dt != kFP32) return 0;
    const SplitPlan split = split_plan(M, N, K);
    return takes_split(gemm_plan(dt, M, N, K), split, ldw) ? (int)split.ks : 0;
}

template <int DT>
static hipError_t row_sums_launch(const RowGemm& p, hipStream_t s) {
    const size_t count = (size_t)p.M * p.N / (p.wide ? 4u : 1u);
    const dim3 sums((uint32_t)((count + 255u) / 256u));
    if (p.wide) hipLaunchKernelGGL((row_gemm_sum_kernel<DT, true>), sums, dim3(256), 0, s, p);
    else hipLaunchKernelGGL((row_gemm_sum_kernel<DT, false>), sums, dim3(256), 0, s, p);
    return hipGetLastError();
}

template <int DT, int TM>
static hipError_t row_gemm_launch(const RowGemm& p, hipStream_t s) {
    using G = GemmShape<DT>;
    constexpr size_t lds = 2u * (size_t)G::blocks * G::pieces * 16u * TM * 64u;
    if (hipError_t e = allow_lds<row_gemm_kernel<DT, TM>>(lds); e != hipSuccess) return e;
    const dim3 grid((p.N + kGemmBN - 1u) / kGemmBN, (p.M + 16u * TM - 1u) / (16u * TM), p.ks);
    hipLaunchKernelGGL((row_gemm_kernel<DT, TM>), grid, dim3(256), lds, s, p);
    if (hipError_t e = hipGetLastError(); e != hipSuccess || p.ks == 1u) return e;
    return row_sums_launch<DT>(p, s);
}

static hipError_t row_gemm_fp32(uint32_t tm, const RowGemm& p, hipStream_t s) {
    switch (tm) {
        case 4u: return row_gemm_launch<kFP32, 4>(p, s);
        case 5u: return row_gemm_launch<kFP32, 5>(p, s);
        case 6u: return row_gemm_launch<kFP32, 6>(p, s);
        case 7u: return row_gemm_launch<kFP32, 7>(p, s);
        default: return row_gemm_launch<kFP32, 8>(p, s);
    }
}

hipError_t launch_row_gemm(int dt, const void* x, uint32_t ldx, const void* w, uint32_t ldw, void* out, uint32_t ldo, void* ws, uint32_t M,
                           uint32_t N, uint32_t K, hipStream_t s) {
    const GemmPlan plan = gemm_plan(dt, M, N, K);
    RowGemm p{x, w, out, (float*)ws, M, N, K, ldx, ldw, ldo, plan.ks, 0u, 0u};
    const uint32_t step = dt == kFP32 ? 32u : 64u;
    p.steps = ((K + step - 1u) / step + p.ks - 1u) / p.ks;
    p.wide = N % 4u == 0 && ldo % 4u == 0 && (((uintptr_t)out | (uintptr_t)ws) % 16u) == 0;
    if (dt == kFP32) {
        const SplitPlan split = split_plan(M, N, K);
        if (!takes_split(plan, split, ldw)) return row_gemm_fp32(plan.tm, p, s);
        p.ks = split.ks;
        p.part = split_sums(split, ws, M, K);
        const hipError_t e = launch_split_gemm(split, (const float*)x, ldx, (const float*)w, ldw, (float*)out, ldo, ws, M, N, K, p.wide != 0u, s);
        return e != hipSuccess || p.ks == 1u ? e : row_sums_launch<kFP32>(p, s);
    }
    return plan.tm == 1u ? row_gemm_launch<kBF16, 1>(p, s) : row_gemm_launch<kBF16, 2>(p, s);
}

}  // namespace decdec
