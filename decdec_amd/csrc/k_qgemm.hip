// Packed products in tiles of 128 tokens (qgemm_tile.h): how one is dealt to workgroups, the sums of split tiles, and its launch.
#include "qgemm_tile.h"

namespace decdec {

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

template <int DT>
static hipError_t launch_qgemm_sum(const QgemmParams& p, const QgemmPlan& g, hipStream_t s) {
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
    const hipError_t e = (fmt == kAnyprec ? launch_qgemm_anyprec : fmt == kLutgemm ? launch_qgemm_lutgemm : launch_qgemm_sqllm)(dt, bits, flag, p, g, s);
    if (e != hipSuccess || g.tiles == g.whole) return e;
    return dt == kFP16 ? launch_qgemm_sum<kFP16>(p, g, s) : launch_qgemm_sum<kBF16>(p, g, s);
}

}  // namespace decdec
