// Causal softmax attention over cached keys and values, with an optional valueless score (sink) in the denominator and an
// optional gate per head on the read-out.
//
// Many tokens: one tiled kernel for keys of a head's own, or of a head's own part and a part that all heads share (latent
// attention).  Grouped attention: normed, partly rotated queries and keys; the cache holds the keys by head and the values
// transposed, which is how the products read them; one token takes two launches (shares of the sequence, then their merge).
// Scores, weights and sums are fp32; on bf16 storage a weight enters the value product as the sum of two bf16 numbers.
#include "mixers.h"
#include "mma.h"
#include "grouped_merge.h"

namespace decdec {

// ---- many tokens: which instance of the tiled kernel --------------------------------------------------------
template <int DT, int MT, int NK>
static hipError_t tile_nv(const TileAttention& p, uint32_t start, uint32_t rows, hipStream_t s) {
    if (p.vdim <= 64u) return tile_launch<DT, MT, NK, 4>(p, start, rows, s);
    if (p.vdim <= 128u) return tile_launch<DT, MT, NK, 8>(p, start, rows, s);
    return tile_launch<DT, 1, NK, 16>(p, start, rows, s);
}

template <int DT, int MT>
static hipError_t tile_dt(const TileAttention& p, uint32_t start, uint32_t rows, hipStream_t s) {
    const uint32_t Dq = p.dim + p.rot;
    if (((p.dim | p.rot) % 8u | (p.k_row | p.k_head | p.shared_row | (uintptr_t)p.shared / Elem<DT>::bytes) % 8u) != 0)
        return tile_launch<DT, 1, 10, 16, false>(p, start, rows, s);
    if (Dq <= 128u) return tile_nv<DT, MT, 4>(p, start, rows, s);
    if (Dq <= 192u) return tile_nv<DT, MT, 6>(p, start, rows, s);
    return tile_nv<DT, 1, 10>(p, start, rows, s);
}

hipError_t launch_tile_attention(int dt, const TileAttention& p, uint32_t start, uint32_t rows, hipStream_t s) {
    if (p.dim + p.rot > 320u || p.vdim > 256u) return hipErrorInvalidValue;
    return dt == kBF16 ? tile_dt<kBF16, 2>(p, start, rows, s) : tile_dt<kFP32, 1>(p, start, rows, s);
}


// ---- grouped attention: queries, keys and values of new tokens ----------------------------------------------
// One head of one token by a wave: RMS norm over dim (weight may be null), then the pairs (2i, 2i + 1) of the first `rot`
// elements turned.  A lane takes elements 2 lane + 128 j and the next; dim is at most 320.
constexpr int kPairs = 3;

struct HeadRow { float x[kPairs][2], w[kPairs][2], c[kPairs], s[kPairs]; };
template <int DT>
__device__ __forceinline__ HeadRow head_fetch(const void* proj, size_t at, const void* weight, const decdec_grouped& p, size_t trow) {
    using E = Elem<DT>;
    const uint32_t lane = threadIdx.x & 63u, D = p.dim;
    HeadRow f;
#pragma unroll
    for (int j = 0; j < kPairs; ++j) {
        const uint32_t i0 = 2u * lane + 128u * (uint32_t)j;
        const bool turn = i0 < p.rot;
#pragma unroll
        for (uint32_t e = 0; e < 2u; ++e) {
            const bool in = i0 + e < D;
            f.x[j][e] = in ? E::load(proj, at + i0 + e) : 0.f;
            f.w[j][e] = (weight != nullptr && in) ? E::load(weight, i0 + e) : 1.f;
        }
        f.c[j] = turn ? p.cos_table[trow + i0 / 2u] : 1.f;
        f.s[j] = turn ? p.sin_table[trow + i0 / 2u] : 0.f;
    }
    return f;
}
__device__ __forceinline__ void norm_rotate(const HeadRow& f, bool norm, const decdec_grouped& p, float (&x)[kPairs][2]) {
    float r = 1.f;
    if (norm) {
        float ss = 0.f;
#pragma unroll
        for (int j = 0; j < kPairs; ++j) ss += f.x[j][0] * f.x[j][0] + f.x[j][1] * f.x[j][1];
        r = 1.f / sqrtf(wave_sum(ss) / (float)p.dim + p.eps);
    }
#pragma unroll
    for (int j = 0; j < kPairs; ++j) {
        const float u = f.x[j][0] * r * f.w[j][0], v = f.x[j][1] * r * f.w[j][1];
        x[j][0] = u * f.c[j] - v * f.s[j];
        x[j][1] = v * f.c[j] + u * f.s[j];
    }
}

template <int DT>
__device__ __forceinline__ void store_pairs(void* dst, size_t at, uint32_t D, const float (&x)[kPairs][2]) {
    const uint32_t lane = threadIdx.x & 63u;
#pragma unroll
    for (int j = 0; j < kPairs; ++j) {
        const uint32_t i = 2u * lane + 128u * (uint32_t)j;
        if (i + 1u < D && (D & 1u) == 0u) {
            if constexpr (DT == kBF16) *(uint32_t*)((uint16_t*)dst + at + i) = pack_bf16(x[j][0], x[j][1]);
            else *(u32x2*)((float*)dst + at + i) = u32x2{__float_as_uint(x[j][0]), __float_as_uint(x[j][1])};
        } else {
            if (i < D) Elem<DT>::store(dst, at + i, x[j][0]);
            if (i + 1u < D) Elem<DT>::store(dst, at + i + 1u, x[j][1]);
        }
    }
}

// Queries to q_out [rows][heads][dim], keys to the cache: a wave per head of a token.
template <int DT>
__global__ __launch_bounds__(256) void grouped_append_kernel(const decdec_grouped p, void* __restrict__ q_out, const uint32_t rows) {
    const uint32_t at = blockIdx.x * 4u + (threadIdx.x >> 6), all = p.heads + p.kv_heads, t = at / all, j = at - t * all;
    if (t >= rows) return;
    const long long pos = *p.pos + (long long)t;
    if (pos < 0 || pos >= (long long)p.max_seq) return;
    const bool isq = j < p.heads;
    const uint32_t h = isq ? j : j - p.heads;
    const void* weight = isq ? p.q_norm : p.k_norm;
    float x[kPairs][2];
    norm_rotate(head_fetch<DT>(p.proj, (size_t)t * p.ld + (isq ? p.off_q : p.off_k) + h * p.dim, weight, p, (size_t)pos * (p.rot / 2u)),
                weight != nullptr, p, x);
    if (isq) store_pairs<DT>(q_out, ((size_t)t * p.heads + h) * p.dim, p.dim, x);
    else store_pairs<DT>(p.keys, ((size_t)h * p.max_seq + (size_t)pos) * p.dim, p.dim, x);
}

// The same for dim a multiple of 8 and rot of 8: gl lanes share a head, eight neighbouring elements each.
template <int DT>
__global__ __launch_bounds__(256) void grouped_append_vec_kernel(const decdec_grouped p, void* __restrict__ q_out, const uint32_t rows,
                                                                 const uint32_t gl) {
    using T = typename LaneOf<DT>::t;
    const uint32_t all = p.heads + p.kv_heads, D = p.dim, sub = threadIdx.x % gl, c = 8u * sub;
    const uint32_t at = blockIdx.x * (256u / gl) + threadIdx.x / gl, t = at / all, j = at - t * all;
    const long long pos = *p.pos + (long long)t;
    const bool ok = t < rows && pos >= 0 && pos < (long long)p.max_seq, live = ok && c < D, isq = j < p.heads;
    const uint32_t h = isq ? j : j - p.heads;
    const void* weight = isq ? p.q_norm : p.k_norm;
    const size_t trow = (size_t)(ok ? pos : 0) * (p.rot / 2u);
    float x[8], w[8], cs[4], sn[4], ss = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) { x[e] = 0.f; w[e] = 1.f; }
    if (live) {
        frag_values(frag_load((const T*)p.proj + (size_t)t * p.ld + (isq ? p.off_q : p.off_k) + h * D + c), x);
        if (weight != nullptr) frag_values(frag_load((const T*)weight + c), w);
    }
    const bool turn = live && c < p.rot;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        cs[e] = turn ? p.cos_table[trow + c / 2u + e] : 1.f;
        sn[e] = turn ? p.sin_table[trow + c / 2u + e] : 0.f;
    }
    float r = 1.f;
    if (weight != nullptr) {
#pragma unroll
        for (int e = 0; e < 8; ++e) ss += x[e] * x[e];
    }
    for (uint32_t off = 1; off < gl; off <<= 1) ss += __shfl_xor(ss, (int)off, 64);
    if (weight != nullptr) r = 1.f / sqrtf(ss / (float)D + p.eps);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const float u = x[2 * e] * r * w[2 * e], v = x[2 * e + 1] * r * w[2 * e + 1];
        x[2 * e] = u * cs[e] - v * sn[e];
        x[2 * e + 1] = v * cs[e] + u * sn[e];
    }
    if (!live) return;
    T* dst = isq ? (T*)q_out + ((size_t)t * p.heads + h) * D + c : (T*)p.keys + ((size_t)h * p.max_seq + (size_t)pos) * D + c;
    store8(dst, frag_of(x, Frag<DT>{}));
}

// Values, transposed, to the cache: grid (tokens / 64, channels / 64).
template <int DT>
__global__ __launch_bounds__(256) void grouped_values_kernel(const decdec_grouped p, const uint32_t rows) {
    using T = typename LaneOf<DT>::t;
    __shared__ T tile[64][65];
    const uint32_t t0 = blockIdx.x * 64u, c0 = blockIdx.y * 64u, chans = p.kv_heads * p.vdim, a = threadIdx.x & 63u, b = threadIdx.x >> 6;
    const long long pos = *p.pos + (long long)(t0 + a);
    for (uint32_t i = b; i < 64u; i += 4u)
        if (t0 + i < rows && c0 + a < chans) tile[i][a] = ((const T*)p.proj)[(size_t)(t0 + i) * p.ld + p.off_v + c0 + a];
    __syncthreads();
    if (t0 + a >= rows || pos < 0 || pos >= (long long)p.max_seq) return;
    for (uint32_t i = b; i < 64u && c0 + i < chans; i += 4u) ((T*)p.values)[(size_t)(c0 + i) * p.max_seq + (size_t)pos] = tile[a][i];
}

template <int DT>
static hipError_t grouped_append_dt(const decdec_grouped& p, void* q_out, uint32_t rows, hipStream_t s) {
    const uint32_t all = rows * (p.heads + p.kv_heads);
    uint32_t gl = 1;
    while (8u * gl < p.dim) gl *= 2;                        // at most 64: dim is at most 320
    const bool vec = (p.dim | p.rot | p.ld | p.off_q | p.off_k) % 8u == 0 &&
                     ((uintptr_t)p.proj | (uintptr_t)p.q_norm | (uintptr_t)p.k_norm) % 16u == 0;
    if (vec) hipLaunchKernelGGL((grouped_append_vec_kernel<DT>), dim3((all + 256u / gl - 1u) / (256u / gl)), dim3(256), 0, s, p, q_out, rows, gl);
    else hipLaunchKernelGGL((grouped_append_kernel<DT>), dim3((all + 3u) / 4u), dim3(256), 0, s, p, q_out, rows);
    hipLaunchKernelGGL((grouped_values_kernel<DT>), dim3((rows + 63u) / 64u, (p.kv_heads * p.vdim + 63u) / 64u), dim3(256), 0, s, p, rows);
    return hipGetLastError();
}

hipError_t launch_grouped_append(int dt, const decdec_grouped& p, void* q_out, uint32_t rows, hipStream_t s) {
    return dt == kBF16 ? grouped_append_dt<kBF16>(p, q_out, rows, s) : grouped_append_dt<kFP32>(p, q_out, rows, s);
}

hipError_t launch_grouped_attention(int dt, const decdec_grouped& p, const void* q, void* out, uint32_t start, uint32_t rows,
                                    hipStream_t s) {
    TileAttention a{};
    a.q = q; a.k = p.keys; a.vt = p.values; a.out = out;
    a.k_head = (size_t)p.max_seq * p.dim; a.k_row = p.dim;
    a.vt_ld = p.max_seq; a.out_ld = p.out_ld;
    a.heads = p.heads; a.share = p.heads / p.kv_heads; a.dim = p.dim; a.vdim = p.vdim;
    a.scale = p.scale; a.sink_score = p.sink; a.out_scale = p.out_scale;
    if (p.gated) { a.gate = (const char*)p.proj + (size_t)p.off_g * (dt == kBF16 ? 2u : 4u); a.gate_ld = p.ld; }
    return launch_tile_attention(dt, a, start, rows, s);
}

// ---- grouped attention, one token -----------------------------------------------------------------------------
// A pass is 128 keys: 256 left two thirds of the compute units without a workgroup at a few thousand keys, and one workgroup a unit at
// most, since more of them leave the merge more.  us a step of the whole decoder, four layers of 2048 of which two attend with 8 key heads
// of 128, bf16, with passes of 256 keys and 512 workgroups, of 128 and 512, 1024 and 256: 300 keys 198.1, 193.7, 193.5, 193.6; 1500
// 200.0, 197.4, 197.9, 197.9; 4000 207.0, 207.7, 207.1, 204.5; 15000 230.3, 217.4, 230.2, 218.2.  The step alone, 512 workgroups (bf16 and heads up
// to 128: passes of 256) / 256 of 128 keys, 300, 4000, 8000 and 16000 keys: 8 key heads of 128 bf16 17.6 / 13.7, 18.2 / 15.1, 18.9 / 17.3, 31.5 / 23.9,
// fp32 16.4 / 15.5, 17.5 / 16.6, 29.2 / 23.4, 39.8 / 32.7; 8 of 256 bf16 23.2 / 22.9, 25.6 / 24.9, 43.7 / 28.8, 52.8 / 41.0, fp32 26.8 / 26.1, 29.1 / 28.8,
// 51.0 / 43.2, 77.3 / 67.9; no number of heads from 2 to 32 and no length is slower.
static bool grouped_small(const decdec_grouped& p) { return p.dim <= 128u && p.vdim <= 128u; }
static uint32_t grouped_max_splits(const decdec_grouped& p) {
    const uint32_t groups = p.kv_heads * ((p.heads / p.kv_heads + 15u) / 16u);
    const uint32_t want = 256u / groups, tiles = (p.max_seq + kGroupedUnit - 1u) / kGroupedUnit;
    const uint32_t n = want < 8u ? 8u : (want > kGroupedSplits ? kGroupedSplits : want);
    return n < tiles ? n : tiles;
}

// grid (splits, kv_heads, heads that share a key / 16), four waves, 16 KB keys a wave and pass.  Scores transposed (keys x
// heads): a wave's keys and values come from memory straight into the operands of its products.  Wave 0 of split 0 starts
// from the new token (which it also appends), every other wave from nothing; the waves are merged through LDS.
template <int DT, int NK, int NV>
__global__ __launch_bounds__(256, 1) void grouped_step_kernel(const decdec_grouped p, float* __restrict__ parts, const uint32_t max_splits) {
    using T = typename LaneOf<DT>::t;
    using E = Elem<DT>;
    constexpr uint32_t PAD = DT == kFP32 ? 4u : 8u, QL = 32u * NK + PAD, OL = 16u * NV + 4u, UNIT = kGroupedUnit;
    constexpr int KB = UNIT / 64;                          // 16-key blocks of a wave
    extern __shared__ __align__(16) float ol[];             // [4][16][OL]
    __shared__ __align__(16) T Ql[16][QL];
    __shared__ T knew[32 * NK], vnew[256];
    __shared__ float mxs[4][16], sums[4][16], snew[16];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6, l16 = lane & 15u, lg = lane >> 4;
    const uint32_t kvh = blockIdx.y, share = p.heads / p.kv_heads, g0 = blockIdx.z * 16u, D = p.dim, V = p.vdim;
    const uint32_t h0 = kvh * share + g0, nh = share - g0 < 16u ? share - g0 : 16u;
    const long long pos = *p.pos;
    if (pos < 0 || pos >= (long long)p.max_seq) return;
    const GroupedSplit sp = grouped_split((uint32_t)pos, max_splits);
    if (blockIdx.x >= sp.splits) return;
    const uint32_t lo = blockIdx.x * sp.span, hi = lo + sp.span < (uint32_t)pos ? lo + sp.span : (uint32_t)pos;
    const bool vec = D % 8u == 0, first = blockIdx.x == 0u;
    const T* kb = (const T*)p.keys + (size_t)kvh * p.max_seq * D;
    const T* vb = (const T*)p.values + (size_t)kvh * V * p.max_seq;
    Frag<DT> kf[KB][NK], vf[NV][KB / 2];
    // keys past the last repeat it and value columns past it are finite: neither is weighted
    auto request = [&](uint32_t k0) {
#pragma unroll
        for (int b = 0; b < KB; ++b) {
            const uint32_t key = k0 + 16u * (uint32_t)b + l16 < hi ? k0 + 16u * (uint32_t)b + l16 : hi - 1u;
            const T* row = kb + (size_t)key * D;
#pragma unroll
            for (int s = 0; s < NK; ++s) {
                const uint32_t c = 32u * (uint32_t)s + 8u * lg;
                if (vec) {
                    kf[b][s] = frag_load(row + (c < D ? c : 0u));
                    if (c >= D) kf[b][s] = Frag<DT>{};
                } else {
                    kf[b][s] = load8<DT>(row + c, (int)D - (int)c, false);
                }
            }
        }
#pragma unroll
        for (int n = 0; n < NV; ++n) {
            const uint32_t d = 16u * (uint32_t)n + l16;
            const T* row = vb + (size_t)(d < V ? d : 0u) * p.max_seq + k0 + 4u * lg;
#pragma unroll
            for (int t = 0; t < KB / 2; ++t) {
                if constexpr (DT == kFP32) {
                    const f32x4 x = *(const f32x4*)(row + 32 * t), y = *(const f32x4*)(row + 32 * t + 16);
#pragma unroll
                    for (int e = 0; e < 4; ++e) { vf[n][t].v[e] = x[e]; vf[n][t].v[4 + e] = y[e]; }
                } else {
                    const u32x2 x = *(const u32x2*)(row + 32 * t), y = *(const u32x2*)(row + 32 * t + 16);
                    vf[n][t].v = u32x4{x[0], x[1], y[0], y[1]};
                }
            }
        }
    };
    // the wave's first query head and the new key ahead of the cache: memory answers in order
    const size_t trow = (size_t)pos * (p.rot / 2u);
    const HeadRow q0 = head_fetch<DT>(p.proj, p.off_q + (size_t)(h0 + (wave < nh ? wave : 0u)) * D, p.q_norm, p, trow);
    HeadRow kn{};
    T vn = (T)0;
    if (first) {
        if (wave == 3u) kn = head_fetch<DT>(p.proj, p.off_k + (size_t)kvh * D, p.k_norm, p, trow);
        if (tid < V) vn = ((const T*)p.proj)[p.off_v + kvh * V + tid];
    }
    uint32_t k0 = lo + wave * 16u * KB;
    if (k0 < hi) request(k0);
    for (uint32_t i = tid; i < 16u * 32u * NK; i += 256u) {                // zeros past dim and past the last head
        const uint32_t r = i / (32u * NK), c = i % (32u * NK);
        if (r >= nh || c >= D) Ql[r][c] = (T)0;
    }
    for (uint32_t j = wave; j < nh; j += 4u) {
        float x[kPairs][2];
        norm_rotate(j == wave ? q0 : head_fetch<DT>(p.proj, p.off_q + (size_t)(h0 + j) * D, p.q_norm, p, trow), p.q_norm != nullptr, p, x);
        store_pairs<DT>(&Ql[j][0], 0, D, x);
    }
    if (first && tid < V) {
        vnew[tid] = vn;
        if (blockIdx.z == 0u) ((T*)p.values)[(size_t)(kvh * V + tid) * p.max_seq + (size_t)pos] = vn;
    }
    if (first && wave == 3u) {
        float x[kPairs][2];
        norm_rotate(kn, p.k_norm != nullptr, p, x);
        store_pairs<DT>(knew, 0, D, x);
        if (blockIdx.z == 0u) store_pairs<DT>(p.keys, ((size_t)kvh * p.max_seq + (size_t)pos) * D, D, x);
    }
    __syncthreads();
    const float scale2 = p.scale * kLog2e;
    float mx = -__builtin_inff(), sum = 0.f;
    f32x4 o[NV];
#pragma unroll
    for (int n = 0; n < NV; ++n) o[n] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (first) {
        const uint32_t r = tid >> 4, c = tid & 15u;
        float x = 0.f;
        for (uint32_t i = c; i < D; i += 16u) x = __builtin_fmaf(E::load(&Ql[r][0], i), E::load(knew, i), x);
#pragma unroll
        for (int off = 1; off < 16; off <<= 1) x += __shfl_xor(x, off, 64);
        if (c == 0u) snew[r] = x * scale2;
        __syncthreads();
        if (wave == 0u) {
            mx = snew[l16];
            sum = lg == 0u ? 1.f : 0.f;                                    // lane groups hold partial sums
#pragma unroll
            for (int n = 0; n < NV; ++n)
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const uint32_t d = 16u * (uint32_t)n + 4u * lg + (uint32_t)v;
                    o[n][v] = d < V ? E::load(vnew, d) : 0.f;
                }
        }
    }
    Frag<DT> qf[NK];
#pragma unroll
    for (int s = 0; s < NK; ++s) qf[s] = frag_load(&Ql[l16][32u * s + 8u * lg]);
    for (; k0 < hi; k0 += UNIT) {
        f32x4 sc[KB];
#pragma unroll
        for (int b = 0; b < KB; ++b) {
            sc[b] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int s = 0; s < NK; ++s) mma(kf[b][s], qf[s], sc[b]);
        }
        float best = mx;
#pragma unroll
        for (int b = 0; b < KB; ++b)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const float x = k0 + 16u * (uint32_t)b + 4u * lg + (uint32_t)v < hi ? sc[b][v] * scale2 : -__builtin_inff();
                sc[b][v] = x;
                best = fmaxf(best, x);
            }
        best = fmaxf(best, __shfl_xor(best, 16, 64));
        best = fmaxf(best, __shfl_xor(best, 32, 64));                      // finite: the tile has a key
        const float corr = __builtin_amdgcn_exp2f(mx - best);
        mx = best;
        sum *= corr;
#pragma unroll
        for (int n = 0; n < NV; ++n) o[n] *= corr;
        Frag<DT> whi[KB / 2], wlo[KB / 2];
#pragma unroll
        for (int t = 0; t < KB / 2; ++t) {
            float w[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                w[e] = __builtin_amdgcn_exp2f(sc[2 * t + (e >> 2)][e & 3] - best);
                sum += w[e];
            }
            frag_split(w, whi[t], wlo[t]);
        }
#pragma unroll
        for (int n = 0; n < NV; ++n)
#pragma unroll
            for (int t = 0; t < KB / 2; ++t) {
                mma(vf[n][t], whi[t], o[n]);
                if constexpr (DT != kFP32) mma(vf[n][t], wlo[t], o[n]);
            }
        if (k0 + UNIT < hi) request(k0 + UNIT);
    }
    sum += __shfl_xor(sum, 16, 64);
    sum += __shfl_xor(sum, 32, 64);
    if (lg == 0u) { mxs[wave][l16] = mx; sums[wave][l16] = sum; }
#pragma unroll
    for (int n = 0; n < NV; ++n) *(f32x4*)&ol[(wave * 16u + l16) * OL + 16u * (uint32_t)n + 4u * lg] = o[n];
    __syncthreads();
    // partial result of a head: [vdim] sums, maximum, sum of weights; wave 0 has a key or the new token: M is finite
    for (uint32_t i = tid; i < nh * V; i += 256u) {
        const uint32_t h = i / V, d = i - h * V;
        const float M = fmaxf(fmaxf(mxs[0][h], mxs[1][h]), fmaxf(mxs[2][h], mxs[3][h]));
        float acc = 0.f, l = 0.f;
#pragma unroll
        for (uint32_t w = 0; w < 4u; ++w) {
            const float f = __builtin_amdgcn_exp2f(mxs[w][h] - M);
            acc = __builtin_fmaf(f, ol[(w * 16u + h) * OL + d], acc);
            l = __builtin_fmaf(f, sums[w][h], l);
        }
        float* dst = parts + ((size_t)blockIdx.x * p.heads + h0 + h) * (V + 2u);
        dst[d] = acc;
        if (d == 0u) { dst[V] = M; dst[V + 1u] = l; }
    }
}

// Merge of the splits, sink and gate: a workgroup per head.
template <int DT>
__global__ __launch_bounds__(1024) void grouped_merge_kernel(const GroupedMerge m) {
    __shared__ float share[1024], ws[kGroupedSplits];
    grouped_merge<DT>(m, blockIdx.x, share, ws);
}

size_t grouped_step_workspace(const decdec_grouped& p) { return (size_t)kGroupedSplits * p.heads * (p.vdim + 2u) * sizeof(float); }

template <int DT, int NK, int NV>
static hipError_t grouped_step_launch(const decdec_grouped& p, float* parts, dim3 grid, uint32_t splits, hipStream_t s) {
    constexpr size_t lds = 4u * 16u * (16u * NV + 4u) * sizeof(float);
    if (hipError_t e = allow_lds<grouped_step_kernel<DT, NK, NV>>(lds); e != hipSuccess) return e;
    hipLaunchKernelGGL((grouped_step_kernel<DT, NK, NV>), grid, dim3(256), lds, s, p, parts, splits);
    return hipGetLastError();
}

template <int DT>
static hipError_t grouped_step_dt(const decdec_grouped& p, float* parts, hipStream_t s) {
    const uint32_t splits = grouped_max_splits(p);
    const dim3 grid(splits, p.kv_heads, (p.heads / p.kv_heads + 15u) / 16u);
    return grouped_small(p) ? grouped_step_launch<DT, 4, 8>(p, parts, grid, splits, s) : grouped_step_launch<DT, 10, 16>(p, parts, grid, splits, s);
}

GroupedMerge grouped_merge_of(const decdec_grouped& p, void* out, void* ws) {
    return GroupedMerge{(const float*)ws, out, p.pos, p.gated ? p.proj : nullptr, p.off_g, p.heads, p.vdim, p.max_seq, grouped_max_splits(p), p.sink, p.out_scale};
}

hipError_t launch_grouped_shares(int dt, const decdec_grouped& p, void* ws, hipStream_t s) {
    return dt == kBF16 ? grouped_step_dt<kBF16>(p, (float*)ws, s) : grouped_step_dt<kFP32>(p, (float*)ws, s);
}

hipError_t launch_grouped_step(int dt, const decdec_grouped& p, void* out, void* ws, hipStream_t s) {
    if (hipError_t e = launch_grouped_shares(dt, p, ws, s); e != hipSuccess) return e;
    const GroupedMerge m = grouped_merge_of(p, out, ws);
    if (dt == kBF16) hipLaunchKernelGGL((grouped_merge_kernel<kBF16>), dim3(p.heads), dim3(1024), 0, s, m);
    else hipLaunchKernelGGL((grouped_merge_kernel<kFP32>), dim3(p.heads), dim3(1024), 0, s, m);
    return hipGetLastError();
}

}  // namespace decdec
