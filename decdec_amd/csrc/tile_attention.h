// Tiled causal softmax attention of many tokens over cached keys and values.
#pragma once
#include "common.h"
#include "mma.h"

namespace decdec {

// Operands of the tiled attention kernel, strides in elements.  A key row is `dim` elements of the (shared) head's own and
// `rot` elements all heads share.
struct TileAttention {
    const void* q;              // [rows][heads][dim + rot]
    const void* k;              // kv head k_head apart, key k_row apart
    const void* shared;         // key shared_row apart, or null (rot = 0)
    const void* vt;             // [kv heads * vdim][vt_ld], or with values in rows: kv head v_head apart, key k_row apart
    const void* sink;           // E [heads], or null: sink_score for all heads (minus infinity: no sink)
    const void* gate;           // rows gate_ld apart, one number per head, through a sigmoid; or null
    void* out;                  // rows out_ld apart, [heads][vdim]
    const long long* positions; // of the queries, or null: start + row
    size_t k_head, k_row, v_head;
    uint32_t shared_row, vt_ld, gate_ld, out_ld, heads, share, dim, rot, vdim;
    float scale, sink_score, out_scale;
};

// Workgroups of four waves with 16 MT queries each, one per query block and head; neighbouring heads go to one die, so that
// the tiles of a head's keys and values (and of heads that share them) stay in one L2.  The transposed scores (keys x
// queries) leave a query in one lane column: its running maximum and sum are lane values, its weights are at once the right
// operand of the value product (out^T = V^T P^T), and nothing passes through LDS but the key and value tiles.  The
// contraction of that product visits keys 4 (lane / 16) + e of one 16-key tile, then of the next, in both operands.  The
// next tile is requested into registers while the present one is worked on.  Scores are kept in units of log 2.
//
// What bounds it: matrix products and vector instructions (softmax, and splitting the weights in two) are busy about 46 % of
// the cycles each, and overlap only where the order of instructions lets them.  So 16-bit products are asked for in an order:
// operands three reads ahead, the weights of a tile's second half between the products of its first, and score products at
// a higher priority than what the other wave of the SIMD does meanwhile; bounds and masks are uniform branches, and nothing
// looks at a loaded key before it is put into LDS.  32 heads, keys of 128 + 64, values of 128, 4096 tokens behind 4096: 990 us
// with the compiler's order, padded rows and masks everywhere, now 804 (641 TFLOP/s, 900 with the trailing halves counted);
// 4096 tokens alone 452 -> 342.  Two tiles in LDS and one barrier a tile instead of two: 828.
//
// ROWS (16-bit, VEC): the values lie in rows like the keys, and the queries' positions are read from memory (in any order; the
// keys number vt_ld).  A thread then requests eight elements of four neighbouring keys' values and turns them around on the
// way into LDS, so that both layouts look the same to the products.  These are the plain decoder's prompts, whose weights torch
// operations multiplied in 32 bits: bf16 weights enter as three numbers, which are exactly the 32-bit weight (1999 tokens, 32 query
// and 8 key heads of 128: 116 us with two numbers, 16 bits of it; 120 with three, cut off and with all vector instructions asked for
// ahead of the products; 135 with three rounded ones between the products, as two are), and fp16 ones as two on a
// scale of 2 ^ 15.  Share of outputs that are not the rounded 64-bit result, 1999 tokens: bf16 3e-4 (two numbers 23e-4, torch
// operations 6e-4), fp16 21e-4 (torch operations 34e-4); 3000 keys of a weight of 2 ^ -22 each beside one of 1, fp16, error over norm 2.18e-4, on a
// scale of 1 10.8e-4.
constexpr uint32_t kKeys = 64;

// Where a tile in LDS holds column c of row r (16-bit): rows are an odd number of 16-byte pieces long, and rows 4 .. 11 of every
// 16 have neighbouring pieces swapped, so that each of the quarters in which a 16-byte read by rows lane % 16 and pieces
// lane / 16 is served (its first one is lanes 0 .. 3, 12 .. 15 and 20 .. 27) meets every bank once.  Values lie in the order
// in which the products visit the keys, four of one 16-key tile beside four of the next: one read per operand.
template <int DT>
__device__ __forceinline__ uint32_t tile_slot(uint32_t r, uint32_t c) {
    return DT == kFP32 ? c : c ^ ((((r >> 2) ^ (r >> 3)) & 1u) << 3);
}
template <int DT>
__device__ __forceinline__ uint32_t value_slot(uint32_t r, uint32_t key) {
    return DT == kFP32 ? key : tile_slot<DT>(r, (key & ~31u) | ((key & 12u) << 1) | ((key & 16u) >> 2) | (key & 3u));
}

template <int DT, int MT, int NK, int NV, bool VEC, bool ROWS = false>
__global__ __launch_bounds__(256, DT == kFP32 ? 1 : 2) void tile_attention_kernel(const TileAttention p, const uint32_t start,
                                                                             const uint32_t rows, const uint32_t blocks) {
    using T = typename LaneOf<DT>::t;
    using E = Elem<DT>;
    constexpr uint32_t PAD = DT == kFP32 ? 4u : 8u, KL = 32u * NK + PAD, VL = kKeys + PAD;
    constexpr int P = DT == kFP32 ? 1 : (ROWS && DT == kBF16 ? 3 : 2);     // parts of a weight
    extern __shared__ __align__(16) unsigned char smem[];
    T* Kl = (T*)smem;                       // [kKeys][KL]
    T* Vl = Kl + kKeys * KL;                // [16 NV][VL]
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = __builtin_amdgcn_readfirstlane(tid >> 6), l16 = lane & 15u, lg = lane >> 4;
    const uint32_t die_heads = (p.heads + 7u) / 8u, count = die_heads * blocks;
    uint32_t turn = blockIdx.x >> 3;
    if (count <= 64u && turn >= 32u) turn = count + 31u - turn;            // the second ones of a die's 32 units
    const uint32_t h = (blockIdx.x & 7u) * die_heads + turn % die_heads;
    if (h >= p.heads) return;
    const uint32_t kvh = h / p.share;
    const uint32_t q0 = (blocks - 1u - turn / die_heads) * (64u * MT);     // longest rows first
    const uint32_t Dq = p.dim + p.rot, D = p.dim, V = p.vdim, keys_total = ROWS ? p.vt_ld : start + rows;
    const T* q = (const T*)p.q;
    Frag<DT> qf[MT][NK];
    uint32_t qpos[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) {
        const uint32_t r = q0 + 16u * (MT * wave + (uint32_t)m) + l16, rc = r < rows ? r : rows - 1u;
        qpos[m] = ROWS ? (uint32_t)p.positions[rc] : start + rc;
        if (ROWS && qpos[m] >= keys_total) qpos[m] = keys_total - 1u;
#pragma unroll
        for (int s = 0; s < NK; ++s)
            qf[m][s] = load8<DT>(q + ((size_t)rc * p.heads + h) * Dq + 32u * s + 8u * lg, (int)Dq - (int)(32u * s + 8u * lg), VEC);
    }
    // a negative scale's sign goes to the queries; at least the smallest normal number, so that a masked score stays minus infinity
    const float scale2 = fmaxf(fabsf(p.scale * kLog2e), 1.1754944e-38f);
    if (p.scale < 0.f) {
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int s = 0; s < NK; ++s) negate(qf[m][s]);
    }
    const float sink = (p.sink != nullptr ? E::load(p.sink, h) : p.sink_score) * kLog2e;      // minus infinity: none
    // Weights are taken relative to this, which cancels in the division: 2 ^ 15 for the largest in fp16, whose trailing parts would
    // end at 2 ^ -24 of it otherwise; not where scores are so large that their rounding moves the exponent.
    auto base = [](float m) { return DT == kFP16 && fabsf(m) < 4194304.f ? m - 15.f : m; };
    float mx[MT], from[MT], sum[MT];
    f32x4 o[MT][NV];
#pragma unroll
    for (int m = 0; m < MT; ++m) {
        mx[m] = fmaxf(sink, -3.4028235e38f);                           // finite also where no score is: minus infinity has no weight
        from[m] = base(mx[m]);
        sum[m] = (sink > -__builtin_inff() && lg == 0u) ? __builtin_amdgcn_exp2f(sink - from[m]) : 0.f;   // lane groups hold partial sums
#pragma unroll
        for (int n = 0; n < NV; ++n) o[m][n] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    const uint32_t last = q0 + 64u * MT < rows ? q0 + 64u * MT : rows;     // one past the block's last query
    uint32_t kend = start + last, wave_first = start + q0 + 16u * MT * wave, wave_last = wave_first + 16u * MT - 1u;
    if constexpr (ROWS) {
        __shared__ uint32_t furthest[4];
        wave_first = wave_last = qpos[0];
#pragma unroll
        for (int m = 1; m < MT; ++m) { wave_first = wave_first < qpos[m] ? wave_first : qpos[m]; wave_last = wave_last > qpos[m] ? wave_last : qpos[m]; }
#pragma unroll
        for (int off = 1; off < 16; off <<= 1) {
            const uint32_t a = __shfl_xor(wave_first, off, 64), b = __shfl_xor(wave_last, off, 64);
            wave_first = wave_first < a ? wave_first : a;
            wave_last = wave_last > b ? wave_last : b;
        }
        wave_first = __builtin_amdgcn_readfirstlane(wave_first);
        wave_last = __builtin_amdgcn_readfirstlane(wave_last);
        if (lane == 0u) furthest[wave] = wave_last;
        __syncthreads();
        kend = 0u;
#pragma unroll
        for (int w = 0; w < 4; ++w) kend = kend > furthest[w] ? kend : furthest[w];
        kend = __builtin_amdgcn_readfirstlane(kend) + 1u;
    }
    const size_t kld = p.k_row, cld = p.shared_row, vt_ld = p.vt_ld;
    const T* kb = (const T*)p.k + kvh * p.k_head;
    const T* cb = (const T*)(p.shared != nullptr ? p.shared : p.k);
    const T* vb = (const T*)p.vt + (ROWS ? kvh * p.v_head : (size_t)kvh * V * vt_ld);
    // A key row is [part of the head's own | part that the heads share]; keys past the end repeat the last one and are never
    // weighted, value rows past vdim repeat the first one and are never stored.  A thread loads eight elements of every
    // slice of one key, and of every 32nd value row.
    Frag<DT> kr[VEC ? NK : 1], vr[ROWS ? 4 : (VEC ? NV / 2 : 1)];
    const uint32_t slot = tile_slot<DT>(l16, 8u * lg);
    const uint32_t krow = tid >> 2, kcol = (tid & 3u) * 8u;
    const uint32_t vrow = ROWS ? (tid >> 4) * 8u : tid >> 3, vcol = ROWS ? (tid & 15u) * 4u : (tid & 7u) * 8u;   // element, key
    static_assert(!ROWS || (VEC && DT != kFP32 && NV <= 8), "values in rows");
    auto request = [&](uint32_t k0) {
        const uint32_t key = k0 + krow < keys_total ? k0 + krow : keys_total - 1u;
        const T* un = kb + key * kld + kcol;
        const T* ro = cb + key * cld + kcol;
#pragma unroll
        for (int j = 0; j < NK; ++j) {
            const uint32_t c = 32u * j + kcol;
            kr[j] = frag_load<DT>(c < D ? un + 32u * j : (c < Dq ? ro + (32 * j - (int)D) : cb));
        }
        if constexpr (ROWS) {
#pragma unroll
            for (uint32_t j = 0; j < 4u; ++j)
                vr[j] = frag_load<DT>(vb + (k0 + vcol + j < keys_total ? k0 + vcol + j : keys_total - 1u) * kld + (vrow < V ? vrow : 0u));
        } else {
            const T* vp = vb + k0 + vcol;
#pragma unroll
            for (int j = 0; j < NV / 2; ++j) vr[j] = frag_load<DT>(vp + (vrow + 32u * j < V ? vrow + 32u * j : 0u) * vt_ld);
        }
    };
    if constexpr (VEC) request(0u);
    for (uint32_t k0 = 0; k0 < kend; k0 += kKeys) {
        __syncthreads();
        if constexpr (VEC) {
            if (Dq < 32u * NK) {                                           // here, where the loads have long arrived
#pragma unroll
                for (int j = 0; j < NK; ++j)
                    if (32u * j + kcol >= Dq) kr[j] = Frag<DT>{};
            }
#pragma unroll
            for (int j = 0; j < NK; ++j) store8(Kl + krow * KL + tile_slot<DT>(krow, kcol) + 32u * j, kr[j]);
            if constexpr (ROWS) {
                if (vrow < 16u * NV) {
#pragma unroll
                    for (uint32_t i = 0; i < 8u; ++i) {
                        const uint32_t sel = (i & 1u) ? 0x07060302u : 0x05040100u;
                        *(u32x2*)(Vl + (vrow + i) * VL + value_slot<DT>(vrow + i, vcol)) = u32x2{__builtin_amdgcn_perm(vr[1].v[i >> 1], vr[0].v[i >> 1], sel),
                                                                       __builtin_amdgcn_perm(vr[3].v[i >> 1], vr[2].v[i >> 1], sel)};
                    }
                }
            } else {
#pragma unroll
                for (int j = 0; j < NV / 2; ++j) {
                    T* row = Vl + (vrow + 32u * j) * VL;
                    if constexpr (DT == kFP32) store8(row + vcol, vr[j]);
                    else {
                        *(u32x2*)(row + value_slot<DT>(vrow, vcol)) = u32x2{vr[j].v[0], vr[j].v[1]};
                        *(u32x2*)(row + value_slot<DT>(vrow, vcol + 4u)) = u32x2{vr[j].v[2], vr[j].v[3]};
                    }
                }
            }
        } else {
            for (uint32_t i = tid; i < kKeys * 32u * NK; i += 256u) {
                const uint32_t r = i / (32u * NK), c = i % (32u * NK), key = k0 + r < keys_total ? k0 + r : keys_total - 1u;
                Kl[r * KL + tile_slot<DT>(r, c)] = c < D ? kb[key * kld + c] : (c < Dq ? cb[key * cld + c - D] : (T)0);
            }
            for (uint32_t i = tid; i < 16u * NV * kKeys; i += 256u) {
                const uint32_t d = i / kKeys, c = i % kKeys;
                Vl[d * VL + value_slot<DT>(d, c)] = d < V ? vb[d * vt_ld + k0 + c] : (T)0;
            }
        }
        __syncthreads();
        if constexpr (VEC) { if (k0 + kKeys < kend) request(k0 + kKeys); }
        if (k0 > wave_last) continue;                                      // every key of the tile lies after the wave's queries
        f32x4 sc[MT][4];
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int t = 0; t < 4; ++t) sc[m][t] = f32x4{0.f, 0.f, 0.f, 0.f};
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int s = 0; s < NK; ++s)
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const Frag<DT> a = frag_load<DT>(Kl + (16u * t + l16) * KL + 32u * s + slot);
#pragma unroll
                for (int m = 0; m < MT; ++m) mma(a, qf[m][s], sc[m][t]);
            }
        __builtin_amdgcn_s_setprio(0);
        const bool edge = k0 + kKeys > wave_first + 1u;                    // some key may lie after some query of the wave
        if (edge) {
#pragma unroll
            for (int m = 0; m < MT; ++m)
#pragma unroll
                for (int t = 0; t < 4; ++t)
#pragma unroll
                    for (int v = 0; v < 4; ++v)
                        if (k0 + 16u * t + 4u * lg + (uint32_t)v > qpos[m]) sc[m][t][v] = -__builtin_inff();
        }
        float best[MT];
        bool more = false;
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            best[m] = -__builtin_inff();
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
                for (int v = 0; v < 4; ++v) best[m] = fmaxf(best[m], sc[m][t][v]);
        }
#pragma unroll
        for (int m = 0; m < MT; ++m) best[m] = fmaxf(best[m], __shfl_xor(best[m], 16, 64));
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            best[m] = fmaxf(best[m], __shfl_xor(best[m], 32, 64));
            best[m] = fmaxf(mx[m], best[m] * scale2);
            more |= best[m] > mx[m];
        }
        if (__any(more)) {
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                const float corr = __builtin_amdgcn_exp2f(from[m] - base(best[m]));
                mx[m] = best[m];
                from[m] = base(mx[m]);
                sum[m] *= corr;
#pragma unroll
                for (int n = 0; n < NV; ++n) o[m][n] *= corr;
            }
        }
        Frag<DT> part[2][MT][P];
#pragma unroll
        for (int t = 0; t < 2; ++t) {
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                float w[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    w[e] = __builtin_amdgcn_exp2f(__builtin_fmaf(sc[m][2 * t + (e >> 2)][e & 3], scale2, -from[m]));
                    sum[m] += w[e];
                }
                frag_parts(w, part[t][m]);
            }
        }
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int n = 0; n < NV; ++n) {
                Frag<DT> a;
                if constexpr (DT == kFP32) {
                    const T* vk = Vl + (16u * n + l16) * VL + 32u * t + 4u * lg;
                    const f32x4 x = *(const f32x4*)vk, y = *(const f32x4*)(vk + 16);
#pragma unroll
                    for (int e = 0; e < 4; ++e) { a.v[e] = x[e]; a.v[4 + e] = y[e]; }
                } else {
                    a = frag_load<DT>(Vl + (16u * n + l16) * VL + 32u * t + slot);
                }
#pragma unroll
                for (int m = 0; m < MT; ++m)
#pragma unroll
                    for (int i = 0; i < P; ++i) mma(a, part[t][m][i], o[m][n]);
            }
        if constexpr (DT != kFP32) {                                       // vector instructions of eight scores: about 6.5 a score, up to 14 in three parts
            constexpr int AHEAD = 3, VEC8 = P == 3 ? 112 : 52;
            __builtin_amdgcn_sched_group_barrier(0x100, AHEAD, 0);
            __builtin_amdgcn_sched_group_barrier(0x002, VEC8 * MT, 0);
#pragma unroll
            for (int i = 0; i < 2 * NV; ++i) {
#pragma unroll
                for (int j = 0; j < P * MT; ++j) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                    if (i < NV) __builtin_amdgcn_sched_group_barrier(0x002, (VEC8 + P * NV - 1) / (P * NV), 0);
                }
                if (i + AHEAD < 2 * NV) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            }
        }
    }
#pragma unroll
    for (int m = 0; m < MT; ++m) {
        float t = sum[m];
        t += __shfl_xor(t, 16, 64);
        t += __shfl_xor(t, 32, 64);
        const uint32_t row = q0 + 16u * (MT * wave + (uint32_t)m) + l16;
        if (row < rows) {
            float r = p.out_scale / t;
            if (p.gate != nullptr) r *= sigmoid_f(E::load(p.gate, (size_t)row * p.gate_ld + h));
#pragma unroll
            for (int n = 0; n < NV; ++n)
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const uint32_t d = 16u * n + 4u * lg + (uint32_t)v;
                    if (d < V) E::store(p.out, (size_t)row * p.out_ld + h * V + d, o[m][n][v] * r);
                }
        }
    }
}

template <int DT, int MT, int NK, int NV, bool VEC = true, bool ROWS = false>
static hipError_t tile_launch(const TileAttention& p, uint32_t start, uint32_t rows, hipStream_t s) {
    constexpr uint32_t PAD = DT == kFP32 ? 4u : 8u;
    constexpr size_t lds = (size_t)(kKeys * (32u * NK + PAD) + 16u * NV * (kKeys + PAD)) * Elem<DT>::bytes;
    static_assert(lds <= 160u * 1024u, "tiles must fit the LDS of a compute unit");
    if (hipError_t e = allow_lds<tile_attention_kernel<DT, MT, NK, NV, VEC, ROWS>>(lds); e != hipSuccess) return e;
    const uint32_t blocks = (rows + 64u * MT - 1u) / (64u * MT);
    hipLaunchKernelGGL((tile_attention_kernel<DT, MT, NK, NV, VEC, ROWS>), dim3(blocks * ((p.heads + 7u) / 8u * 8u)), dim3(256), lds, s,
                       p, start, rows, blocks);
    return hipGetLastError();
}

}  // namespace decdec
