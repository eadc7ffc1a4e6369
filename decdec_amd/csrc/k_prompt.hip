// Attention of a prompt in the plain decoder: rotary embedding and cache append of all its tokens in one launch, then the tiled
// kernel over the cache (tile_attention.h).  Tokens may stand at any positions.  Bound by the tiled kernel's products and
// softmax instructions: 32 query and 8 key heads of 128, 1999 tokens in bf16 12 and 120 us, 512 in fp16 5 and 20 us.  torch
// operations (batched products in fp32, softmax, mask, copies) took 4 of the 6.0 ms of the first prompt through two layers, and 0.5
// of the 1.6 ms of the second.
#include "launch.h"
#include "tile_attention.h"

namespace decdec {

// Queries to q_out [rows][n_head][D], keys and values to the caches [n_kv][max_seq][D].  cos / sin [rows][D], the rows of the
// tokens (tables: [max_seq][D], and a token's row is its position's, not a number where the tables have none); pair (i, i + D / 2)
// turns, in fp32, rounded once.  A thread takes eight elements of each half of a head.
template <int DT, int D>
__global__ __launch_bounds__(256) void prompt_append_kernel(const PromptParams p) {
    using T = uint16_t;
    using E = Elem<DT>;
    constexpr uint32_t PER = D / 16;                       // threads of a head
    const uint32_t heads = p.n_head + 2u * p.n_kv, id = blockIdx.x * 256u + threadIdx.x, c = id % PER * 8u;
    const uint32_t t = id / PER / heads, h = id / PER % heads;
    if (t >= p.rows) return;
    const long long pos = p.positions[t];
    const T* src = (const T*)p.qkv + ((size_t)t * heads + h) * D + c;
    u32x4 a = *(const u32x4*)src, b = *(const u32x4*)(src + D / 2);
    const bool cached = pos >= 0 && pos < (long long)p.max_seq;
    if (p.tables && !cached) a = b = u32x4{~0u, ~0u, ~0u, ~0u};
    else if (h < p.n_head + p.n_kv) {
        const size_t row = p.tables ? (size_t)pos : t;
        const T* cs = (const T*)p.cos + row * D + c;
        const T* sn = (const T*)p.sin + row * D + c;
        const u32x4 ca = *(const u32x4*)cs, cb = *(const u32x4*)(cs + D / 2), sa = *(const u32x4*)sn, sb = *(const u32x4*)(sn + D / 2);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            uint32_t lo = 0u, hi = 0u;
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const auto at = [&](const u32x4& v) { return E::from_raw((v[i] >> (16 * e)) & 0xFFFFu); };
                const float u = at(a), w = at(b);
                lo |= E::to_raw(u * at(ca) - w * at(sa)) << (16 * e);
                hi |= E::to_raw(w * at(cb) + u * at(sb)) << (16 * e);
            }
            a[i] = lo;
            b[i] = hi;
        }
    }
    T* dst;
    if (h < p.n_head) dst = (T*)p.q_out + ((size_t)t * p.n_head + h) * D;
    else {
        if (!cached) return;
        const bool key = h < p.n_head + p.n_kv;
        dst = (T*)(key ? p.k_cache : p.v_cache) + ((size_t)(h - p.n_head - (key ? 0u : p.n_kv)) * p.max_seq + (size_t)pos) * D;
    }
    *(u32x4*)(dst + c) = a;
    *(u32x4*)(dst + c + D / 2) = b;
}

template <int DT, int D>
static hipError_t prompt_dt(const PromptParams& p, hipStream_t s) {
    const uint64_t threads = (uint64_t)p.rows * (p.n_head + 2u * p.n_kv) * (D / 16);
    hipLaunchKernelGGL((prompt_append_kernel<DT, D>), dim3((uint32_t)((threads + 255u) / 256u)), dim3(256), 0, s, p);
    if (hipError_t e = hipGetLastError(); e != hipSuccess) return e;
    TileAttention a{};
    a.q = p.q_out; a.k = p.k_cache; a.vt = p.v_cache; a.out = p.out; a.positions = p.positions;
    a.k_head = a.v_head = (size_t)p.max_seq * D; a.k_row = D; a.vt_ld = p.max_seq; a.out_ld = p.n_head * D;
    a.heads = p.n_head; a.share = p.n_head / p.n_kv; a.dim = a.vdim = D;
    a.scale = 1.f / sqrtf((float)D); a.sink_score = -__builtin_inff(); a.out_scale = 1.f;
    // 128 queries a workgroup read the tiles half as often as 64; 64 where 128 would leave compute units without one
    if ((p.rows + 127u) / 128u * p.n_head >= 512u) return tile_launch<DT, 2, D / 32, D / 16, true, true>(a, 0u, p.rows, s);
    return tile_launch<DT, 1, D / 32, D / 16, true, true>(a, 0u, p.rows, s);
}

hipError_t launch_prompt_attention(int dt, const PromptParams& p, hipStream_t s) {
    if (dt == kFP16) return p.head_dim == 128u ? prompt_dt<kFP16, 128>(p, s) : prompt_dt<kFP16, 64>(p, s);
    return p.head_dim == 128u ? prompt_dt<kBF16, 128>(p, s) : prompt_dt<kBF16, 64>(p, s);
}

}  // namespace decdec
