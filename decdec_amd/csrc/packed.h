// Packed weights, 3 and 4 bits, decoded 32 channels of an output at a time: byte-permute look-ups in tables of 16-bit values.
#pragma once
#include "common.h"
#include "mma.h"
#include "anyprec_role.h"

namespace decdec {

enum { kAnyprec = 0, kLutgemm = 1, kSqllm = 2 };

// Byte tables of an output: LO = low bytes of the entries, HI = high bytes.
template <int BITS> struct Tables { uint32_t lo[1 << (BITS - 2)], hi[1 << (BITS - 2)]; };

template <int BITS>
__device__ __forceinline__ Tables<BITS> tables_of(const uint32_t (&e)[1 << (BITS - 1)]) {
    Tables<BITS> t;
#pragma unroll
    for (int i = 0; i < (1 << (BITS - 2)); ++i) {
        t.lo[i] = __builtin_amdgcn_perm(e[2 * i + 1], e[2 * i], 0x06040200u);
        t.hi[i] = __builtin_amdgcn_perm(e[2 * i + 1], e[2 * i], 0x07050301u);
    }
    return t;
}

// Four weights by their indices in the bytes of `idx` (bits above the index may be set): a = the first two, b = the others.
template <int BITS>
__device__ __forceinline__ void look_up(const Tables<BITS>& t, uint32_t idx, uint32_t& a, uint32_t& b) {
    const uint32_t sel = idx & 0x07070707u;
    uint32_t L = __builtin_amdgcn_perm(t.lo[1], t.lo[0], sel), H = __builtin_amdgcn_perm(t.hi[1], t.hi[0], sel);
    if constexpr (BITS == 4) {
        const uint32_t top = (idx >> 3) & 0x01010101u, half = (top << 8) - top;        // 0xFF where the index is 8 or more
        L = bit_select(half, __builtin_amdgcn_perm(t.lo[3], t.lo[2], sel), L);
        H = bit_select(half, __builtin_amdgcn_perm(t.hi[3], t.hi[2], sel), H);
    }
    a = __builtin_amdgcn_perm(H, L, 0x05010400u);
    b = __builtin_amdgcn_perm(H, L, 0x07030602u);
}

// Eight neighbouring channels of a SqueezeLLM unit, j a constant after unrolling.
template <int BITS>
__device__ __forceinline__ u32x4 sqllm_piece(const uint32_t (&w)[BITS], const Tables<BITS>& t, int j) {
    uint32_t v[4];
    if constexpr (BITS == 4) {
        const uint32_t odd = w[j] >> 4;
        look_up<4>(t, __builtin_amdgcn_perm(odd, w[j], 0x05010400u), v[0], v[1]);
        look_up<4>(t, __builtin_amdgcn_perm(odd, w[j], 0x07030602u), v[2], v[3]);
    } else {                                               // eight 3-bit fields from bit 24 j of the 96
        const uint32_t part = j == 0 ? w[0] : j == 1 ? __builtin_amdgcn_alignbit(w[1], w[0], 24) : j == 2 ? __builtin_amdgcn_alignbit(w[2], w[1], 16) : w[2] >> 8;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const uint32_t s = part >> (12 * h);
            look_up<3>(t, (s & 7u) | ((s << 5) & 0x700u) | ((s << 10) & 0x70000u) | ((s << 15) & 0x7000000u), v[2 * h], v[2 * h + 1]);
        }
    }
    return u32x4{v[0], v[1], v[2], v[3]};
}

// The 32 weights of a unit (w: its words) as four fragments of eight neighbouring channels, in their order.  Indices are brought next to
// each other before they are looked up, by eight byte permutes a unit in SqueezeLLM's four bits and four in the planes of the others, so that
// neither the activations (which every workgroup would have to arrange again) nor the weights have to be put in order afterwards (sixteen).
template <int FMT, int BITS>
__device__ __forceinline__ void decode(const uint32_t (&w)[BITS], const Tables<BITS>& t, u32x4 (&f)[4]) {
    if constexpr (FMT == kSqllm) {
#pragma unroll
        for (int j = 0; j < 4; ++j) f[j] = sqllm_piece<BITS>(w, t, j);
    } else {
        // T[o]: nibble n carries the index of bit 4 n + o of the planes, plane 0 its top bit
        uint32_t T[4];
#pragma unroll
        for (int o = 0; o < 4; ++o) {
            uint32_t v = 0u;
#pragma unroll
            for (int p = 0; p < BITS; ++p) {
                const int to = BITS - 1 - p;               // bit of the nibble
                const uint32_t moved = to >= o ? w[p] << (to - o) : w[p] >> (o - to);
                v = bit_select(0x11111111u << to, moved, v);
            }
            T[o] = v;
        }
        // channel e of piece j -- LUT-GEMM: bit 8 j + e; any-precision: bit 31 - (8 j + e).  Two neighbouring channels of two
        // neighbouring pieces side by side: (piece 2 h, c), (2 h, c + 1), (2 h + 1, c), (2 h + 1, c + 1) for c = 0 or 2 in one nibble of
        // the bytes and c + 4 in the other
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int c = 0; c < 4; c += 2) {
                const uint32_t x = FMT == kLutgemm ? T[c] : T[3 - c], y = FMT == kLutgemm ? T[c + 1] : T[2 - c];
                const uint32_t sel = FMT == kLutgemm ? (h ? 0x07030602u : 0x05010400u) : (h ? 0x04000501u : 0x06020703u);
                const uint32_t both = __builtin_amdgcn_perm(y, x, sel);
#pragma unroll
                for (int e = c; e < 8; e += 4) {
                    const bool high = FMT == kLutgemm ? e >= 4 : e < 4;
                    uint32_t a, b;
                    look_up<BITS>(t, high ? both >> 4 : both, a, b);
                    f[2 * h][e >> 1] = a;
                    f[2 * h + 1][e >> 1] = b;
                }
            }
    }
}

// The values of a LUT-GEMM group (a: its scales and bias), plane 0 the top bit of the index: planes summed in order, then the bias, rounded once.
template <int DT, int BITS>
__device__ __forceinline__ Tables<BITS> group_tables(const float (&a)[BITS + 1]) {
    constexpr int V = 1 << BITS;
    float s[V];
#pragma unroll
    for (int i = 0; i < V; ++i) {
        s[i] = (i >> (BITS - 1)) & 1 ? a[0] : -a[0];
#pragma unroll
        for (int p = 1; p < BITS; ++p) s[i] = (i >> (BITS - 1 - p)) & 1 ? s[i] + a[p] : s[i] - a[p];
        s[i] += a[BITS];
    }
    uint32_t e[V / 2];
#pragma unroll
    for (int i = 0; i < V / 2; ++i) {
        if constexpr (DT == kBF16) e[i] = pack_bf16(s[2 * i], s[2 * i + 1]);
        else e[i] = Elem<DT>::to_raw(s[2 * i]) | (Elem<DT>::to_raw(s[2 * i + 1]) << 16);
    }
    return tables_of<BITS>(e);
}

}  // namespace decdec
