// Pieces of the router kernels (router.hip, decode.hip): the two 16-bit element types, sort keys of logits, and the top-k and
// softmax of a token by sixteen lanes.
#pragma once

#include "common.h"

namespace fmahip {
namespace {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(8))) _Float16 f16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;

constexpr int kTok = 16;         // tokens per workgroup = rows of one MFMA tile
constexpr int kStepK = 128;      // reduction elements per step of one wavefront: 4 lane groups x 32 elements
constexpr int kMaxTopK = 64;     // top_k limit (FMA_MAX_ROUTER_TOP_K)
constexpr int kRowPad = 16;      // keeps the four token rows one wavefront scans in different LDS banks

struct RouterBf16 {
    using frag = bf16x8;
    static constexpr uint32_t kInfBits = 0x7f80u, kNanBits = 0x7fc0u;
    static __device__ __forceinline__ float round(float x) { return (float)(__bf16)x; }
    static __device__ __forceinline__ uint16_t bits(float x) { return __builtin_bit_cast(uint16_t, (__bf16)x); }
    static __device__ __forceinline__ float from_bits(uint16_t b) { return bf16_bits_to_float(b); }
    static __device__ __forceinline__ f32x4 mfma(frag a, frag b, f32x4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
    }
};
struct RouterF16 {
    using frag = f16x8;
    static constexpr uint32_t kInfBits = 0x7c00u, kNanBits = 0x7e00u;
    static __device__ __forceinline__ float round(float x) { return (float)(_Float16)x; }
    static __device__ __forceinline__ uint16_t bits(float x) { return __builtin_bit_cast(uint16_t, (_Float16)x); }
    static __device__ __forceinline__ float from_bits(uint16_t b) { return (float)__builtin_bit_cast(_Float16, b); }
    static __device__ __forceinline__ f32x4 mfma(frag a, frag b, f32x4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
    }
};

struct RouterArgs {
    const uint16_t* x;       // [T, H]
    const uint16_t* w;       // [E, H]
    uint16_t* logits;        // [T, E]
    uint16_t* weights;       // [T, k]
    int32_t* selected;       // [T, k]
    uint32_t* counts;        // [E] or null
    uint32_t* hist;          // [ceil(T / 16), E] or null: choices per expert among each 16 consecutive tokens
    int64_t T;
    int32_t H, E, k;
};

template <typename F>
__device__ __forceinline__ F load_frag(const uint16_t* p) {
    return __builtin_bit_cast(F, *reinterpret_cast<const u32x4*>(p));
}

// ---- sort keys ------------------------------------------------------------------------------------------------------
// The top-k works on one 32-bit key per logit: the 16 bits of the (already rounded) logit mapped so that unsigned order
// equals numeric order, with NaN above everything (where torch.topk puts it) and -0 equal to +0, then 0xffff - column
// in the low half. The unsigned maximum of such keys is the largest logit and, among equal logits, the lowest column.
// Key 0 marks a column that is already taken (no real key is 0: the low half of a real key is at least 0xffff - 1023).
template <typename EL>
__device__ __forceinline__ uint32_t make_key(uint32_t bits, int column) {
    uint32_t ord;
    if ((bits & 0x7fffu) > EL::kInfBits) ord = 0xffffu;
    else {
        if (bits == 0x8000u) bits = 0;
        ord = (bits & 0x8000u) ? (~bits & 0xffffu) : (bits | 0x8000u);
    }
    return (ord << 16) | (0xffffu - (uint32_t)column);
}
template <typename EL>
__device__ __forceinline__ float key_value(uint32_t key) {
    const uint32_t ord = key >> 16;
    const uint32_t bits = ord == 0xffffu ? EL::kNanBits : ((ord & 0x8000u) ? (ord & 0x7fffu) : (~ord & 0xffffu));
    return EL::from_bits((uint16_t)bits);
}
__device__ __forceinline__ int key_column(uint32_t key) { return (int)(0xffffu - (key & 0xffffu)); }

// All-reduce over the 16 lanes of a DPP row (lanes 16g .. 16g+15 of the wavefront) with data-parallel-primitive
// moves: neighbours inside a quad, the other pair of the quad, the mirrored quad of the half row, the mirrored half.
// Every lane ends up with the same value; for the float sum the order of additions is the same fixed tree in all lanes.
template <int CTRL>
__device__ __forceinline__ uint32_t dpp_u32(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xf, 0xf, false);
}
constexpr int kDppXor1 = 0xb1, kDppXor2 = 0x4e, kDppHalfMirror = 0x141, kDppMirror = 0x140;
__device__ __forceinline__ uint32_t row16_max(uint32_t v) {
    v = max(v, dpp_u32<kDppXor1>(v));
    v = max(v, dpp_u32<kDppXor2>(v));
    v = max(v, dpp_u32<kDppHalfMirror>(v));
    v = max(v, dpp_u32<kDppMirror>(v));
    return v;
}
__device__ __forceinline__ float row16_sum(float v) {
    v += __uint_as_float(dpp_u32<kDppXor1>(__float_as_uint(v)));
    v += __uint_as_float(dpp_u32<kDppXor2>(__float_as_uint(v)));
    v += __uint_as_float(dpp_u32<kDppHalfMirror>(__float_as_uint(v)));
    v += __uint_as_float(dpp_u32<kDppMirror>(__float_as_uint(v)));
    return v;
}

// Weights of NR tokens by the 16 lanes of a DPP row from their sorted choices: choice j is the key mine[t][j / 16] of lane j % 16,
// first[t] the first of them (the largest logit) in every lane.
template <typename EL, int NR>
__device__ __forceinline__ void softmax_tokens(const uint32_t (&mine)[NR][kMaxTopK / 16], const uint32_t (&first)[NR], int c,
                                               const int64_t (&token)[NR], const int64_t tok0, const RouterArgs& a,
                                               uint32_t* s_hist) {
    const int E = a.E, k = a.k;
#pragma unroll
    for (int t = 0; t < NR; ++t) {
        const float vmax = key_value<EL>(first[t]);
        float e[kMaxTopK / 16];
        float sum = 0.f;
#pragma unroll
        for (int i = 0; i < kMaxTopK / 16; ++i) {
            e[i] = c + 16 * i < k ? expf(key_value<EL>(mine[t][i]) - vmax) : 0.f;
            sum += e[i];
        }
        sum = row16_sum(sum);
        if (token[t] < a.T) {
#pragma unroll
            for (int i = 0; i < kMaxTopK / 16; ++i) {
                const int j = c + 16 * i;
                if (j < k) {
                    const int col = key_column(mine[t][i]);
                    a.selected[token[t] * k + j] = col;
                    a.weights[token[t] * k + j] = EL::bits(e[i] / sum);
                    if (a.counts || a.hist) atomicAdd(&s_hist[(int)((token[t] - tok0) >> 4) * E + col], 1u);
                }
            }
        }
    }
}


// Top-k and softmax of NR tokens at once by the 16 lanes of a DPP row (the NR chains of dependent reductions are
// independent of each other, which is what hides their latency); keys[t] is token t's row of sort keys in LDS, of which
// lane c owns (reads, and clears when chosen) the columns congruent to c mod 16. Choice j is remembered by lane
// j % 16, so that after the k rounds every lane turns its own choices into weights and writes them.
template <typename EL, int NR>
__device__ __forceinline__ void topk_softmax_tokens(uint32_t* const (&keys)[NR], int c, const int64_t (&token)[NR],
                                                    const int64_t tok0, const RouterArgs& a, uint32_t* s_hist) {
    const int E = a.E, k = a.k;
    uint32_t mine[NR][kMaxTopK / 16];
    uint32_t first[NR];
#pragma unroll
    for (int t = 0; t < NR; ++t) {
        first[t] = 0;
#pragma unroll
        for (int i = 0; i < kMaxTopK / 16; ++i) mine[t][i] = 0;
    }
    for (int j = 0; j < k; ++j) {
        uint32_t best[NR];
#pragma unroll
        for (int t = 0; t < NR; ++t) best[t] = 0;
        for (int n = c; n < E; n += 16)
#pragma unroll
            for (int t = 0; t < NR; ++t) best[t] = max(best[t], keys[t][n]);
#pragma unroll
        for (int t = 0; t < NR; ++t) best[t] = row16_max(best[t]);  // top_k <= E: a real key
#pragma unroll
        for (int t = 0; t < NR; ++t) {
            const int col = key_column(best[t]);
            if ((col & 15) == c) keys[t][col] = 0;
            if (j == 0) first[t] = best[t];
#pragma unroll
            for (int i = 0; i < kMaxTopK / 16; ++i)
                if (c == (j & 15) && (j >> 4) == i) mine[t][i] = best[t];
        }
    }
    softmax_tokens<EL, NR>(mine, first, c, token, tok0, a, s_hist);
}

// The same for one token whose keys are in registers: lane c holds the keys of the columns congruent to c mod 16 (0 where there
// is none), NK = ceil(E / 16) of them.
template <typename EL, int NK>
__device__ __forceinline__ void topk_softmax_in_registers(uint32_t (&keys)[NK], int c, int64_t token, const RouterArgs& a,
                                                          int64_t tok0 = 0, uint32_t* s_hist = nullptr) {
    uint32_t mine[1][kMaxTopK / 16] = {};
    uint32_t first[1] = {0};
    for (int j = 0; j < a.k; ++j) {
        uint32_t best = keys[0];
#pragma unroll
        for (int i = 1; i < NK; ++i) best = max(best, keys[i]);
        best = row16_max(best);  // top_k <= E: a real key, and no two keys are equal
#pragma unroll
        for (int i = 0; i < NK; ++i) keys[i] = keys[i] == best ? 0u : keys[i];
        if (j == 0) first[0] = best;
#pragma unroll
        for (int i = 0; i < kMaxTopK / 16; ++i)
            if (c == (j & 15) && (j >> 4) == i) mine[0][i] = best;
    }
    const int64_t tokens[1] = {token};
    softmax_tokens<EL, 1>(mine, first, c, tokens, tok0, a, s_hist);
}

}  // namespace
}  // namespace fmahip
