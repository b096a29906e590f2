// The router's product for few tokens (router.hip, decode.hip): a workgroup per 16 tokens x 16 experts, operands by direct global ->
// LDS loads of whole lines, 128 KB in flight. It is bound by the latency of one or two trips to memory, not by the 16 x 16 x H product
// or the bytes, as the kernels of router.hip are that give 16 to 64 tokens one workgroup with the whole router matrix. The same sums in
// the same order as those (for up to 16 experts: four wavefronts with every fourth step each, partial sums added in that order), so
// logits and choice have the same bits.
#pragma once

#include "gemm_parts.h"
#include "router_parts.h"

namespace fmahip {
namespace {

constexpr uint32_t kRowBytes = kStepK * 2;  // bytes of a row per step
constexpr uint32_t kStepBytes = 32 * kRowBytes;
constexpr int kBatch = 8;  // steps per batch; two batches (128 KB) in LDS

// LDS position of 16-byte chunk c of row r (16 chunks per row): the sixteen rows of a fragment read take sixteen columns
__device__ __forceinline__ uint32_t chunk_off(uint32_t r, uint32_t c) { return r * kRowBytes + ((c ^ (r & 15u)) << 4); }

// One workgroup per 16 tokens x 16 experts. Four wavefronts fetch, 16 of the 64 load instructions of a batch each (a step: 16
// token rows and 16 expert rows of 256 bytes, four rows per instruction), two batches in flight: up to a row of 2048 elements is
// one trip to memory, however cold. SPLIT: step s is multiplied by wavefront s % 4; otherwise by the first, in order.
template <typename EL, bool SPLIT>
__global__ __launch_bounds__(256) void router_logits_kernel(const RouterArgs a) {
    using frag = typename EL::frag;
    __shared__ __attribute__((aligned(1024))) uint8_t s_steps[2][kBatch * kStepBytes];
    __shared__ float s_part[SPLIT ? 4 : 1][kTok][16];
    const uint32_t lane = threadIdx.x & 63u, wave = gemm::uniform(threadIdx.x >> 6);
    const uint32_t tok0 = blockIdx.x * kTok, e0 = blockIdx.y * 16u;
    const uint32_t H2 = (uint32_t)a.H * 2u;
    const uint32_t toks = (uint32_t)a.T - tok0 < 16u ? (uint32_t)a.T - tok0 : 16u;
    const uint32_t exps = (uint32_t)a.E - e0 < 16u ? (uint32_t)a.E - e0 : 16u;
    // rows past the end are out of the descriptors' range and arrive as zeros, and so do the chunks past the end of a row
    const gemm::u32x4 rx = gemm::make_rsrc_words(a.x + (uint64_t)tok0 * a.H, toks * H2);
    const gemm::u32x4 rw = gemm::make_rsrc_words(a.w + (uint64_t)e0 * a.H, exps * H2);
    const uint32_t lr = lane >> 4, lp = lane & 15u;
    const uint32_t nbatch = (H2 + kBatch * kRowBytes - 1) / (kBatch * kRowBytes);

    // wavefronts 0 and 1 fetch the token rows, 2 and 3 the expert rows, eight rows of every step each
    const gemm::u32x4 src = wave < 2 ? rx : rw;
    const uint32_t half = (wave & 1u) * 8u;
    auto issue = [&](uint32_t b) {
        const uint32_t lds0 = gemm::lds_address(s_steps[b & 1u]) + wave * (kStepBytes / 4);
#pragma unroll
        for (uint32_t s = 0; s < kBatch; ++s) {
            const uint32_t kb = (b * kBatch + s) * kRowBytes;
#pragma unroll
            for (uint32_t l = 0; l < 2; ++l) {
                const uint32_t row = half + l * 4u;
                const uint32_t chunk = lp ^ ((row + lr) & 15u);
                const uint32_t v = kb + chunk * 16u < H2 ? lr * H2 + chunk * 16u : gemm::kOutOfRange;
                gemm::load_lds<false>(src, v, row * H2 + kb, lds0 + s * kStepBytes + l * 1024u);
            }
        }
    };
    f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
    const uint32_t r = lane & 15u, q = lane >> 4;
    issue(0);
    issue(1);
    for (uint32_t b = 0; b < nbatch; ++b) {
        gemm::wait_vm<2 * kBatch>();
        __syncthreads();
        const uint8_t* steps = s_steps[b & 1u];
#pragma unroll
        for (uint32_t s = 0; s < kBatch; ++s) {
            if (SPLIT ? (s & 3u) != wave : wave != 0) continue;
            const uint8_t* stage = steps + s * kStepBytes;
#pragma unroll
            for (uint32_t j = 0; j < 4; ++j) {
                const frag xf = load_frag<frag>(reinterpret_cast<const uint16_t*>(stage + chunk_off(r, q * 4u + j)));
                const frag wf = load_frag<frag>(reinterpret_cast<const uint16_t*>(stage + 16 * kRowBytes + chunk_off(r, q * 4u + j)));
                acc = EL::mfma(xf, wf, acc);
            }
        }
        gemm::wait_lds();
        __syncthreads();
        issue(b + 2);  // past the end of the rows: zeros, so that the count above holds
    }
    gemm::wait_vm<0>();
    // a lane holds tokens 4 q .. 4 q + 3 of expert r
    if constexpr (SPLIT) {
#pragma unroll
        for (int i = 0; i < 4; ++i) s_part[wave][q * 4 + i][r] = acc[i];
        __syncthreads();
        const uint32_t tok = threadIdx.x >> 4, c = threadIdx.x & 15u;
        const float v = (s_part[0][tok][c] + s_part[1][tok][c]) + (s_part[2][tok][c] + s_part[3][tok][c]);
        if (tok < toks && c < exps) a.logits[(uint64_t)(tok0 + tok) * a.E + e0 + c] = EL::bits(v);
    } else if (wave == 0) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t tok = q * 4 + i;
            if (tok < toks && r < exps) a.logits[(uint64_t)(tok0 + tok) * a.E + e0 + r] = EL::bits(acc[i]);
        }
    }
}

}  // namespace
}  // namespace fmahip
