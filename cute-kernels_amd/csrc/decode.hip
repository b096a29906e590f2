// The MoE layer for a few tokens (a decode step): router and routing index in two small launches, the two expert projections of
// thin_experts.hip and the combine, enqueued by one call.
//
// What bounds a step of one to sixteen tokens besides the expert weights is latency: every launch is a few microseconds of
// ramp-up, and the kernels for many tokens put a small batch on one or two compute units. The router's product (router.hip)
// gives every 16 to 64 tokens ONE workgroup, which then fetches the whole router matrix through one compute unit's address path
// (64 x 2048: 16 us, 128 x 4096: 46 us), and the index build behind it is two more launches of 4 to 8 us.
//  * router_logits_kernel (router_logits.h): a workgroup per 16 tokens x 16 experts, the same sums in the same order as the kernels
//    of router.hip, so logits and choice have the same bits.
//  * topk_index_kernel: ONE workgroup turns the logits of up to 1024 (token, choice) slots into weights, choice, counts, offsets
//    and both permutations: keys stay in registers, choices, histograms and ranks in LDS. It replaces the top-k tail of the router, the
//    scan and the placement.
//  * One token with up to eight choices needs no index: its two products choose their experts from the logits, and the second one
//    combines (thin_experts.hip).
#include "gemm_parts.h"
#include "router_logits.h"
#include "thin_experts.h"

namespace fmahip {
namespace {

constexpr int kIndexThreads = 1024;
constexpr int kIndexWaves = kIndexThreads / kWave;
constexpr int kIndexTokens = kIndexThreads / 16;  // tokens whose top-k runs at the same time
static_assert(FMA_MAX_DECODE_ROWS == kIndexThreads, "a thread per (token, choice) slot");

// NK = ceil(E / 16), rounded up to a power of two: keys per lane
template <typename EL, int NK>
__global__ __launch_bounds__(kIndexThreads) void topk_index_kernel(RouterArgs a, uint32_t nbits, uint32_t* __restrict__ counts,
                                                                   uint32_t* __restrict__ offsets, int32_t* __restrict__ perm,
                                                                   int32_t* __restrict__ inv) {
    constexpr int kEMax = FMA_MAX_DECODE_EXPERTS;
    __shared__ int32_t s_sel[kIndexThreads];
    __shared__ uint32_t s_cnt[kIndexWaves][kEMax];  // slots of each wavefront per expert, then where they start
    __shared__ uint32_t s_tot[kEMax / kWave];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    const uint32_t E = (uint32_t)a.E, R = (uint32_t)(a.T * a.k);

    // ---- weights and choice ----
    a.selected = s_sel;
    const uint32_t c = tid & 15u;
    for (uint32_t t0 = 0; t0 < (uint32_t)a.T; t0 += kIndexTokens) {
        if (t0 + (tid >> 6) * 4u >= (uint32_t)a.T) break;  // no token for this wavefront
        const uint32_t token = t0 + (tid >> 4);
        const uint32_t from = token < (uint32_t)a.T ? token : (uint32_t)a.T - 1u;  // (real keys; nothing is stored for it)
        uint32_t keys[NK];
#pragma unroll
        for (int i = 0; i < NK; ++i) {
            const uint32_t n = c + 16u * i;
            keys[i] = n < E ? make_key<EL>(a.logits[(uint64_t)from * E + n], (int)n) : 0u;
        }
        topk_softmax_in_registers<EL, NK>(keys, (int)c, (int64_t)token, a);
    }
    for (uint32_t i = tid; i < (uint32_t)kIndexWaves * E; i += kIndexThreads) s_cnt[i / E][i % E] = 0;
    __syncthreads();

    // ---- stable counting sort of the slots: rank among the wavefront's slots of the same expert, by ballots ----
    const bool live = tid < R;
    const uint32_t id = live ? (uint32_t)s_sel[tid] : 0u;
    uint64_t same = __ballot(live);
    for (uint32_t b = 0; b < nbits; ++b) {
        const bool bit = (id >> b) & 1u;
        const uint64_t bal = __ballot(bit);
        same &= bit ? bal : ~bal;
    }
    const uint32_t rank = (uint32_t)__popcll(same & ((1ull << lane) - 1ull));
    if (live && rank == 0) s_cnt[wave][id] = (uint32_t)__popcll(same);
    __syncthreads();
    uint32_t total = 0;
    if (tid < E)
        for (int w = 0; w < kIndexWaves; ++w) {
            const uint32_t v = s_cnt[w][tid];
            s_cnt[w][tid] = total;
            total += v;
        }
    uint32_t incl = 0;
    if (tid < (uint32_t)kEMax) {
        incl = wave_inclusive_scan<uint32_t>(total);
        if (lane == 63u) s_tot[wave] = incl;
    }
    __syncthreads();
    if (tid < E) {
        for (uint32_t w = 0; w < wave; ++w) incl += s_tot[w];
        counts[tid] = total;
        offsets[tid] = incl;
        for (int w = 0; w < kIndexWaves; ++w) s_cnt[w][tid] += incl - total;
    }
    __syncthreads();
    if (live) {
        const uint32_t pos = s_cnt[wave][id] + rank;
        perm[pos] = (int32_t)tid;
        inv[tid] = (int32_t)pos;
    }
}

template <typename EL>
int launch_router_logits(const RouterArgs& a, hipStream_t st) {
    const dim3 grid((uint32_t)((a.T + kTok - 1) / kTok), (uint32_t)((a.E + 15) / 16));
    if (a.E <= 16) hipLaunchKernelGGL((router_logits_kernel<EL, true>), grid, dim3(256), 0, st, a);
    else hipLaunchKernelGGL((router_logits_kernel<EL, false>), grid, dim3(256), 0, st, a);
    return launch_status("router_topk_index (logits)");
}

template <typename EL>
int launch_router_index(const RouterArgs& a, uint32_t* counts, uint32_t* offsets, int32_t* perm, int32_t* inv, hipStream_t st) {
    const int rc = launch_router_logits<EL>(a, st);
    if (rc) return rc;
    uint32_t nbits = 0;
    while ((1u << nbits) < (uint32_t)a.E) ++nbits;
    auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(1), dim3(kIndexThreads), 0, st, a, nbits, counts, offsets, perm, inv);
    };
    if (a.E <= 16) launch(topk_index_kernel<EL, 1>);
    else if (a.E <= 32) launch(topk_index_kernel<EL, 2>);
    else if (a.E <= 64) launch(topk_index_kernel<EL, 4>);
    else if (a.E <= 128) launch(topk_index_kernel<EL, 8>);
    else launch(topk_index_kernel<EL, 16>);
    return launch_status("router_topk_index (top-k and index)");
}

int64_t round_up(int64_t n) { return (n + 255) / 256 * 256; }

int check_router(const char* who, const void* x, const void* gate_weight, int64_t T, int64_t H, int64_t E, int64_t top_k, void* logits,
                 int dtype) {
    FMA_REQUIRE(dtype == FMA_BF16 || dtype == FMA_F16, FMA_ERR_BAD_DTYPE, "%s: dtype must be FMA_BF16 or FMA_F16 (got %d)", who, dtype);
    FMA_REQUIRE(E >= 1 && E <= FMA_MAX_DECODE_EXPERTS, FMA_ERR_TOO_MANY_EXPERTS, "%s: E must be in [1, %d] (got %lld)", who,
                FMA_MAX_DECODE_EXPERTS, (long long)E);
    FMA_REQUIRE(top_k >= 1 && top_k <= E && top_k <= FMA_MAX_ROUTER_TOP_K, FMA_ERR_BAD_SIZE,
                "%s: top_k must be in [1, min(E, %d)] (got %lld)", who, FMA_MAX_ROUTER_TOP_K, (long long)top_k);
    FMA_REQUIRE(T >= 1 && T <= FMA_MAX_DECODE_ROWS && T * top_k <= FMA_MAX_DECODE_ROWS, FMA_ERR_BAD_SIZE,
                "%s: T * top_k must be in [1, %d] (T=%lld, top_k=%lld)", who, FMA_MAX_DECODE_ROWS, (long long)T, (long long)top_k);
    FMA_REQUIRE(H >= 8 && H % 8 == 0 && H < (1 << 21), FMA_ERR_BAD_SIZE, "%s: H must be a multiple of 8 in [8, 2^21) (got %lld)",
                who, (long long)H);
    FMA_REQUIRE(x && gate_weight && logits, FMA_ERR_NULL_POINTER, "%s: NULL pointer", who);
    FMA_REQUIRE(aligned16(x) && aligned16(gate_weight), FMA_ERR_MISALIGNED, "%s: x and gate_weight must be 16-byte aligned", who);
    return FMA_OK;
}

RouterArgs router_args(const void* x, const void* gate_weight, int64_t T, int64_t H, int64_t E, int64_t top_k, void* logits) {
    RouterArgs a{};
    a.x = (const uint16_t*)x;
    a.w = (const uint16_t*)gate_weight;
    a.logits = (uint16_t*)logits;
    a.T = T;
    a.H = (int32_t)H;
    a.E = (int32_t)E;
    a.k = (int32_t)top_k;
    return a;
}

}  // namespace
}  // namespace fmahip

extern "C" {

int fma_router_topk_index(const void* x, const void* gate_weight, int64_t T, int64_t H, int64_t E, int64_t top_k, void* logits,
                          void* weights, uint32_t* counts, uint32_t* offsets, int32_t* perm, int32_t* inv, int dtype,
                          void* stream) {
    using namespace fmahip;
    const char* who = "router_topk_index";
    const int rc = check_router(who, x, gate_weight, T, H, E, top_k, logits, dtype);
    if (rc) return rc;
    FMA_REQUIRE(weights && counts && offsets && perm && inv, FMA_ERR_NULL_POINTER, "%s: NULL pointer", who);
    RouterArgs a = router_args(x, gate_weight, T, H, E, top_k, logits);
    a.weights = (uint16_t*)weights;
    hipStream_t st = (hipStream_t)stream;
    return dtype == FMA_BF16 ? launch_router_index<RouterBf16>(a, counts, offsets, perm, inv, st)
                             : launch_router_index<RouterF16>(a, counts, offsets, perm, inv, st);
}

int64_t fma_moe_decode_workspace_bytes(int64_t T, int64_t H, int64_t I, int64_t E, int64_t top_k) {
    if (T < 0 || H < 0 || I < 0 || E < 0 || top_k < 0) return 0;
    using fmahip::round_up;
    const int64_t R = T * top_k;
    return 2 * round_up(4 * E) + 2 * round_up(4 * R) + round_up(2 * R) + round_up(2 * R * H) +
           round_up(fma_thin_swiglu_experts_workspace_bytes(R, I));
}

int fma_moe_decode(const void* x, const void* gate_weight, const void* W1, const void* bias1, const void* W2, const void* bias2,
                   int64_t T, int64_t H, int64_t I, int64_t E, int64_t top_k, void* y, void* logits, void* workspace,
                   int64_t workspace_bytes, int dtype, void* stream) {
    using namespace fmahip;
    FMA_REQUIRE(workspace != nullptr && aligned16(workspace), FMA_ERR_MISALIGNED, "moe_decode: the workspace must be 16-byte aligned");
    FMA_REQUIRE(workspace_bytes >= fma_moe_decode_workspace_bytes(T, H, I, E, top_k), FMA_ERR_WORKSPACE_TOO_SMALL,
                "moe_decode: workspace of %lld bytes is smaller than the %lld needed", (long long)workspace_bytes,
                (long long)fma_moe_decode_workspace_bytes(T, H, I, E, top_k));
    const int64_t R = T * top_k;
    uint8_t* p = (uint8_t*)workspace;
    auto take = [&p](int64_t bytes) {
        uint8_t* at = p;
        p += round_up(bytes);
        return at;
    };
    uint32_t* counts = (uint32_t*)take(4 * E);
    uint32_t* offsets = (uint32_t*)take(4 * E);
    int32_t* perm = (int32_t*)take(4 * R);
    int32_t* inv = (int32_t*)take(4 * R);
    void* weights = take(2 * R);
    const int64_t experts_bytes = fma_thin_swiglu_experts_workspace_bytes(R, I);
    void* experts = take(experts_bytes);
    void* out = take(2 * R * H);
    int rc;
    if (gemm::thin::takes_one_token(T, top_k)) {
        const char* who = "moe_decode";
        hipStream_t st = (hipStream_t)stream;
        rc = check_router(who, x, gate_weight, T, H, E, top_k, logits, dtype);
        if (!rc) rc = gemm::thin::check(who, x, T, perm, 1, W1, experts, counts, offsets, R, E, 2 * I, H, 1, dtype);
        if (!rc) rc = gemm::thin::check(who, experts, R, nullptr, 1, W2, out, counts, offsets, R, E, H, I, 0, dtype);
        if (rc) return rc;
        FMA_REQUIRE(y, FMA_ERR_NULL_POINTER, "moe_decode: NULL pointer");
        FMA_REQUIRE((reinterpret_cast<uintptr_t>(y) & 1u) == 0, FMA_ERR_MISALIGNED, "moe_decode: y not aligned to the element size");
        const RouterArgs a = router_args(x, gate_weight, T, H, E, top_k, logits);
        rc = dtype == FMA_BF16 ? launch_router_logits<RouterBf16>(a, st) : launch_router_logits<RouterF16>(a, st);
        return rc ? rc : gemm::thin::one_token(x, logits, W1, bias1, W2, bias2, experts, y, E, H, I, top_k, dtype, st);
    }
    rc = fma_router_topk_index(x, gate_weight, T, H, E, top_k, logits, weights, counts, offsets, perm, inv, dtype, stream);
    if (rc) return rc;
    // (a token's choices are distinct: no expert has more than T rows)
    rc = fma_thin_swiglu_experts(x, T, perm, (int32_t)top_k, W1, bias1, W2, bias2, out, counts, offsets, R, T, E, H, I, experts,
                                 experts_bytes, dtype, stream);
    if (rc) return rc;
    return fma_combine(out, inv, weights, T, top_k, H, y, dtype, stream);
}

}  // extern "C"
