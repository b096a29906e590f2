// Entry points of the grouped GEMM for launches whose groups differ in one dimension (the kernel: ragged_kernel.h), and the
// choice and the second pass of a split reduction.
#include <algorithm>
#include <cmath>

#include "ragged_kernel.h"

namespace fmahip {
namespace gemm {
namespace ragged {

// every instantiation the entry points launch (explicit, so that host stub and device code are both emitted)
#define FMA_RAGGED_INSTANTIATE(EL)                                                                          \
    template __global__ void ragged_gemm_kernel<EL, true, true, EPI_PLAIN, false, false, false>(const Args);    \
    template __global__ void ragged_gemm_kernel<EL, true, false, EPI_PLAIN, false, false, false>(const Args);   \
    template __global__ void ragged_gemm_kernel<EL, false, true, EPI_PLAIN, false, false, false>(const Args);   \
    template __global__ void ragged_gemm_kernel<EL, false, false, EPI_PLAIN, false, false, false>(const Args);  \
    template __global__ void ragged_gemm_kernel<EL, true, true, EPI_PLAIN, true, false, false>(const Args);     \
    template __global__ void ragged_gemm_kernel<EL, true, false, EPI_PLAIN, true, false, false>(const Args);    \
    template __global__ void ragged_gemm_kernel<EL, false, true, EPI_PLAIN, true, false, false>(const Args);    \
    template __global__ void ragged_gemm_kernel<EL, false, false, EPI_PLAIN, true, false, false>(const Args);   \
    template __global__ void ragged_gemm_kernel<EL, true, true, EPI_SWIGLU, false, false, false>(const Args);   \
    template __global__ void ragged_gemm_kernel<EL, true, true, EPI_SWIGLU_ACT, false, false, false>(const Args); \
    template __global__ void ragged_gemm_kernel<EL, true, true, EPI_PLAIN, false, true, false>(const Args);     \
    template __global__ void ragged_gemm_kernel<EL, true, true, EPI_SWIGLU, false, true, false>(const Args);    \
    template __global__ void ragged_gemm_kernel<EL, true, true, EPI_SWIGLU_ACT, false, true, false>(const Args); \
    template __global__ void ragged_gemm_kernel<EL, true, false, EPI_SWIGLU_BWD, false, false, false>(const Args); \
    template __global__ void ragged_gemm_kernel<EL, true, true, EPI_PLAIN, false, false, true>(const Args);     \
    template __global__ void ragged_gemm_kernel<EL, true, true, EPI_SWIGLU, false, false, true>(const Args);    \
    template __global__ void ragged_gemm_kernel<EL, true, true, EPI_SWIGLU_ACT, false, false, true>(const Args); \
    template __global__ void ragged_gemm_kernel<EL, true, true, EPI_PLAIN, false, true, true>(const Args);      \
    template __global__ void ragged_gemm_kernel<EL, true, true, EPI_SWIGLU, false, true, true>(const Args);     \
    template __global__ void ragged_gemm_kernel<EL, true, true, EPI_SWIGLU_ACT, false, true, true>(const Args); \
    template __global__ void ragged_gemm_kernel<EL, false, false, EPI_PLAIN, true, false, true>(const Args);    \
    template __global__ void ragged_gemm_kernel<EL, true, true, EPI_SPLIT, false, false, false>(const Args);    \
    template __global__ void ragged_gemm_kernel<EL, true, false, EPI_SPLIT, false, false, false>(const Args);
FMA_RAGGED_INSTANTIATE(ElemBf16)
FMA_RAGGED_INSTANTIATE(ElemF16)
#undef FMA_RAGGED_INSTANTIATE

template <typename EL, bool A_KC, bool B_KC, int EPI, bool VARY_K, bool BIAS = false, bool GATHER = false>
int launch(const Args& args, hipStream_t st) {
    int cus = num_compute_units();
    if (cus <= 0) cus = 256;
    hipLaunchKernelGGL((ragged_gemm_kernel<EL, A_KC, B_KC, EPI, VARY_K, BIAS, GATHER>), dim3((uint32_t)cus), dim3(NT), 0, st,
                       args);
    return launch_status("grouped_gemm_ragged");
}

// the forward (NT) kernels by epilogue, bias and gather
template <typename EL, int EPI>
int launch_forward(const Args& args, hipStream_t st) {
    const bool bias = args.bias != nullptr, gather = args.row_index != nullptr;
    if (bias && gather) return launch<EL, true, true, EPI, false, true, true>(args, st);
    if (bias) return launch<EL, true, true, EPI, false, true, false>(args, st);
    if (gather) return launch<EL, true, true, EPI, false, false, true>(args, st);
    return launch<EL, true, true, EPI, false, false, false>(args, st);
}

template <typename EL, bool VARY_K>
int launch_plain(const Args& args, bool a_kc, bool b_kc, hipStream_t st) {
    if (a_kc && b_kc) return launch<EL, true, true, EPI_PLAIN, VARY_K>(args, st);
    if (a_kc && !b_kc) return launch<EL, true, false, EPI_PLAIN, VARY_K>(args, st);
    if (!a_kc && b_kc) return launch<EL, false, true, EPI_PLAIN, VARY_K>(args, st);
    return launch<EL, false, false, EPI_PLAIN, VARY_K>(args, st);
}

// ---- split reduction ---------------------------------------------------------------------------------------------
// A launch with fewer tiles than compute units leaves the others idle for the whole reduction: the second projection of
// 1021 tokens on 8 experts (2048 x 8192) is 96 tiles of 128 K steps, 205 us. With the reduction in two parts (192 tiles of
// 64 steps, fp32 sums to memory and one pass over them) it takes 130 us. More of the same (parts; before -> now):
//   NT 2048 x 8192, 8 groups of 64 / 128 rows (4)            167 -> 69 us, 180 -> 84 us
//   NT 4096 x 14336, 8 groups of 128 / 512 rows (2 / 3)      357 -> 234 us, 690 -> 570 us
//   NN 2048 x 16384, 8 groups of 128 / 512 / 1024 rows       339 -> 133 us (4), 380 -> 317 us (3), 700 -> 580 us (3)
//   NN 4096 x 28672, 8 groups of 32 / 64 / 512 rows          496 -> 310 us (2), 633 -> 371 us (2), 1330 -> 1015 us (4)
//
// How many parts: the number with the least predicted time, rounds of tiles times (K steps + a tile's fixed cost) or the
// weights at the rate they stream, plus the traffic of the sums. The row counts lie in device memory, so the number of tiles
// is the expected one for evenly loaded groups. Parts have at least kSplitMinSteps steps, the sums at most kSplitMaxBytes (they
// stay in the last-level cache), and a split has to promise a tenth less than none. Groups of few rows run the three-stage
// loop, whose steps are shorter, without a split on half-width tiles in the NT layout: NT 4096 x 14336 on 8 groups of 32 rows
// streams its weights in 176 us as it is and would take 184 us in two parts.
// Uneven loads make fewer tiles, which a split helps the more; where they happen to fill the compute units exactly once as they are, the
// sums are the price. Training steps without -> with splits: 2048 tokens, hidden 4096, I 14336, E 8, k 2, evenly 5100 -> 4630 us, all
// on two experts 3870 -> 3990 us; 4000 tokens, hidden 2048, I 8192: 2775 -> 2627 and 2157 -> 2225 us; 512 and 1021 tokens gain either way
// (2219 -> 1779 and 2727 -> 2478 us, 886 -> 565 us at 256 tokens of the second shape).
constexpr double kStepUs = 1.45, kThinStepUs[2] = {1.1, 0.75}, kTileSteps = 6.0, kThinRows = 48.0, kWeightBytesPerUs = 5.5e6;
constexpr double kReduceUs = 4.0, kReduceBytesPerUs = 4.5e6, kSplitGain = 0.9;
constexpr uint32_t kSplitMinSteps = 24;
constexpr int64_t kSplitMaxBytes = 256ll << 20;
struct SplitPlan {
    uint32_t splits, steps;  // parts and K steps of each (even; the last part takes what is left); splits 1: no split
};
SplitPlan plan_split(int64_t R, int64_t E, int64_t N, int64_t K, bool b_kc) {
    const uint32_t all = (uint32_t)((K + BK - 1) / BK);
    SplitPlan best{1u, all};
    // (the sizes for which every tile takes the matrix-instruction path)
    if (R < 1 || E < 1 || N < 8 || N % 8 || N >= (1 << 23) || K % 8 || K >= (1 << 21) || R > 0x7fffffffll) return best;
    if (all < 2 * kSplitMinSteps) return best;
    const int cus = num_compute_units() > 0 ? num_compute_units() : 256;
    const double active = (double)(R < E ? R : E), mean = (double)R / active;
    const double row_tiles = active * (mean < BM / 2 ? 1.0 : mean / BM + 0.5);
    const double tiles = row_tiles * (double)((N + BN - 1) / BN);
    const bool thin = mean <= kThinRows, narrow = thin && b_kc && 2.0 * tiles <= cus;
    const double step_us = thin ? kThinStepUs[b_kc] : kStepUs;
    const double weights_us = active * N * K * 2.0 / kWeightBytesPerUs;
    auto us = [&](uint32_t parts, uint32_t steps) {
        const double units = tiles * parts * (parts == 1 && narrow ? 2.0 : 1.0);
        const double products = std::ceil(units / cus - 1e-9) * (steps + kTileSteps) * step_us;
        const double sums = parts > 1 ? kReduceUs + (double)R * N * (8.0 * parts + 2.0) / kReduceBytesPerUs : 0.0;
        return std::max(products, weights_us) + sums;
    };
    double best_us = us(1, all) * kSplitGain;
    for (uint32_t parts = 2; parts * kSplitMinSteps <= all && parts <= 32; ++parts) {
        const uint32_t steps = ((all + parts - 1) / parts + 1u) & ~1u;
        const uint32_t used = (all + steps - 1) / steps;
        if (used != parts || R * N * 4 * (int64_t)parts > kSplitMaxBytes) continue;
        const double t = us(parts, steps);
        if (t < best_us) {
            best_us = t;
            best = SplitPlan{parts, steps};
        }
    }
    return best;
}

// out[r, :] = round(alpha * (sum over the parts, in order)), plus the bias of the row's group as the kernels' epilogue adds it.
// Bound by memory (parts * 4 + 2 bytes per element). A workgroup takes kReduceRows rows; which group a row belongs to is
// read off a prefix of the sizes (built per workgroup: E values, one scan), and rows past the last group are left alone.
constexpr int kReduceThreads = 256, kReduceRows = 4;
template <typename EL, bool BIAS>
__global__ __launch_bounds__(kReduceThreads) void split_reduce_kernel(const Args args) {
    __shared__ uint32_t s_end[FMA_MAX_GROUPS];
    const uint32_t tid = threadIdx.x, E = args.E, N = args.n;
    if (tid < 64u) {
        uint32_t carry = 0;
        for (uint32_t base = 0; base < E; base += 64u) {
            const uint32_t e = base + tid;
            const uint32_t incl = wave_inclusive_scan<uint32_t>(e < E ? args.sizes[e] : 0u);
            if (e < E) s_end[e] = carry + incl;
            carry += __shfl(incl, 63, 64);
        }
    }
    __syncthreads();
    const uint32_t vecs = N / 8u;  // of 8 columns
    const uint64_t part = (uint64_t)args.rows * N;
    const uint32_t first = blockIdx.x * (uint32_t)kReduceRows;
    for (uint32_t i = tid; i < (uint32_t)kReduceRows * vecs; i += kReduceThreads) {
        const uint32_t r = first + i / vecs, col = (i % vecs) * 8u;
        if (r >= args.rows || r >= s_end[E - 1u]) return;
        const float* src = args.partial + (uint64_t)r * N + col;
        float sum[8];
#pragma unroll
        for (int x = 0; x < 8; ++x) sum[x] = 0.0f;
        for (uint32_t s = 0; s < args.splits; ++s, src += part) {
            const float4 lo = reinterpret_cast<const float4*>(src)[0], hi = reinterpret_cast<const float4*>(src)[1];
            sum[0] += lo.x; sum[1] += lo.y; sum[2] += lo.z; sum[3] += lo.w;
            sum[4] += hi.x; sum[5] += hi.y; sum[6] += hi.z; sum[7] += hi.w;
        }
#pragma unroll
        for (int x = 0; x < 8; ++x) sum[x] *= args.alpha;
        if constexpr (BIAS) {
            uint32_t lo = 0, hi = E - 1u;  // the first group that ends past row r
            while (lo < hi) {
                const uint32_t mid = (lo + hi) >> 1;
                if (s_end[mid] > r) hi = mid;
                else lo = mid + 1u;
            }
            const uint16_t* b = args.bias + (uint64_t)lo * N + col;
#pragma unroll
            for (int x = 0; x < 8; ++x) sum[x] = EL::round(sum[x]) + EL::from_bits(b[x]);
        }
        uint4 packed;
        packed.x = EL::pack2(sum[0], sum[1]);
        packed.y = EL::pack2(sum[2], sum[3]);
        packed.z = EL::pack2(sum[4], sum[5]);
        packed.w = EL::pack2(sum[6], sum[7]);
        *reinterpret_cast<uint4*>(args.D + (uint64_t)r * N + col) = packed;
    }
}

template <typename EL>
int launch_split(const Args& args, bool b_kc, hipStream_t st) {
    const int rc = b_kc ? launch<EL, true, true, EPI_SPLIT, false>(args, st) : launch<EL, true, false, EPI_SPLIT, false>(args, st);
    if (rc != FMA_OK) return rc;
    const dim3 grid((args.rows + kReduceRows - 1) / kReduceRows), block(kReduceThreads);
    if (args.bias) hipLaunchKernelGGL((split_reduce_kernel<EL, true>), grid, block, 0, st, args);
    else hipLaunchKernelGGL((split_reduce_kernel<EL, false>), grid, block, 0, st, args);
    return launch_status("grouped_gemm_ragged(reduce)");
}

// The forward product of an expert projection, out_e = x_e W_e^T (+ bias_e), with the rows of x_e packed (row_index
// NULL) or picked through row_index; swiglu: N = 2 I, out is the pre-activation (may be NULL) and act its activation.
// taken, pass_bits: see Args.
int up_projection(const char* who, const void* x, int64_t x_rows, const int32_t* row_index, int32_t divisor, const void* W,
                  const void* bias, void* out, void* act, const uint32_t* M_arr, int64_t E, int64_t N, int64_t K, int swiglu,
                  int dtype, hipStream_t st, uint32_t* taken = nullptr, uint32_t pass_bits = 0) {
    FMA_REQUIRE(dtype == FMA_BF16 || dtype == FMA_F16, dtype_bytes(dtype) ? FMA_ERR_UNSUPPORTED : FMA_ERR_BAD_DTYPE,
                "%s: bf16 and fp16 operands are implemented (dtype code %d)", who, dtype);
    FMA_REQUIRE(E >= 0, FMA_ERR_BAD_SIZE, "%s: negative group count %lld", who, (long long)E);
    FMA_REQUIRE(E <= FMA_MAX_GROUPS, FMA_ERR_TOO_MANY_EXPERTS, "%s: E=%lld exceeds the limit %d", who, (long long)E,
                FMA_MAX_GROUPS);
    // the upper bounds are those of the kernel's 32-bit tile offsets; these entry points have no scalar path beyond them
    if (swiglu) {
        FMA_REQUIRE(N >= 16 && N % 16 == 0 && N < (1ll << 23), FMA_ERR_BAD_SIZE,
                    "%s: intermediate size %lld must be a positive multiple of 8 below 2^22", who, (long long)(N / 2));
    } else {
        FMA_REQUIRE(N >= 8 && N % 8 == 0 && N < (1ll << 23), FMA_ERR_BAD_SIZE,
                    "%s: N=%lld must be a positive multiple of 8 below 2^23", who, (long long)N);
    }
    FMA_REQUIRE(K >= 8 && K % 8 == 0 && K < (1ll << 21), FMA_ERR_BAD_SIZE,
                "%s: K=%lld must be a positive multiple of 8 below 2^21", who, (long long)K);
    if (E == 0) return FMA_OK;
    FMA_REQUIRE(x && W && M_arr && (swiglu ? act != nullptr : out != nullptr), FMA_ERR_NULL_POINTER, "%s: NULL pointer", who);
    FMA_REQUIRE(aligned16(x) && aligned16(W) && aligned16(act) && aligned16(out), FMA_ERR_MISALIGNED,
                "%s: x, W and the outputs must be 16-byte aligned", who);
    FMA_REQUIRE((reinterpret_cast<uintptr_t>(bias) & 3u) == 0 && (reinterpret_cast<uintptr_t>(row_index) & 3u) == 0,
                FMA_ERR_MISALIGNED, "%s: bias and row_index must be 4-byte aligned", who);
    Args args{};
    args.A = (const uint16_t*)x;
    args.B = (const uint16_t*)W;
    args.D = (uint16_t*)out;
    args.ACT = swiglu ? (uint16_t*)act : nullptr;
    args.sizes = M_arr;
    args.bias = (const uint16_t*)bias;
    args.row_index = row_index;
    args.divisor = (uint32_t)divisor;
    args.a_rows = (uint32_t)x_rows;
    args.E = (uint32_t)E;
    args.m = 0;
    args.n = (uint32_t)N;
    args.k = (uint32_t)K;
    args.alpha = 1.0f;
    args.taken = taken;
    args.pass_bits = pass_bits;
    // whether the pre-activation is stored is a compile-time property of the kernel: the epilogue is then one
    // straight-line block
    if (!swiglu) return dtype == FMA_BF16 ? launch_forward<ElemBf16, EPI_PLAIN>(args, st) : launch_forward<ElemF16, EPI_PLAIN>(args, st);
    if (out) return dtype == FMA_BF16 ? launch_forward<ElemBf16, EPI_SWIGLU>(args, st) : launch_forward<ElemF16, EPI_SWIGLU>(args, st);
    return dtype == FMA_BF16 ? launch_forward<ElemBf16, EPI_SWIGLU_ACT>(args, st) : launch_forward<ElemF16, EPI_SWIGLU_ACT>(args, st);
}

}  // namespace ragged

// fma_grouped_gemm's launch (per-group M, N and K arrays in device memory) offered to the two kernels of this file: each
// reads the arrays and runs only if the launch has its form (one varying dimension), otherwise it ends at once.
int launch_ragged_from_arrays(const void* A, const void* B, void* D, const uint32_t* M_arr, const uint32_t* N_arr,
                              const uint32_t* K_arr, int64_t E, bool a_kc, bool b_kc, float alpha, int dtype, hipStream_t st) {
    ragged::Args args{};
    args.A = (const uint16_t*)A;
    args.B = (const uint16_t*)B;
    args.D = (uint16_t*)D;
    args.E = (uint32_t)E;
    args.alpha = alpha;
    args.m_dev = M_arr;
    args.n_dev = N_arr;
    args.k_dev = K_arr;
    args.sizes = M_arr;
    int rc = dtype == FMA_BF16 ? ragged::launch_plain<ElemBf16, false>(args, a_kc, b_kc, st)
                               : ragged::launch_plain<ElemF16, false>(args, a_kc, b_kc, st);
    if (rc != FMA_OK) return rc;
    args.sizes = K_arr;
    return dtype == FMA_BF16 ? ragged::launch_plain<ElemBf16, true>(args, a_kc, b_kc, st)
                             : ragged::launch_plain<ElemF16, true>(args, a_kc, b_kc, st);
}

}  // namespace gemm
}  // namespace fmahip

extern "C" {


int64_t fma_grouped_gemm_ragged_workspace_bytes(int64_t R, int64_t E, int64_t N, int64_t K, int trans_b) {
    const fmahip::gemm::ragged::SplitPlan plan = fmahip::gemm::ragged::plan_split(R, E, N, K, trans_b != 0);
    return plan.splits > 1 ? R * N * 4 * (int64_t)plan.splits : 0;
}

int fma_grouped_gemm_ragged(const void* A, const void* B, void* D, const uint32_t* sizes, const void* bias, int64_t E,
                            int vary, int64_t M, int64_t N, int64_t K, int trans_a, int trans_b, float alpha, int dtype,
                            void* stream) {
    return fma_grouped_gemm_ragged_split(A, B, D, sizes, bias, E, vary, M, N, K, trans_a, trans_b, alpha, 0, nullptr, 0, dtype,
                                         stream);
}

int fma_grouped_gemm_ragged_split(const void* A, const void* B, void* D, const uint32_t* sizes, const void* bias, int64_t E,
                                  int vary, int64_t M, int64_t N, int64_t K, int trans_a, int trans_b, float alpha,
                                  int64_t rows, void* workspace, int64_t workspace_bytes, int dtype, void* stream) {
    using namespace fmahip;
    using namespace fmahip::gemm;
    FMA_REQUIRE(dtype == FMA_BF16 || dtype == FMA_F16, dtype_bytes(dtype) ? FMA_ERR_UNSUPPORTED : FMA_ERR_BAD_DTYPE,
                "grouped_gemm_ragged: bf16 and fp16 operands are implemented (dtype code %d)", dtype);
    FMA_REQUIRE(vary == FMA_VARY_M || vary == FMA_VARY_K, FMA_ERR_BAD_SIZE,
                "grouped_gemm_ragged: vary must be FMA_VARY_M or FMA_VARY_K (got %d)", vary);
    FMA_REQUIRE(E >= 0, FMA_ERR_BAD_SIZE, "grouped_gemm_ragged: negative group count %lld", (long long)E);
    FMA_REQUIRE(E <= FMA_MAX_GROUPS, FMA_ERR_TOO_MANY_EXPERTS, "grouped_gemm_ragged: E=%lld exceeds the limit %d",
                (long long)E, FMA_MAX_GROUPS);
    if (vary == FMA_VARY_M) M = 0;
    else K = 0;
    FMA_REQUIRE(M >= 0 && N >= 0 && K >= 0 && M <= 0xffffffffll && N <= 0xffffffffll && K <= 0xffffffffll, FMA_ERR_BAD_SIZE,
                "grouped_gemm_ragged: dimensions must lie in [0, 2^32) (M=%lld N=%lld K=%lld)", (long long)M, (long long)N,
                (long long)K);
    if (E == 0) return FMA_OK;
    FMA_REQUIRE(A && B && D && sizes, FMA_ERR_NULL_POINTER, "grouped_gemm_ragged: NULL pointer");
    FMA_REQUIRE(aligned16(A) && aligned16(B) && aligned16(D), FMA_ERR_MISALIGNED,
                "grouped_gemm_ragged: A, B and D must be 16-byte aligned");
    hipStream_t st = (hipStream_t)stream;
    const bool a_kc = trans_a == 0;  // A stored [M, K]: reduction dim contiguous
    const bool b_kc = trans_b != 0;  // B stored [N, K]: reduction dim contiguous
    FMA_REQUIRE(!bias || (vary == FMA_VARY_M && a_kc && b_kc && alpha == 1.0f), FMA_ERR_UNSUPPORTED,
                "grouped_gemm_ragged: a bias is added in the forward form only (rows vary, A not transposed, B transposed, "
                "alpha 1)");
    // (with these sizes every tile takes the matrix-instruction path, the only one that adds the bias)
    FMA_REQUIRE(!bias || (N % 8 == 0 && K % 8 == 0 && N < (1 << 23) && K < (1 << 21)), FMA_ERR_UNSUPPORTED,
                "grouped_gemm_ragged: with a bias, N and K must be multiples of 8, N < 2^23 and K < 2^21");
    FMA_REQUIRE(!bias || (reinterpret_cast<uintptr_t>(bias) & 3u) == 0, FMA_ERR_MISALIGNED,
                "grouped_gemm_ragged: the bias must be 4-byte aligned");
    ragged::Args args{};
    args.A = (const uint16_t*)A;
    args.B = (const uint16_t*)B;
    args.D = (uint16_t*)D;
    args.ACT = nullptr;
    args.sizes = sizes;
    args.bias = (const uint16_t*)bias;
    args.E = (uint32_t)E;
    args.m = (uint32_t)M;
    args.n = (uint32_t)N;
    args.k = (uint32_t)K;
    args.alpha = alpha;
    const ragged::SplitPlan plan =
        workspace && vary == FMA_VARY_M && a_kc ? ragged::plan_split(rows, E, N, K, b_kc) : ragged::SplitPlan{1u, 0u};
    if (plan.splits > 1) {
        FMA_REQUIRE(aligned16(workspace), FMA_ERR_MISALIGNED, "grouped_gemm_ragged: the workspace must be 16-byte aligned");
        const int64_t need = rows * N * 4 * (int64_t)plan.splits;
        FMA_REQUIRE(workspace_bytes >= need, FMA_ERR_WORKSPACE_TOO_SMALL,
                    "grouped_gemm_ragged: workspace of %lld bytes is smaller than the %lld needed", (long long)workspace_bytes,
                    (long long)need);
        args.partial = (float*)workspace;
        args.splits = plan.splits;
        args.split_steps = plan.steps;
        args.rows = (uint32_t)rows;
        return dtype == FMA_BF16 ? ragged::launch_split<ElemBf16>(args, b_kc, st) : ragged::launch_split<ElemF16>(args, b_kc, st);
    }
    if (bias)
        return dtype == FMA_BF16 ? ragged::launch_forward<ElemBf16, EPI_PLAIN>(args, st)
                                 : ragged::launch_forward<ElemF16, EPI_PLAIN>(args, st);
    if (vary == FMA_VARY_K)
        return dtype == FMA_BF16 ? ragged::launch_plain<ElemBf16, true>(args, a_kc, b_kc, st)
                                 : ragged::launch_plain<ElemF16, true>(args, a_kc, b_kc, st);
    return dtype == FMA_BF16 ? ragged::launch_plain<ElemBf16, false>(args, a_kc, b_kc, st)
                             : ragged::launch_plain<ElemF16, false>(args, a_kc, b_kc, st);
}

int fma_grouped_gemm_swiglu(const void* x, const void* W, const void* bias, void* h, void* act, const uint32_t* M_arr,
                            int64_t E, int64_t I, int64_t K, int dtype, void* stream) {
    return fmahip::gemm::ragged::up_projection("grouped_gemm_swiglu", x, 0, nullptr, 1, W, bias, h, act, M_arr, E, 2 * I, K,
                                               1, dtype, (hipStream_t)stream);
}

int fma_grouped_gemm_swiglu_bwd(const void* dy, const void* W, const void* h, void* dh, const uint32_t* M_arr, int64_t E,
                                int64_t I, int64_t K, int dtype, void* stream) {
    using namespace fmahip;
    using namespace fmahip::gemm;
    FMA_REQUIRE(dtype == FMA_BF16 || dtype == FMA_F16, dtype_bytes(dtype) ? FMA_ERR_UNSUPPORTED : FMA_ERR_BAD_DTYPE,
                "grouped_gemm_swiglu_bwd: bf16 and fp16 operands are implemented (dtype code %d)", dtype);
    FMA_REQUIRE(E >= 0, FMA_ERR_BAD_SIZE, "grouped_gemm_swiglu_bwd: negative group count %lld", (long long)E);
    FMA_REQUIRE(E <= FMA_MAX_GROUPS, FMA_ERR_TOO_MANY_EXPERTS, "grouped_gemm_swiglu_bwd: E=%lld exceeds the limit %d",
                (long long)E, FMA_MAX_GROUPS);
    // (with these sizes every tile takes the matrix-instruction path, the only one with this epilogue)
    FMA_REQUIRE(I >= 8 && I % 8 == 0 && I < (1ll << 22), FMA_ERR_BAD_SIZE,
                "grouped_gemm_swiglu_bwd: intermediate size %lld must be a positive multiple of 8 below 2^22", (long long)I);
    FMA_REQUIRE(K >= 8 && K % 8 == 0 && K < (1ll << 21), FMA_ERR_BAD_SIZE,
                "grouped_gemm_swiglu_bwd: K=%lld must be a positive multiple of 8 below 2^21", (long long)K);
    if (E == 0) return FMA_OK;
    FMA_REQUIRE(dy && W && h && dh && M_arr, FMA_ERR_NULL_POINTER, "grouped_gemm_swiglu_bwd: NULL pointer");
    FMA_REQUIRE(aligned16(dy) && aligned16(W) && aligned16(h) && aligned16(dh), FMA_ERR_MISALIGNED,
                "grouped_gemm_swiglu_bwd: dy, W, h and dh must be 16-byte aligned");
    ragged::Args args{};
    args.A = (const uint16_t*)dy;
    args.B = (const uint16_t*)W;
    args.D = (uint16_t*)dh;
    args.h_in = (const uint16_t*)h;
    args.sizes = M_arr;
    args.E = (uint32_t)E;
    args.m = 0;
    args.n = (uint32_t)I;
    args.k = (uint32_t)K;
    args.alpha = 1.0f;
    hipStream_t st = (hipStream_t)stream;
    return dtype == FMA_BF16 ? ragged::launch<ElemBf16, true, false, EPI_SWIGLU_BWD, false>(args, st)
                             : ragged::launch<ElemF16, true, false, EPI_SWIGLU_BWD, false>(args, st);
}

int fma_grouped_gemm_gathered_wgrad(const void* dy, const void* x, int64_t x_rows, const int32_t* row_index, int32_t divisor,
                                    void* dW, const uint32_t* K_arr, int64_t E, int64_t M, int64_t N, float alpha, int dtype,
                                    void* stream) {
    using namespace fmahip;
    using namespace fmahip::gemm;
    const char* who = "grouped_gemm_gathered_wgrad";
    FMA_REQUIRE(dtype == FMA_BF16 || dtype == FMA_F16, dtype_bytes(dtype) ? FMA_ERR_UNSUPPORTED : FMA_ERR_BAD_DTYPE,
                "%s: bf16 and fp16 operands are implemented (dtype code %d)", who, dtype);
    FMA_REQUIRE(E >= 0, FMA_ERR_BAD_SIZE, "%s: negative group count %lld", who, (long long)E);
    FMA_REQUIRE(E <= FMA_MAX_GROUPS, FMA_ERR_TOO_MANY_EXPERTS, "%s: E=%lld exceeds the limit %d", who, (long long)E,
                FMA_MAX_GROUPS);
    // (with these sizes every tile takes the matrix-instruction path, the only one that gathers)
    FMA_REQUIRE(M >= 8 && M % 8 == 0 && M < (1ll << 23) && N >= 8 && N % 8 == 0 && N < (1ll << 23), FMA_ERR_BAD_SIZE,
                "%s: M=%lld and N=%lld must be positive multiples of 8 below 2^23", who, (long long)M, (long long)N);
    FMA_REQUIRE(divisor >= 1 && divisor <= 65536, FMA_ERR_BAD_SIZE, "%s: divisor must lie in [1, 65536] (got %d)", who, divisor);
    if (E == 0) return FMA_OK;
    FMA_REQUIRE(dy && x && row_index && dW && K_arr, FMA_ERR_NULL_POINTER, "%s: NULL pointer", who);
    FMA_REQUIRE(x_rows >= 1, FMA_ERR_BAD_SIZE, "%s: x has no rows (%lld)", who, (long long)x_rows);
    // the loads address x with 32-bit byte offsets below 2^31
    FMA_REQUIRE(x_rows <= ((1ll << 31) - 1) / (2 * N), FMA_ERR_UNSUPPORTED,
                "%s: x must be smaller than 2 GiB (%lld rows of %lld elements)", who, (long long)x_rows, (long long)N);
    FMA_REQUIRE(aligned16(dy) && aligned16(x) && aligned16(dW), FMA_ERR_MISALIGNED, "%s: dy, x and dW must be 16-byte aligned", who);
    FMA_REQUIRE((reinterpret_cast<uintptr_t>(row_index) & 3u) == 0, FMA_ERR_MISALIGNED, "%s: row_index must be 4-byte aligned", who);
    ragged::Args args{};
    args.A = (const uint16_t*)dy;
    args.B = (const uint16_t*)x;
    args.D = (uint16_t*)dW;
    args.sizes = K_arr;
    args.row_index = row_index;
    args.divisor = (uint32_t)divisor;
    args.a_rows = (uint32_t)x_rows;
    args.E = (uint32_t)E;
    args.m = (uint32_t)M;
    args.n = (uint32_t)N;
    args.k = 0;
    args.alpha = alpha;
    hipStream_t st = (hipStream_t)stream;
    return dtype == FMA_BF16 ? ragged::launch<ElemBf16, false, false, EPI_PLAIN, true, false, true>(args, st)
                             : ragged::launch<ElemF16, false, false, EPI_PLAIN, true, false, true>(args, st);
}

int fma_grouped_gemm_gathered(const void* x, int64_t x_rows, const int32_t* row_index, int32_t divisor, const void* W,
                              const void* bias, void* out, void* act, const uint32_t* M_arr, int64_t E, int64_t N,
                              int64_t K, int swiglu, int dtype, void* stream) {
    using namespace fmahip;
    FMA_REQUIRE(row_index != nullptr || E == 0, FMA_ERR_NULL_POINTER, "grouped_gemm_gathered: row_index is NULL");
    FMA_REQUIRE(divisor >= 1 && divisor <= 65536, FMA_ERR_BAD_SIZE,
                "grouped_gemm_gathered: divisor must lie in [1, 65536] (got %d)", divisor);
    FMA_REQUIRE(x_rows >= 1 || E == 0, FMA_ERR_BAD_SIZE, "grouped_gemm_gathered: x has no rows (%lld)", (long long)x_rows);
    // the loads address x with 32-bit byte offsets below 2^31
    FMA_REQUIRE(K <= 0 || x_rows <= ((1ll << 31) - 1) / (2 * K), FMA_ERR_UNSUPPORTED,
                "grouped_gemm_gathered: x must be smaller than 2 GiB (%lld rows of %lld elements)", (long long)x_rows,
                (long long)K);
    return gemm::ragged::up_projection("grouped_gemm_gathered", x, x_rows, row_index, divisor, W, bias, out, act, M_arr, E,
                                       N, K, swiglu, dtype, (hipStream_t)stream);
}

}  // extern "C"
