// Entry points of the grouped GEMM for launches whose groups differ in one dimension (the kernel: ragged_kernel.h).
#include <algorithm>
#include <type_traits>

#include "ragged_kernel.h"

namespace fmahip {
namespace gemm {
namespace ragged {

// every instantiation the entry points launch (explicit, so that host stub and device code are both emitted)
#define FMA_RAGGED_INSTANTIATE(EL)                                                                          \
    template __global__ void ragged_gemm_kernel<EL, true, true, EPI_PLAIN, false, false, false, false>(const Args);    \
    template __global__ void ragged_gemm_kernel<EL, true, false, EPI_PLAIN, false, false, false, false>(const Args);   \
    template __global__ void ragged_gemm_kernel<EL, false, true, EPI_PLAIN, false, false, false, false>(const Args);   \
    template __global__ void ragged_gemm_kernel<EL, false, false, EPI_PLAIN, false, false, false, false>(const Args);  \
    template __global__ void ragged_gemm_kernel<EL, true, true, EPI_PLAIN, true, false, false, false>(const Args);     \
    template __global__ void ragged_gemm_kernel<EL, true, false, EPI_PLAIN, true, false, false, false>(const Args);    \
    template __global__ void ragged_gemm_kernel<EL, false, true, EPI_PLAIN, true, false, false, false>(const Args);    \
    template __global__ void ragged_gemm_kernel<EL, false, false, EPI_PLAIN, true, false, false, false>(const Args);   \
    template __global__ void ragged_gemm_kernel<EL, true, true, EPI_SWIGLU, false, false, false, false>(const Args);   \
    template __global__ void ragged_gemm_kernel<EL, true, true, EPI_SWIGLU_ACT, false, false, false, false>(const Args); \
    template __global__ void ragged_gemm_kernel<EL, true, true, EPI_PLAIN, false, true, false, false>(const Args);     \
    template __global__ void ragged_gemm_kernel<EL, true, true, EPI_SWIGLU, false, true, false, false>(const Args);    \
    template __global__ void ragged_gemm_kernel<EL, true, true, EPI_SWIGLU_ACT, false, true, false, false>(const Args); \
    template __global__ void ragged_gemm_kernel<EL, true, false, EPI_SWIGLU_BWD, false, false, false, false>(const Args); \
    template __global__ void ragged_gemm_kernel<EL, true, true, EPI_PLAIN, false, false, true, false>(const Args);     \
    template __global__ void ragged_gemm_kernel<EL, true, true, EPI_SWIGLU, false, false, true, false>(const Args);    \
    template __global__ void ragged_gemm_kernel<EL, true, true, EPI_SWIGLU_ACT, false, false, true, false>(const Args); \
    template __global__ void ragged_gemm_kernel<EL, true, true, EPI_PLAIN, false, true, true, false>(const Args);      \
    template __global__ void ragged_gemm_kernel<EL, true, true, EPI_SWIGLU, false, true, true, false>(const Args);     \
    template __global__ void ragged_gemm_kernel<EL, true, true, EPI_SWIGLU_ACT, false, true, true, false>(const Args); \
    template __global__ void ragged_gemm_kernel<EL, false, false, EPI_PLAIN, true, false, true, false>(const Args);    \
    template __global__ void ragged_gemm_kernel<EL, true, true, EPI_SPLIT, false, false, false, false>(const Args);    \
    template __global__ void ragged_gemm_kernel<EL, true, false, EPI_SPLIT, false, false, false, false>(const Args);
FMA_RAGGED_INSTANTIATE(ElemBf16)
FMA_RAGGED_INSTANTIATE(ElemF16)
#undef FMA_RAGGED_INSTANTIATE

template <typename EL, int EPI>
int launch_forward(const Args& args, hipStream_t st) {
    if (args.E <= kTallGroups) return launch_tall(args, EPI, true, std::is_same<EL, ElemBf16>::value, st);
    return launch_forward_as<EL, EPI, false>(args, st);
}

template <typename EL, bool VARY_K>
int launch_plain(const Args& args, bool a_kc, bool b_kc, hipStream_t st) {
    if constexpr (!VARY_K) {
        if (a_kc && args.E <= kTallGroups) return launch_tall(args, EPI_PLAIN, b_kc, std::is_same<EL, ElemBf16>::value, st);
    }
    if (a_kc && b_kc) return launch<EL, true, true, EPI_PLAIN, VARY_K, false, false, false>(args, st);
    if (a_kc && !b_kc) return launch<EL, true, false, EPI_PLAIN, VARY_K, false, false, false>(args, st);
    if (!a_kc && b_kc) return launch<EL, false, true, EPI_PLAIN, VARY_K, false, false, false>(args, st);
    return launch<EL, false, false, EPI_PLAIN, VARY_K, false, false, false>(args, st);
}

// a product with its reduction in args.splits parts: the parts, then their sum
int launch_split(const Args& args, bool b_kc, bool bf16, hipStream_t st) {
    const int rc = args.E <= kTallGroups ? launch_tall(args, EPI_SPLIT, b_kc, bf16, st)
                   : bf16 ? (b_kc ? launch<ElemBf16, true, true, EPI_SPLIT, false, false, false, false>(args, st)
                                  : launch<ElemBf16, true, false, EPI_SPLIT, false, false, false, false>(args, st))
                          : (b_kc ? launch<ElemF16, true, true, EPI_SPLIT, false, false, false, false>(args, st)
                                  : launch<ElemF16, true, false, EPI_SPLIT, false, false, false, false>(args, st));
    return rc != FMA_OK ? rc : launch_split_reduce(args, bf16, st);
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


int64_t fma_grouped_gemm_ragged_split_bytes(int64_t R, int64_t E, int64_t N, int64_t K, int trans_b) {
    const uint32_t parts = fmahip::gemm::ragged::plan_split(R, E, N, K, trans_b != 0, E <= fmahip::gemm::ragged::kTallGroups).splits;
    return parts > 1 ? R * N * 4 * (int64_t)parts : 0;
}

int64_t fma_grouped_gemm_ragged_workspace_bytes(int64_t R, int64_t E, int64_t N, int64_t K, int trans_b) {
    // (enough for either kernel: callers may pad their groups with empty ones past the number that decides between them)
    uint32_t parts = 1;
    for (const bool tall : {false, true})
        parts = std::max(parts, fmahip::gemm::ragged::plan_split(R, E, N, K, trans_b != 0, tall).splits);
    return parts > 1 ? R * N * 4 * (int64_t)parts : 0;
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
        workspace && vary == FMA_VARY_M && a_kc ? ragged::plan_split(rows, E, N, K, b_kc, E <= ragged::kTallGroups) : ragged::SplitPlan{1u, 0u};
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
        return ragged::launch_split(args, b_kc, dtype == FMA_BF16, st);
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
    if (args.E <= ragged::kTallGroups) return ragged::launch_tall(args, EPI_SWIGLU_BWD, false, dtype == FMA_BF16, st);
    return dtype == FMA_BF16 ? ragged::launch<ElemBf16, true, false, EPI_SWIGLU_BWD, false, false, false, false>(args, st)
                             : ragged::launch<ElemF16, true, false, EPI_SWIGLU_BWD, false, false, false, false>(args, st);
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
    return dtype == FMA_BF16 ? ragged::launch<ElemBf16, false, false, EPI_PLAIN, true, false, true, false>(args, st)
                             : ragged::launch<ElemF16, false, false, EPI_PLAIN, true, false, true, false>(args, st);
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
