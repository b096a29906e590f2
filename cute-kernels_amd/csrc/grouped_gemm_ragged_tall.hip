// The tall kernels of the grouped GEMM for launches whose groups differ in one dimension (ragged_kernel.h), in a source of their own
// so that they are compiled beside the others.
#include "ragged_kernel.h"

namespace fmahip {
namespace gemm {
namespace ragged {

// every instantiation the entry points launch (explicit, so that host stub and device code are both emitted)
#define FMA_RAGGED_INSTANTIATE(EL)                                                                          \
    template __global__ void ragged_gemm_kernel<EL, true, true, EPI_PLAIN, false, false, false, true>(const Args);    \
    template __global__ void ragged_gemm_kernel<EL, true, false, EPI_PLAIN, false, false, false, true>(const Args);   \
    template __global__ void ragged_gemm_kernel<EL, true, true, EPI_SWIGLU, false, false, false, true>(const Args);   \
    template __global__ void ragged_gemm_kernel<EL, true, true, EPI_SWIGLU_ACT, false, false, false, true>(const Args); \
    template __global__ void ragged_gemm_kernel<EL, true, true, EPI_PLAIN, false, true, false, true>(const Args);     \
    template __global__ void ragged_gemm_kernel<EL, true, true, EPI_SWIGLU, false, true, false, true>(const Args);    \
    template __global__ void ragged_gemm_kernel<EL, true, true, EPI_SWIGLU_ACT, false, true, false, true>(const Args); \
    template __global__ void ragged_gemm_kernel<EL, true, false, EPI_SWIGLU_BWD, false, false, false, true>(const Args); \
    template __global__ void ragged_gemm_kernel<EL, true, true, EPI_PLAIN, false, false, true, true>(const Args);     \
    template __global__ void ragged_gemm_kernel<EL, true, true, EPI_SWIGLU, false, false, true, true>(const Args);    \
    template __global__ void ragged_gemm_kernel<EL, true, true, EPI_SWIGLU_ACT, false, false, true, true>(const Args); \
    template __global__ void ragged_gemm_kernel<EL, true, true, EPI_PLAIN, false, true, true, true>(const Args);      \
    template __global__ void ragged_gemm_kernel<EL, true, true, EPI_SWIGLU, false, true, true, true>(const Args);     \
    template __global__ void ragged_gemm_kernel<EL, true, true, EPI_SWIGLU_ACT, false, true, true, true>(const Args); \
    template __global__ void ragged_gemm_kernel<EL, true, true, EPI_SPLIT, false, false, false, true>(const Args);    \
    template __global__ void ragged_gemm_kernel<EL, true, false, EPI_SPLIT, false, false, false, true>(const Args);
FMA_RAGGED_INSTANTIATE(ElemBf16)
FMA_RAGGED_INSTANTIATE(ElemF16)
#undef FMA_RAGGED_INSTANTIATE

namespace {

template <typename EL>
int launch_as(const Args& args, int epi, bool b_kc, hipStream_t st) {
    if (!b_kc) {
        if (epi == EPI_SWIGLU_BWD) return launch<EL, true, false, EPI_SWIGLU_BWD, false, false, false, true>(args, st);
        if (epi == EPI_SPLIT) return launch<EL, true, false, EPI_SPLIT, false, false, false, true>(args, st);
        return launch<EL, true, false, EPI_PLAIN, false, false, false, true>(args, st);
    }
    if (epi == EPI_SPLIT) return launch<EL, true, true, EPI_SPLIT, false, false, false, true>(args, st);
    if (epi == EPI_SWIGLU) return launch_forward_as<EL, EPI_SWIGLU, true>(args, st);
    if (epi == EPI_SWIGLU_ACT) return launch_forward_as<EL, EPI_SWIGLU_ACT, true>(args, st);
    return launch_forward_as<EL, EPI_PLAIN, true>(args, st);
}

}  // namespace

int launch_tall(const Args& args, int epi, bool b_kc, bool bf16, hipStream_t st) {
    return bf16 ? launch_as<ElemBf16>(args, epi, b_kc, st) : launch_as<ElemF16>(args, epi, b_kc, st);
}

}  // namespace ragged
}  // namespace gemm
}  // namespace fmahip
