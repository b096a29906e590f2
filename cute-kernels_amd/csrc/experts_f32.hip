// The expert path of an fp32 SwiGLU layer, forward and backward, enqueued by one call each: the kernels of the entry points named in
// the header, in their order. fp32 layers are small, and five and seven calls through an operator, each with its own node in the
// autograd graph, took longer on the host than the kernels on the device.
#include "common.h"

extern "C" {

int fma_swiglu_experts_f32(const void* x, const int32_t* inv, const void* gates, const void* W1, const void* W2, const uint32_t* counts,
                           const uint32_t* N1, const uint32_t* K1, const uint32_t* N2, const uint32_t* K2, int64_t T, int64_t k,
                           int64_t E, int64_t H, int64_t I, void* xg, void* h, void* act, void* o, void* y, void* stream) {
    using namespace fmahip;
    FMA_REQUIRE(T >= 1 && k >= 1 && E >= 1 && H >= 1 && I >= 1, FMA_ERR_BAD_SIZE, "swiglu_experts_f32: sizes must be positive");
    FMA_REQUIRE(x && inv && gates && W1 && W2 && counts && N1 && K1 && N2 && K2 && xg && h && act && o && y, FMA_ERR_NULL_POINTER,
                "swiglu_experts_f32: NULL pointer");
    const int64_t R = T * k;
    float* const hf = (float*)h;
    int rc = fma_dispatch_rows(x, inv, T, k, H, xg, FMA_F32, stream);
    if (!rc) rc = fma_grouped_gemm(xg, W1, h, counts, N1, K1, E, 0, 1, 1.0f, FMA_F32, stream);
    if (!rc) rc = fma_swiglu_forward(hf + I, hf, act, R, I, 2 * I, 2 * I, I, FMA_F32, stream);
    if (!rc) rc = fma_grouped_gemm(act, W2, o, counts, N2, K2, E, 0, 1, 1.0f, FMA_F32, stream);
    if (!rc) rc = fma_combine(o, inv, gates, T, k, H, y, FMA_F32, stream);
    return rc;
}

int fma_swiglu_experts_bwd_f32(const void* dy, const int32_t* inv, const void* gates, const void* W1, const void* W2, const void* xg,
                               const void* h, const void* act, const void* o, const uint32_t* counts, const uint32_t* N1,
                               const uint32_t* K1, const uint32_t* N2, const uint32_t* K2, int64_t T, int64_t k, int64_t E, int64_t H,
                               int64_t I, void* d_o, void* d_act, void* d_h, void* dx, void* d_gates, void* dW1, void* dW2,
                               void* stream) {
    using namespace fmahip;
    FMA_REQUIRE(T >= 1 && k >= 1 && E >= 1 && H >= 1 && I >= 1, FMA_ERR_BAD_SIZE, "swiglu_experts_bwd_f32: sizes must be positive");
    FMA_REQUIRE(dy && inv && gates && W1 && W2 && xg && h && act && o && counts && N1 && K1 && N2 && K2 && d_o,
                FMA_ERR_NULL_POINTER, "swiglu_experts_bwd_f32: NULL pointer");
    FMA_REQUIRE((d_act && d_h) || !(dx || dW1), FMA_ERR_NULL_POINTER, "swiglu_experts_bwd_f32: dx and dW1 need d_act and d_h");
    const int64_t R = T * k;
    const float* const hf = (const float*)h;
    float* const dhf = (float*)d_h;
    int rc = fma_combine_bwd(dy, o, inv, gates, T, k, H, d_o, d_gates, FMA_F32, stream);
    // dW2_e = d_o_e^T act_e
    if (!rc && dW2) rc = fma_grouped_gemm(d_o, act, dW2, N2, K2, counts, E, 1, 0, 1.0f, FMA_F32, stream);
    if (dx || dW1) {
        // d_act_e = d_o_e W2_e, then the activation's backward
        if (!rc) rc = fma_grouped_gemm(d_o, W2, d_act, counts, K2, N2, E, 0, 0, 1.0f, FMA_F32, stream);
        if (!rc) rc = fma_swiglu_backward(hf + I, hf, d_act, dhf + I, dhf, R, I, 2 * I, 2 * I, I, 2 * I, 2 * I, FMA_F32, stream);
        if (!rc && dW1) rc = fma_grouped_gemm(d_h, xg, dW1, N1, K1, counts, E, 1, 0, 1.0f, FMA_F32, stream);
        // the gradient of the grouped rows takes the place of d_o, which nothing reads any more
        if (!rc && dx) rc = fma_grouped_gemm(d_h, W1, d_o, counts, K1, N1, E, 0, 0, 1.0f, FMA_F32, stream);
        if (!rc && dx) rc = fma_combine(d_o, inv, nullptr, T, k, H, dx, FMA_F32, stream);
    }
    return rc;
}

}  // extern "C"
