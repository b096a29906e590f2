// What decode.hip uses of the streaming kernels for a few rows per expert (thin_experts.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace fmahip {
namespace gemm {
namespace thin {

// The argument checks of one product: 0 or an error, with its message stored for fma_last_error_string()
int check(const char* who, const void* x, int64_t x_rows, const int32_t* row_index, int32_t divisor, const void* W,
          const void* out, const uint32_t* counts, const uint32_t* offsets, int64_t R, int64_t E, int64_t N, int64_t K, int swiglu,
          int dtype);

// The expert path of one token: act [top_k, I] is scratch, y [H] the layer's output. E up to FMA_MAX_DECODE_EXPERTS.
bool takes_one_token(int64_t T, int64_t top_k);
int one_token(const void* x, const void* logits, const void* W1, const void* bias1, const void* W2, const void* bias2, void* act, void* y,
              int64_t E, int64_t H, int64_t I, int64_t top_k, int dtype, hipStream_t st);

}  // namespace thin
}  // namespace gemm
}  // namespace fmahip
