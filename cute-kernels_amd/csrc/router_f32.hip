// The router of an fp32 layer in one pass: logits = x @ Wg^T on the fp32 matrix instruction, top-k, softmax over the k kept logits and
// the choices counted per 16 tokens; and the backward of the top-k and softmax. fp32 layers are small, so both are bound by latency:
// what counts is that the product, the selection (two launches in ATen), the softmax and, in the backward, its gradient, the scatter
// and the sum with the logits' own gradient are one launch each. At 512 tokens, hidden 256, E 8, k 2: 8.1 us
// against 27 us of the four launches that stood there, and 4.4 us against 14 us of four.
// A workgroup takes 16 tokens; its four wavefronts share the reduction (16 k per step: a lane loads four consecutive k of one token and
// of one expert per 16 experts, and feeds the four instructions of the step from them) and their partial sums are added in a fixed
// order through LDS. Sixteen lanes then select and weigh the choices of a token.
#include "router_parts.h"

namespace fmahip {
namespace {

constexpr int kThreads = 256, kWaves = kThreads / kWave;
constexpr int kColBlocks = 4, kCols = kColBlocks * 16;  // experts per pass over x

struct F32RouterArgs {
    const float* x;        // [T, H]
    const float* w;        // [E, H]
    float* logits;         // [T, E]
    float* weights;        // [T, k]
    float* kept;           // [T, k] or null: the chosen logits
    int32_t* selected;     // [T, k]
    uint32_t* hist;        // [ceil(T / 16), E] or null
    int64_t T;
    int32_t H, E, k;
};

// unsigned order equals numeric order, NaN above everything, -0 equal to +0; never 0, which marks a column that is taken
__device__ __forceinline__ uint32_t order_of(float x) {
    const uint32_t b = __float_as_uint(x);
    if ((b & 0x7fffffffu) > 0x7f800000u) return 0xffffffffu;
    if (b == 0x80000000u) return 0x80000000u;
    return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}
__device__ __forceinline__ float value_of(uint32_t ord) {
    if (ord == 0xffffffffu) return __uint_as_float(0x7fc00000u);
    return __uint_as_float((ord & 0x80000000u) ? (ord & 0x7fffffffu) : ~ord);
}

template <int EMAX>
__global__ __launch_bounds__(kThreads) void router_topk_f32_kernel(const F32RouterArgs a) {
    __shared__ float s_part[kWaves][kTok][kCols];
    __shared__ uint32_t s_key[kTok][EMAX + kRowPad];
    __shared__ uint32_t s_hist[EMAX];
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid >> 6;
    const int r = lane & 15, q = lane >> 4;
    const int H = a.H, E = a.E;
    const int64_t tok0 = (int64_t)blockIdx.x * kTok;
    for (int n = tid; n < E; n += kThreads) s_hist[n] = 0;

    // rows past the end repeat the last token, columns past E the last expert; neither is stored
    const int64_t t = tok0 + r;
    const float* const xa = a.x + (t < a.T ? t : a.T - 1) * H;
    for (int col0 = 0; col0 < E; col0 += kCols) {
        const float* wb[kColBlocks];
        f32x4 acc[kColBlocks];
#pragma unroll
        for (int b = 0; b < kColBlocks; ++b) {
            const int n = col0 + b * 16 + r;
            wb[b] = a.w + (int64_t)(n < E ? n : E - 1) * H;
            acc[b] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
        for (int k0 = wave * 16; k0 < H; k0 += kWaves * 16) {
            // (H is a multiple of 4: a lane's four k are all inside or all outside; outside they read k 0 and count as zeros)
            const int k = k0 + q * 4;
            const bool in = k < H;
            f32x4 fx = *reinterpret_cast<const f32x4*>(xa + (in ? k : 0)), fw[kColBlocks];
#pragma unroll
            for (int b = 0; b < kColBlocks; ++b) fw[b] = *reinterpret_cast<const f32x4*>(wb[b] + (in ? k : 0));
            if (!in) {
                fx = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int b = 0; b < kColBlocks; ++b) fw[b] = fx;
            }
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int b = 0; b < kColBlocks; ++b) acc[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(fx[j], fw[b][j], acc[b], 0, 0, 0);
        }
        // a lane holds tokens 4 q .. + 3 of expert r of every block
        __syncthreads();  // the sums of the pass before are read
#pragma unroll
        for (int b = 0; b < kColBlocks; ++b)
#pragma unroll
            for (int i = 0; i < 4; ++i) s_part[wave][q * 4 + i][b * 16 + r] = acc[b][i];
        __syncthreads();
        for (int i = tid; i < kTok * kCols; i += kThreads) {
            const int tok = i / kCols, c = i % kCols, n = col0 + c;
            if (n >= E) continue;
            float sum = s_part[0][tok][c];
#pragma unroll
            for (int w = 1; w < kWaves; ++w) sum += s_part[w][tok][c];
            s_key[tok][n] = order_of(sum);
            if (tok0 + tok < a.T) a.logits[(tok0 + tok) * E + n] = sum;
        }
    }
    __syncthreads();

    // ---- top-k and softmax: lane c of a token's sixteen owns the columns congruent to c and remembers choices c, c + 16, ... ----
    const int tok = tid >> 4, c = tid & 15;
    const int64_t token = tok0 + tok;
    uint32_t* const keys = s_key[tok];
    float val[kMaxTopK / 16];
    int col[kMaxTopK / 16];
    float vmax = 0.f;
#pragma unroll
    for (int i = 0; i < kMaxTopK / 16; ++i) {
        val[i] = 0.f;
        col[i] = 0;
    }
    for (int j = 0; j < a.k; ++j) {
        uint32_t mine = 0, at = 0;
        for (int n = c; n < E; n += 16) {
            const uint32_t key = keys[n];
            if (key > mine) {
                mine = key;
                at = (uint32_t)n;
            }
        }
        const uint32_t best = row16_max(mine);                                    // top_k <= E: not 0
        const int chosen = (int)~row16_max(mine == best && mine != 0 ? ~at : 0u);  // the lowest column of that value
        if ((chosen & 15) == c) keys[chosen] = 0;
        if (j == 0) vmax = value_of(best);
#pragma unroll
        for (int i = 0; i < kMaxTopK / 16; ++i)
            if (c == (j & 15) && (j >> 4) == i) {
                val[i] = value_of(best);
                col[i] = chosen;
            }
    }
    if (a.kept && token < a.T) {
#pragma unroll
        for (int i = 0; i < kMaxTopK / 16; ++i)
            if (c + 16 * i < a.k) a.kept[token * a.k + c + 16 * i] = val[i];
    }
    float sum = 0.f;
#pragma unroll
    for (int i = 0; i < kMaxTopK / 16; ++i) {
        val[i] = c + 16 * i < a.k ? expf(val[i] - vmax) : 0.f;
        sum += val[i];
    }
    sum = row16_sum(sum);
    if (token < a.T) {
#pragma unroll
        for (int i = 0; i < kMaxTopK / 16; ++i) {
            const int j = c + 16 * i;
            if (j < a.k) {
                a.selected[token * a.k + j] = col[i];
                a.weights[token * a.k + j] = val[i] / sum;
                if (a.hist) atomicAdd(&s_hist[col[i]], 1u);
            }
        }
    }
    if (a.hist) {
        __syncthreads();
        for (int n = tid; n < E; n += kThreads) a.hist[(int64_t)blockIdx.x * E + n] = s_hist[n];
    }
}

__device__ __forceinline__ double row16_sum(double v) {
#pragma unroll
    for (int d = 1; d < 16; d <<= 1) v += __shfl_xor(v, d, kWave);
    return v;
}

// d_out[t, :] = d_logits[t, :] (zeros if absent), and at the k chosen columns s_j (dw_j - sum_i s_i dw_i) more. 16 lanes per token.
// (s_j and the difference in double: the gradients of a token's choices nearly cancel in it, and these are k values per token)
__global__ __launch_bounds__(kThreads) void router_topk_bwd_f32_kernel(const float* __restrict__ kept,
                                                                       const int32_t* __restrict__ selected,
                                                                       const float* __restrict__ d_weights,
                                                                       const float* __restrict__ d_logits, int64_t T, int E, int k,
                                                                       float* __restrict__ d_out) {
    __shared__ int32_t s_sel[kTok][kMaxTopK];
    __shared__ float s_ds[kTok][kMaxTopK];
    const int tid = threadIdx.x, tok = tid >> 4, c = tid & 15;
    const int64_t t = (int64_t)blockIdx.x * kTok + tok;
    const bool live = t < T;
    const int64_t tt = live ? t : T - 1;
    double s[kMaxTopK / 16], dw[kMaxTopK / 16], sum = 0.0;
    int sel[kMaxTopK / 16];
    const float vmax = kept[tt * k];  // the first choice is the largest kept logit
#pragma unroll
    for (int i = 0; i < kMaxTopK / 16; ++i) {
        const int j = c + 16 * i;
        sel[i] = -1;
        s[i] = dw[i] = 0.0;
        if (j < k) {
            sel[i] = selected[tt * k + j];
            s[i] = (double)expf(kept[tt * k + j] - vmax);
            dw[i] = d_weights ? (double)d_weights[tt * k + j] : 0.0;
            sum += s[i];
        }
    }
    sum = row16_sum(sum);
    double dot = 0.0;
#pragma unroll
    for (int i = 0; i < kMaxTopK / 16; ++i) {
        s[i] = s[i] / sum;
        dot += s[i] * dw[i];
    }
    dot = row16_sum(dot);
#pragma unroll
    for (int i = 0; i < kMaxTopK / 16; ++i) {
        const int j = c + 16 * i;
        if (j < k) {
            s_sel[tok][j] = sel[i];
            s_ds[tok][j] = (float)(s[i] * (dw[i] - dot));
        }
    }
    __syncthreads();
    if (!live) return;
    for (int n = c; n < E; n += 16) {
        float v = d_logits ? d_logits[t * E + n] : 0.f;
        for (int j = 0; j < k; ++j)
            if (s_sel[tok][j] == n) v = s_ds[tok][j] + v;
        d_out[t * E + n] = v;
    }
}

int check_f32(const char* what, int64_t T, int64_t E, int64_t k) {
    FMA_REQUIRE(T >= 0 && T <= 0x7fffffffll, FMA_ERR_BAD_SIZE, "%s: bad token count %lld", what, (long long)T);
    FMA_REQUIRE(E >= 1 && E <= FMA_MAX_GROUPS, FMA_ERR_TOO_MANY_EXPERTS, "%s: E must be in [1, %d] (got %lld)", what, FMA_MAX_GROUPS,
                (long long)E);
    FMA_REQUIRE(k >= 1 && k <= E && k <= FMA_MAX_ROUTER_TOP_K, FMA_ERR_BAD_SIZE,
                "%s: top_k must be in [1, min(E, %d)] (got %lld, E = %lld)", what, FMA_MAX_ROUTER_TOP_K, (long long)k, (long long)E);
    FMA_REQUIRE(T * E <= 0x7fffffffll && T * k <= 0x7fffffffll, FMA_ERR_TOO_MANY_ELEMENTS, "%s: T*E and T*top_k must stay below 2^31",
                what);
    return FMA_OK;
}

}  // namespace
}  // namespace fmahip

extern "C" {

int fma_router_topk_f32(const void* x, const void* gate_weight, int64_t T, int64_t H, int64_t E, int64_t top_k, void* logits,
                        void* weights, int32_t* selected, uint32_t* token_block_hist, void* kept, void* stream) {
    using namespace fmahip;
    const int rc = check_f32("router_topk_f32", T, E, top_k);
    if (rc) return rc;
    FMA_REQUIRE(H >= 4 && H % 4 == 0 && H <= (1 << 24), FMA_ERR_BAD_SIZE, "router_topk_f32: H must be a multiple of 4 in [4, 2^24] (got %lld)",
                (long long)H);
    if (T == 0) return FMA_OK;
    FMA_REQUIRE(x && gate_weight && logits && weights && selected, FMA_ERR_NULL_POINTER, "router_topk_f32: NULL pointer");
    FMA_REQUIRE(aligned16(x) && aligned16(gate_weight), FMA_ERR_MISALIGNED, "router_topk_f32: x and gate_weight must be 16-byte aligned");
    F32RouterArgs a;
    a.x = (const float*)x;
    a.w = (const float*)gate_weight;
    a.logits = (float*)logits;
    a.weights = (float*)weights;
    a.selected = selected;
    a.kept = (float*)kept;
    a.hist = token_block_hist;
    a.T = T;
    a.H = (int32_t)H;
    a.E = (int32_t)E;
    a.k = (int32_t)top_k;
    const dim3 grid((uint32_t)((T + kTok - 1) / kTok)), block(kThreads);
    if (E <= 128) hipLaunchKernelGGL(router_topk_f32_kernel<128>, grid, block, 0, (hipStream_t)stream, a);
    else hipLaunchKernelGGL(router_topk_f32_kernel<FMA_MAX_GROUPS>, grid, block, 0, (hipStream_t)stream, a);
    return launch_status("router_topk_f32");
}

int fma_router_topk_bwd_f32(const void* kept, const int32_t* selected, const void* d_weights, const void* d_logits, int64_t T,
                            int64_t E, int64_t top_k, void* d_out, void* stream) {
    using namespace fmahip;
    const int rc = check_f32("router_topk_bwd_f32", T, E, top_k);
    if (rc) return rc;
    if (T == 0) return FMA_OK;
    FMA_REQUIRE(kept && selected && d_out, FMA_ERR_NULL_POINTER, "router_topk_bwd_f32: NULL pointer");
    hipLaunchKernelGGL(router_topk_bwd_f32_kernel, dim3((uint32_t)((T + kTok - 1) / kTok)), dim3(kThreads), 0, (hipStream_t)stream,
                       (const float*)kept, selected, (const float*)d_weights, (const float*)d_logits, T, (int)E, (int)top_k,
                       (float*)d_out);
    return launch_status("router_topk_bwd_f32");
}

}  // extern "C"
