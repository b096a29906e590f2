// Grouped product for groups of a few rows (a decode step): out_e = x_e W_e^T, rows packed or gathered from the tokens, with
// the bias and the SwiGLU activation in the epilogue if asked for. Same results, bit for bit, as the tile kernel of
// grouped_gemm_ragged.hip: the same 16x16x32 instruction walks the reduction in the same order.
//
// What bounds it: the weights, read once each, against a handful of rows; the product is a stream of E_active * N * K elements.
// The tile kernel spends that stream in 256-column tiles (one workgroup per compute unit, two or three K steps in flight, and for
// one token of the fine-grained shape 88 tiles for 256 compute units). Here the unit of work is ONE wavefront with 16, 32 or 64 weight
// rows over the whole reduction:
//  * no workgroup barrier anywhere: a wavefront fills a private ring of LDS stages by direct global -> LDS loads, each
//    instruction 8 rows x 128 bytes (whole cache lines), waits with a counted vmcnt and multiplies; 6 such wavefronts (3 of the
//    64-row kind) fit a compute unit's LDS and keep 70 to 90 KB in flight there;
//  * the weight loads carry the non-temporal hint where every line is used by one wavefront only. A plain read kernel over 1.9 GB
//    measures 6.3 TB/s without and 7.1 to 7.5 TB/s with it; this kernel 5.7 and 6.3 TB/s (up), 6.0 and 6.9 TB/s (down). The
//    tokens, which every wavefront of an expert reads, are loaded without it (with it: +5 % time at 13 rows per expert).
// Measured, bf16, up / down projection, weights from HBM (three sets in turn), against the tile kernel:
//   hidden 2048, I 1408, E 64, k 8, 1 token:    30.9 / 21.5 us -> 16.7 / 9.4 us (5.5 / 4.9 TB/s: two launches' ramp)
//   hidden 2048, I 1024, E 64, k 8, 8 tokens:   104 / 49 us -> 67 / 29 us
//   hidden 4096, I 14336, E 8, k 2, 16 tokens:  369 / 171 us -> 297 / 136 us (6.3 / 6.9 TB/s)
//   hidden 4096, I 1536, E 128, k 8, 100 tokens: 611 / 290 us -> 506 / 244 us
// Tried: 256 bytes per row and instruction (-0 to +8 % time), deeper rings with fewer wavefronts (0 to +10 %), rings of three
// stages with eight wavefronts (+3 % on the large shapes, -2 % on the small).
// An expert with more rows than a pass holds (32, or 64 of the other kind) streams its weights once per pass. The passes run
// side by side, eight workgroups apart, in step (all with the token blocks of a full pass) and without the non-temporal hint, so that
// the second pass finds the lines in the XCD's L2. Whole layer, us: the tile kernel / one wavefront taking the passes one after
// the other / this, at uneven routing:
//   hidden 2048, I 768, E 128, k 8, 512 tokens, one expert in every token's choice: 355 / 440 / 303
//   hidden 2048, I 768, E 256, k 8, 1024 tokens, two experts in every choice:       619 / 963 / 567
//   hidden 4096, I 14336, E 8, k 2, 64 tokens, all with the same two experts:        255 / 361 / 243
//   hidden 4096, I 1536, E 128, k 8, 128 tokens, all with the same eight experts:    223 / 271 / 190
// With the hint the last two take 269 and 215 us; with the smaller token blocks of a short last pass, which then runs ahead of the
// others, 48 tokens of the third take 286 instead of 230 us.
#include "gemm_parts.h"
#include "router_parts.h"
#include "thin_experts.h"

namespace fmahip {
namespace gemm {
namespace ragged {
// grouped_gemm_ragged.hip
int up_projection(const char* who, const void* x, int64_t x_rows, const int32_t* row_index, int32_t divisor, const void* W,
                  const void* bias, void* out, void* act, const uint32_t* M_arr, int64_t E, int64_t N, int64_t K, int swiglu,
                  int dtype, hipStream_t st, uint32_t* taken, uint32_t pass_bits);
}  // namespace ragged
namespace thin {

struct Args {
    const uint16_t* x;         // row_index: tokens [x_rows, K]; otherwise packed rows [R, K]
    const int32_t* row_index;  // [R] grouped row -> slot, the token being slot / divisor; or NULL
    const uint16_t* W;         // [E, N, K] (swiglu: N = 2 I, "up" rows first)
    const uint16_t* bias;      // [E, N] or NULL
    uint16_t* out;             // [R, N]; swiglu: [R, I]
    const uint32_t* counts;    // [E] rows per expert
    const uint32_t* offsets;   // [E] inclusive prefix of counts
    uint32_t E, N, K;
    uint32_t divisor, x_rows;
    uint32_t units;  // wavefronts per pass of an expert
    uint32_t slots;  // passes of an expert that run side by side
    const uint32_t* taken;  // not NULL: the tile kernel in front has computed the product if *taken
};

constexpr uint32_t kKB = 128;  // bytes of a row per step: one cache line
constexpr uint32_t kRPI = 8;   // rows per load instruction

// Byte offset of 16-byte chunk `chunk` of row `row` in a stage. Two rows share 256 bytes; the flip spreads the 16 rows that a
// fragment read touches at one chunk over all sixteen 16-byte columns (no bank conflicts).
__device__ __forceinline__ uint32_t flip(uint32_t row) { return (row >> 1) & 7u; }
__device__ __forceinline__ uint32_t lds_off(uint32_t row, uint32_t chunk) { return row * kKB + ((chunk ^ flip(row)) << 4); }

template <int ROWS>
struct Config;
template <>
struct Config<16> {  // launches of few units (half_units)
    static constexpr uint32_t kLds = 24576;
    static constexpr uint32_t kMaxTokens = 32;
};
template <>
struct Config<32> {  // up to about 16 rows per expert
    static constexpr uint32_t kLds = 24576;
    static constexpr uint32_t kMaxTokens = 32;
};
template <>
struct Config<64> {  // more: a token fragment feeds twice as many instructions
    static constexpr uint32_t kLds = 51200;
    static constexpr uint32_t kMaxTokens = 64;
};

// ROWS weight rows from column n0 on (swiglu: half of them "up", half "gate") times `rows` <= 16 TB rows from grouped row row0.
// STREAM: weights with the non-temporal hint, for lines that no other wavefront reads.
template <typename EL, int ROWS, bool GLU, bool BIAS, int TB, bool STREAM>
__device__ __forceinline__ void unit(const Args& a, uint8_t* lds, uint32_t e, uint32_t row0, uint32_t rows, uint32_t n0) {
    using frag = typename EL::frag;
    constexpr int WB = ROWS / 16;
    constexpr int kWI = ROWS / kRPI, kTI = TB * 16 / kRPI;  // load instructions per step
    constexpr int kIPS = kWI + kTI;
    constexpr uint32_t kStage = (ROWS + TB * 16) * kKB;
    constexpr int kD = Config<ROWS>::kLds / kStage;  // stages of the ring
    static_assert(kD >= 2 && kIPS * (kD - 1) < 64, "two stages, and vmcnt holds six bits");
    constexpr uint32_t kCols = GLU ? ROWS / 2 : ROWS;
    const uint32_t lane = threadIdx.x;
    const uint32_t K2 = a.K * 2u;
    const uint32_t I = GLU ? a.N / 2 : a.N;
    const uint32_t lr = lane >> 3, lp = lane & 7u;

    // descriptors end with the rows of this unit that exist: the rest arrives as zeros
    const uint64_t We = (uint64_t)e * a.N;
    const uint32_t n_rows = I - n0 < kCols ? I - n0 : kCols;
    const u32x4 rw0 = make_rsrc_words(a.W + (We + n0) * a.K, n_rows * K2);
    const u32x4 rw1 = GLU ? make_rsrc_words(a.W + (We + I + n0) * a.K, n_rows * K2) : rw0;
    const u32x4 rx = a.row_index ? make_rsrc_words(a.x, a.x_rows * K2)
                                 : make_rsrc_words(a.x + (uint64_t)row0 * a.K, rows * K2);
    uint32_t tok_off[kTI];  // this lane's row in each of the token load instructions
#pragma unroll
    for (int i = 0; i < kTI; ++i) {
        const uint32_t r = (uint32_t)i * kRPI + lr;
        uint32_t src = r;
        if (a.row_index) src = r < rows ? (uint32_t)a.row_index[row0 + r] / a.divisor : a.x_rows;
        tok_off[i] = r < rows && (!a.row_index || src < a.x_rows) ? src * K2 : kOutOfRange;
    }
    const uint32_t lds0 = lds_address(lds);
    const uint32_t nsteps = (K2 + kKB - 1) / kKB;

    auto issue = [&](uint32_t s, uint32_t slot) {
        const uint32_t stage = lds0 + slot * kStage;
        const uint32_t kb = s * kKB;
        const bool last = kb + kKB > K2;  // the partial last step, or a step past it: chunks past the row are out of range
#pragma unroll
        for (int i = 0; i < kWI; ++i) {
            const uint32_t chunk = lp ^ flip((uint32_t)i * kRPI + lr);
            const uint32_t rel = GLU ? (uint32_t)(i % (kWI / 2)) * kRPI : (uint32_t)i * kRPI;
            uint32_t v = lr * K2 + chunk * 16u;
            if (last && kb + chunk * 16u >= K2) v = kOutOfRange;
            load_lds<STREAM>(GLU && i >= kWI / 2 ? rw1 : rw0, v, rel * K2 + kb, stage + (uint32_t)i * 1024u);
        }
#pragma unroll
        for (int i = 0; i < kTI; ++i) {
            const uint32_t chunk = lp ^ flip((uint32_t)i * kRPI + lr);
            uint32_t v = tok_off[i] + chunk * 16u;
            if (last && kb + chunk * 16u >= K2) v = kOutOfRange;
            load_lds<false>(rx, v, kb, stage + (uint32_t)(kWI + i) * 1024u);
        }
    };

    f32x4 acc[WB][TB];
#pragma unroll
    for (int b = 0; b < WB; ++b)
#pragma unroll
        for (int t = 0; t < TB; ++t) acc[b][t] = f32x4{0.f, 0.f, 0.f, 0.f};

#pragma unroll
    for (int d = 0; d < kD - 1; ++d) issue((uint32_t)d, (uint32_t)d);
    const uint32_t r16 = lane & 15u, q = lane >> 4;
    uint32_t slot = 0, fill = kD - 1;
    for (uint32_t s = 0; s < nsteps; ++s) {
        wait_lds();  // the stage filled here was read in the previous iteration
        issue(s + kD - 1, fill);
        fill = fill == kD - 1 ? 0 : fill + 1;
        wait_vm<kIPS*(kD - 1)>();
        const uint8_t* stage = lds + slot * kStage;
        slot = slot == kD - 1 ? 0 : slot + 1;
#pragma unroll
        for (int sl = 0; sl < 2; ++sl) {
            const uint32_t c = (uint32_t)sl * 4u + q;
            frag w[WB], t[TB];
#pragma unroll
            for (int b = 0; b < WB; ++b)
                w[b] = __builtin_bit_cast(frag, read_kc_frag(stage + lds_off((uint32_t)b * 16u + r16, c)));
#pragma unroll
            for (int j = 0; j < TB; ++j)
                t[j] = __builtin_bit_cast(frag, read_kc_frag(stage + lds_off((uint32_t)(ROWS + j * 16) + r16, c)));
#pragma unroll
            for (int b = 0; b < WB; ++b)
#pragma unroll
                for (int j = 0; j < TB; ++j) acc[b][j] = EL::mfma16(w[b], t[j], acc[b][j]);
        }
    }
    wait_vm<0>();  // the loads past the end write zeros into the ring: they are done before it is used again

    // a lane holds row r16, columns 4 q .. 4 q + 3 of each block; rounding points as in the tile kernel's epilogue
    // (one block with both halves: 8 "up" columns in lanes 0 .. 31, their "gate" in lanes 32 .. 63)
    constexpr bool kOneBlock = GLU && WB == 1;
#pragma unroll
    for (int j = 0; j < TB; ++j) {
        float gate[4];
        if constexpr (kOneBlock) {
#pragma unroll
            for (int x = 0; x < 4; ++x) gate[x] = __shfl_xor(acc[0][j][x], 32, 64);
        }
        const uint32_t row = (uint32_t)j * 16u + r16;
        if (row >= rows || (kOneBlock && q >= 2u)) continue;
#pragma unroll
        for (int b = 0; b < (GLU && WB > 1 ? WB / 2 : WB); ++b) {
            const uint32_t c = n0 + (uint32_t)b * 16u + 4u * q;
            if (c >= I) continue;
            float y[4];
#pragma unroll
            for (int x = 0; x < 4; ++x) {
                float u = acc[b][j][x];
                if constexpr (BIAS) u = EL::round(u) + EL::from_bits(a.bias[We + c + x]);
                if constexpr (GLU) {
                    float g = kOneBlock ? gate[x] : acc[kOneBlock ? 0 : WB / 2 + b][j][x];
                    if constexpr (BIAS) g = EL::round(g) + EL::from_bits(a.bias[We + I + c + x]);
                    u = EL::round(u);
                    g = EL::round(g);
                    y[x] = u * g * sigmoid_for<typename EL::act_t>(g);
                } else {
                    y[x] = u;
                }
            }
            uint2 w;
            w.x = EL::pack2(y[0], y[1]);
            w.y = EL::pack2(y[2], y[3]);
            *reinterpret_cast<uint2*>(a.out + (uint64_t)(row0 + row) * I + c) = w;
        }
    }
}

// What a launch has to reckon with. One kernel for all three takes 1 % longer at one to eight tokens.
constexpr int ONE_PASS = 0;     // no expert has more rows than a pass (if one has, its passes follow one another)
constexpr int MANY_PASSES = 1;  // some may have
constexpr int MAY_YIELD = 2;    // and the tile kernel in front may have computed the product

// Workgroup = one wavefront: one unit of one pass of an expert, of which up to a.slots run side by side. The host does not know
// how many experts have rows, nor how many passes they take: workgroups beyond the last end at once.
template <typename EL, int ROWS, bool GLU, bool BIAS, int PASSES>
__global__ __launch_bounds__(64) void thin_gemm_kernel(const Args a) {
    __shared__ __attribute__((aligned(1024))) uint8_t lds[Config<ROWS>::kLds];
    constexpr uint32_t kMax = Config<ROWS>::kMaxTokens;
    const uint32_t lane = threadIdx.x;
    if constexpr (PASSES == MAY_YIELD) {
        if (*a.taken) return;
    }
    const uint32_t j = blockIdx.x / a.units;  // slot, counted over all experts
    uint32_t e = a.E, seen = 0, slots = 1;
    for (uint32_t base = 0; base < a.E; base += 64) {
        const uint32_t m = base + lane < a.E ? a.counts[base + lane] : 0u;
        uint32_t before, here, mine = m != 0 ? 1u : 0u;  // slots of the experts before this lane's, of all 64, of this lane's
        if (PASSES == ONE_PASS || __ballot(m > kMax) == 0) {
            const uint64_t mask = __ballot(m != 0);
            before = (uint32_t)__popcll(mask & ((1ull << lane) - 1ull));
            here = (uint32_t)__popcll(mask);
        } else {
            mine = (m + kMax - 1) / kMax;
            mine = mine < a.slots ? mine : a.slots;
            before = wave_inclusive_scan<uint32_t>(mine);
            here = (uint32_t)__builtin_amdgcn_readlane((int)before, 63);
            before -= mine;
        }
        if (seen + here > j) {
            const uint32_t src = (uint32_t)__builtin_ctzll(__ballot(before <= j - seen && j - seen < before + mine));
            e = base + src;
            slots = (uint32_t)__builtin_amdgcn_readlane((int)mine, (int)src);
            seen += (uint32_t)__builtin_amdgcn_readlane((int)before, (int)src);
            break;
        }
        seen += here;
    }
    e = uniform(e);
    if (e >= a.E) return;
    uint32_t slot = 0, u = blockIdx.x - seen * a.units;
    if (PASSES != ONE_PASS && __builtin_expect(slots > 1, 0)) {
        const uint32_t whole = a.units & ~7u;  // the last units of an expert, fewer than eight, lie that many apart
        if (u < whole * slots) {
            slot = u / 8u % slots;
            u = u / (8u * slots) * 8u + u % 8u;
        } else {
            u -= whole * slots;
            slot = u / (a.units - whole);
            u = whole + u % (a.units - whole);
        }
    }
    uint32_t rows = uniform(a.counts[e]);
    uint32_t first = uniform(a.offsets[e]) - rows;
    const uint32_t n0 = u * (GLU ? ROWS / 2 : ROWS);
    if constexpr (PASSES != ONE_PASS) {
        if (__builtin_expect(slots > 1, 0)) {
            for (uint32_t at = slot * kMax; at < rows; at += slots * kMax)
                unit<EL, ROWS, GLU, BIAS, kMax / 16, false>(a, lds, e, first + at, rows - at < kMax ? rows - at : kMax, n0);
            return;
        }
    }
    while (rows) {
        if (rows <= 16) {
            unit<EL, ROWS, GLU, BIAS, 1, true>(a, lds, e, first, rows, n0);
            break;
        }
        if (kMax > 32 && rows <= 32) {
            unit<EL, ROWS, GLU, BIAS, 2, true>(a, lds, e, first, rows, n0);
            break;
        }
        const uint32_t take = rows < kMax ? rows : kMax;
        unit<EL, ROWS, GLU, BIAS, kMax / 16, true>(a, lds, e, first, take, n0);
        first += take;
        rows -= take;
    }
}

template <typename EL, int ROWS, int PASSES>
int launch(Args a, bool glu, int64_t R, int64_t groups, hipStream_t st) {
    const uint32_t cols = glu ? a.N / 2 : a.N, per = glu ? ROWS / 2 : ROWS;
    a.units = (cols + per - 1) / per;
    // slots: one for every expert with rows, and one more for every kMaxTokens rows beyond its first; the grid stays far below the
    // launch limit of 2^32 threads
    constexpr int64_t kMaxSlots = PASSES == ONE_PASS ? 1 : 16, kMaxGrid = 1 << 25;
    const int64_t most = kMaxGrid / (groups * a.units);
    a.slots = (uint32_t)(most < 1 ? 1 : (most < kMaxSlots ? most : kMaxSlots));
    const int64_t extra = (R - groups) / Config<ROWS>::kMaxTokens, spare = groups * (a.slots - 1);
    const dim3 grid((uint32_t)((groups + (extra < spare ? extra : spare)) * a.units)), block(64);
    auto run = [&](auto kernel) { hipLaunchKernelGGL(kernel, grid, block, 0, st, a); };
    if (glu) a.bias ? run(thin_gemm_kernel<EL, ROWS, true, true, PASSES>) : run(thin_gemm_kernel<EL, ROWS, true, false, PASSES>);
    else a.bias ? run(thin_gemm_kernel<EL, ROWS, false, true, PASSES>) : run(thin_gemm_kernel<EL, ROWS, false, false, PASSES>);
    return launch_status("grouped_gemm_thin");
}
// Units of 16 weight rows where a launch has at most two units of 32 per compute unit, a third of what fits its LDS, and a reduction
// long enough to stream: twice as many wavefronts, with rings of five stages in flight instead of three. Whole layer of one token,
// units of 32 -> 16 where the line says so, us: hidden 2048, I 8192, E 8, k 2 (second projection: 128 units) 75.5 -> 66.8, 2 / 4 / 8
// tokens 93.4 -> 83.8, 116.7 -> 109.7, 141.5 -> 137.2; hidden 2880, I 2880, E 32, k 4 53.3 -> 50.8; hidden 2048, I 768, E 128, k 8 34.6
// -> 33.5. With up to three units per compute unit and any reduction: hidden 2048, I 1408, E 64 (K 1408) 42.3 -> 43.2, hidden 2880 with
// two tokens 82.1 -> 84.5.
bool half_units(const Args& a, bool glu, int64_t groups) {
    const int64_t cus = num_compute_units() > 0 ? num_compute_units() : 256;
    const int64_t cols = glu ? a.N / 2 : a.N, per = glu ? 16 : 32;
    return a.K >= 2048 && groups * ((cols + per - 1) / per) <= 2 * cus;
}
// max_rows: as in fma_thin_swiglu_experts, or 0 (not known)
template <typename EL, int ROWS>
int launch(const Args& a, bool glu, int64_t R, int64_t groups, int64_t max_rows, hipStream_t st) {
    if constexpr (ROWS == 32) {
        if (!a.taken && max_rows >= 1 && max_rows <= Config<16>::kMaxTokens && half_units(a, glu, groups))
            return launch<EL, 16, ONE_PASS>(a, glu, R, groups, st);
    }
    if (a.taken) return launch<EL, ROWS, MAY_YIELD>(a, glu, R, groups, st);
    if (max_rows >= 1 && max_rows <= Config<ROWS>::kMaxTokens) return launch<EL, ROWS, ONE_PASS>(a, glu, R, groups, st);
    return launch<EL, ROWS, MANY_PASSES>(a, glu, R, groups, st);
}

}  // namespace thin
}  // namespace gemm
}  // namespace fmahip

namespace fmahip {
namespace gemm {
namespace thin {

// ---- one token -------------------------------------------------------------------------------------------------
// A step of one token is bound by its launches: of 41 us (hidden 2048, I 1408, E 64, k 8) the weights need 24, and router logits, top-k
// and index, two products and combine are five kernels that each fill and drain the chip. Each choice is a group of its own here, in the
// order of the choice, so no index is needed: every wavefront of the products reads the top-k off the logits by itself (about as long as
// looking its expert up in the counts took), and the second product's workgroup holds the same 8 columns of all choices, a wavefront
// for two of them, whose rounded results it combines through LDS. Three launches, the same bits. Whole layer, replayed from a graph, us: hidden 2048, I 1408,
// E 64, k 8 39.9 -> 33.0; I 1024 33.7 -> 26.8; hidden 2048, I 768, E 128, k 8 31.4 -> 26.1; hidden 4096, I 1536, E 128, k 8 69.4 -> 62.4; hidden
// 2880, I 2880, E 32, k 4 49.2 -> 44.9; hidden 2048, I 8192, E 8, k 2 65.5 -> 58.9; hidden 4096, I 14336, E 8, k 2 137.5 -> 130.9. With 16
// columns and a wavefront per choice in a workgroup of the second product (128 workgroups for 2048 columns) the first takes 37.8.
constexpr uint32_t kMostChoices = 8;  // two per wavefront of a workgroup of the second product

// The first `rounds` choices of the one token, choice j in lane j of every sixteen; NK = ceil(E / 16) and more keys per lane
template <typename RT, int NK>
__device__ __forceinline__ uint32_t choices(const uint16_t* logits, uint32_t E, uint32_t rounds, uint32_t lane) {
    const uint32_t c = lane & 15u;
    uint32_t keys[NK], mine = 0;
#pragma unroll
    for (int i = 0; i < NK; ++i) {
        const uint32_t n = c + 16u * i;
        keys[i] = n < E ? make_key<RT>(logits[n], (int)n) : 0u;
    }
    for (uint32_t j = 0; j < rounds; ++j) {
        uint32_t best = keys[0];
#pragma unroll
        for (int i = 1; i < NK; ++i) best = max(best, keys[i]);
        best = row16_max(best);  // top_k <= E: a real key, and no two keys are equal
#pragma unroll
        for (int i = 0; i < NK; ++i) keys[i] = keys[i] == best ? 0u : keys[i];
        if (c == j) mine = best;
    }
    return mine;
}
__device__ __forceinline__ uint32_t expert_of_choice(uint32_t mine, uint32_t j) {
    return uniform((uint32_t)key_column((uint32_t)__builtin_amdgcn_readlane((int)mine, (int)j)));
}

// row j of a.out: the activation of the token's first projection by the expert of choice j
template <typename EL, typename RT, int ROWS, int NK, bool BIAS>
__global__ __launch_bounds__(64) void one_token_up_kernel(Args a, const uint16_t* __restrict__ logits) {
    __shared__ __attribute__((aligned(1024))) uint8_t lds[Config<ROWS>::kLds];
    const uint32_t j = blockIdx.x / a.units, u = blockIdx.x - j * a.units;
    const uint32_t e = expert_of_choice(choices<RT, NK>(logits, a.E, j + 1u, threadIdx.x), j);
    a.out += (uint64_t)j * (a.N / 2);
    unit<EL, ROWS, true, BIAS, 1, true>(a, lds, e, 0u, 1u, u * (ROWS / 2));
}

// Columns n0 .. n0 + 7 of the second projection for two choices, rows `x` and the one behind it (rows: how many of them exist), by the experts
// e0 and e1: the sixteen weight rows of a matrix instruction are eight of each expert, and of its sixteen by sixteen results the two
// blocks of eight that belong together are used. Results, rounded, to s_o[0] and s_o[1].
template <typename EL, bool BIAS, int STAGES>
__device__ __forceinline__ void pair_unit(const Args& a, uint8_t* lds, const uint16_t* x, uint32_t rows, uint32_t e0, uint32_t e1, uint32_t n0,
                                          uint16_t (*s_o)[8]) {
    using frag = typename EL::frag;
    constexpr uint32_t kStage = 24 * kKB;  // sixteen weight rows and eight of x
    constexpr int kIPS = 3;
    static_assert(kIPS * (STAGES - 1) < 64, "vmcnt holds six bits");
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t K2 = a.K * 2u, lr = lane >> 3, lp = lane & 7u;
    const uint32_t n_rows = a.N - n0 < 8u ? a.N - n0 : 8u;
    // descriptors end with the rows that exist: the rest arrives as zeros
    const u32x4 rw0 = make_rsrc_words(a.W + ((uint64_t)e0 * a.N + n0) * a.K, n_rows * K2);
    const u32x4 rw1 = make_rsrc_words(a.W + ((uint64_t)e1 * a.N + n0) * a.K, rows > 1u ? n_rows * K2 : 0u);
    const u32x4 rx = make_rsrc_words(x, rows * K2);
    const uint32_t lds0 = lds_address(lds), nsteps = (K2 + kKB - 1) / kKB;
    auto issue = [&](uint32_t s, uint32_t slot) {
        const uint32_t kb = s * kKB;
#pragma unroll
        for (uint32_t i = 0; i < 3u; ++i) {
            const uint32_t chunk = lp ^ flip(i * kRPI + lr);
            const uint32_t v = kb + chunk * 16u < K2 ? lr * K2 + chunk * 16u : kOutOfRange;
            if (i < 2u) load_lds<true>(i ? rw1 : rw0, v, kb, lds0 + slot * kStage + i * 1024u);
            else load_lds<false>(rx, v, kb, lds0 + slot * kStage + 2048u);
        }
    };
    f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (uint32_t d = 0; d + 1 < (uint32_t)STAGES; ++d) issue(d, d);
    const uint32_t r16 = lane & 15u, q = lane >> 4;
    uint32_t slot = 0, fill = STAGES - 1;
    for (uint32_t s = 0; s < nsteps; ++s) {
        wait_lds();  // the stage filled here was read in the previous iteration
        issue(s + STAGES - 1, fill);
        fill = fill == STAGES - 1 ? 0u : fill + 1u;
        wait_vm<kIPS*(STAGES - 1)>();
        const uint8_t* stage = lds + slot * kStage;
        slot = slot == STAGES - 1 ? 0u : slot + 1u;
#pragma unroll
        for (uint32_t sl = 0; sl < 2u; ++sl) {
            const frag w = __builtin_bit_cast(frag, read_kc_frag(stage + lds_off(r16, sl * 4u + q)));
            const frag t = __builtin_bit_cast(frag, read_kc_frag(stage + lds_off(16u + (r16 & 7u), sl * 4u + q)));
            acc = EL::mfma16(w, t, acc);
        }
    }
    wait_vm<0>();
    // a lane holds row r16 of x, weight rows 4 q .. 4 q + 3: row 0 with the first expert's, row 1 with the second's
    const uint32_t c = 4u * (q & 1u);
    if (r16 == q >> 1 && r16 < rows && n0 + c < a.N) {
        float y[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            y[i] = acc[i];
            if constexpr (BIAS) y[i] = EL::round(y[i]) + EL::from_bits(a.bias[(uint64_t)(r16 ? e1 : e0) * a.N + n0 + c + i]);
        }
        *reinterpret_cast<uint2*>(s_o[r16] + c) = uint2{EL::pack2(y[0], y[1]), EL::pack2(y[2], y[3])};
    }
}

// KW: wavefronts of a workgroup, at least one per two choices (a.units of them)
template <typename EL, typename RT, int NK, int KW, bool BIAS>
__global__ __launch_bounds__(64 * KW) void one_token_down_kernel(Args a, const uint16_t* __restrict__ logits) {
    constexpr int kStages = KW > 2 ? 6 : (KW > 1 ? 12 : 16);  // two and more workgroups fit the LDS of a compute unit
    constexpr uint32_t kRing = kStages * 24 * kKB;
    __shared__ __attribute__((aligned(1024))) uint8_t lds[KW * kRing];
    __shared__ __attribute__((aligned(16))) uint16_t s_o[2 * KW][8];
    __shared__ float s_gate[2 * KW];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, p = uniform(tid >> 6), k = a.units, j = 2u * p;
    const uint32_t n0 = blockIdx.x * 8u, rows = k - j < 2u ? k - j : 2u;
    const uint32_t mine = choices<RT, NK>(logits, a.E, p == 0u ? k : j + rows, lane);
    if (p == 0u) {
        // the weights, with the sums of softmax_tokens (router_parts.h)
        const float vmax = key_value<RT>((uint32_t)__builtin_amdgcn_readlane((int)mine, 0));
        const float ex = (lane & 15u) < k ? expf(key_value<RT>(mine) - vmax) : 0.f;
        const float sum = row16_sum(ex);
        if (lane < k) s_gate[lane] = RT::from_bits(RT::bits(ex / sum));
    }
    pair_unit<EL, BIAS, kStages>(a, lds + p * kRing, a.x + (uint64_t)j * a.K, rows, expert_of_choice(mine, j),
                                 expert_of_choice(mine, j + rows - 1u), n0, s_o + j);
    __syncthreads();
    if (tid < 8u && n0 + tid < a.N) {
        float acc = 0.f;
        for (uint32_t i = 0; i < k; ++i) acc = fmaf(s_gate[i], RT::from_bits(s_o[i][tid]), acc);
        a.out[n0 + tid] = RT::bits(acc);
    }
}

template <typename EL, typename RT, int NK, bool BIAS1, bool BIAS2>
int launch_one_token(Args up, Args down, const uint16_t* logits, uint32_t k, hipStream_t st) {
    const uint32_t I = up.N / 2;
    const bool half = half_units(up, true, k);
    up.units = (I + (half ? 7u : 15u)) / (half ? 8u : 16u);
    if (half) hipLaunchKernelGGL((one_token_up_kernel<EL, RT, 16, NK, BIAS1>), dim3(k * up.units), dim3(64), 0, st, up, logits);
    else hipLaunchKernelGGL((one_token_up_kernel<EL, RT, 32, NK, BIAS1>), dim3(k * up.units), dim3(64), 0, st, up, logits);
    const int rc = launch_status("moe_decode (one token, up)");
    if (rc) return rc;
    down.units = k;
    const dim3 grid((down.N + 7u) / 8u), block(64u * ((k + 1u) / 2u));
    if (k <= 2) hipLaunchKernelGGL((one_token_down_kernel<EL, RT, NK, 1, BIAS2>), grid, block, 0, st, down, logits);
    else if (k <= 4) hipLaunchKernelGGL((one_token_down_kernel<EL, RT, NK, 2, BIAS2>), grid, block, 0, st, down, logits);
    else hipLaunchKernelGGL((one_token_down_kernel<EL, RT, NK, 4, BIAS2>), grid, block, 0, st, down, logits);
    return launch_status("moe_decode (one token, down)");
}
template <typename EL, typename RT, int NK>
int launch_one_token(const Args& up, const Args& down, const uint16_t* logits, uint32_t k, hipStream_t st) {
    if (up.bias) return down.bias ? launch_one_token<EL, RT, NK, true, true>(up, down, logits, k, st)
                                  : launch_one_token<EL, RT, NK, true, false>(up, down, logits, k, st);
    return down.bias ? launch_one_token<EL, RT, NK, false, true>(up, down, logits, k, st)
                     : launch_one_token<EL, RT, NK, false, false>(up, down, logits, k, st);
}

// Up to 16 rows per expert on average 32 weight rows per wavefront, beyond that 64. Up / down projection, E 8, k 2, hidden
// 4096, I 14336: 16 rows (64 tokens) 317 / 154 us against 322 / 150 us, 32 rows 466 / 227 against 334 / 167 us; the shape
// with E 128 at 6 rows 506 / 244 against 531 / 250 us, E 64 at one row 16.8 / 9.3 against 18.6 / 11.6 us.
bool wide(int64_t R, int64_t E) { return R > 16 * (R < E ? R : E); }

int check(const char* who, const void* x, int64_t x_rows, const int32_t* row_index, int32_t divisor, const void* W,
          const void* out, const uint32_t* counts, const uint32_t* offsets, int64_t R, int64_t E, int64_t N, int64_t K, int swiglu,
          int dtype) {
    FMA_REQUIRE(dtype == FMA_BF16 || dtype == FMA_F16, dtype_bytes(dtype) ? FMA_ERR_UNSUPPORTED : FMA_ERR_BAD_DTYPE,
                "%s: bf16 and fp16 operands are implemented (dtype code %d)", who, dtype);
    FMA_REQUIRE(E >= 0, FMA_ERR_BAD_SIZE, "%s: negative group count %lld", who, (long long)E);
    FMA_REQUIRE(E <= FMA_MAX_GROUPS, FMA_ERR_TOO_MANY_EXPERTS, "%s: E=%lld exceeds the limit %d", who, (long long)E,
                FMA_MAX_GROUPS);
    FMA_REQUIRE(N >= 8 && N % (swiglu ? 16 : 8) == 0 && N < (1ll << 23), FMA_ERR_BAD_SIZE,
                "%s: N=%lld must be a positive multiple of %d below 2^23", who, (long long)N, swiglu ? 16 : 8);
    FMA_REQUIRE(K >= 8 && K % 8 == 0 && K < (1ll << 21), FMA_ERR_BAD_SIZE,
                "%s: K=%lld must be a positive multiple of 8 below 2^21", who, (long long)K);
    FMA_REQUIRE(R >= 0 && R <= 0x7fffffffll, FMA_ERR_BAD_SIZE, "%s: bad row count %lld", who, (long long)R);
    FMA_REQUIRE(divisor >= 1 && divisor <= 65536, FMA_ERR_BAD_SIZE, "%s: divisor must lie in [1, 65536] (got %d)", who, divisor);
    if (E == 0 || R == 0) return FMA_OK;
    FMA_REQUIRE(x && W && out && counts && offsets, FMA_ERR_NULL_POINTER, "%s: NULL pointer", who);
    // the loads address gathered rows with 32-bit byte offsets below 2^31
    FMA_REQUIRE(!row_index || (x_rows >= 1 && x_rows <= ((1ll << 31) - 1) / (2 * K)), FMA_ERR_UNSUPPORTED,
                "%s: x must have rows and be smaller than 2 GiB (%lld rows of %lld elements)", who, (long long)x_rows,
                (long long)K);
    FMA_REQUIRE(aligned16(x) && aligned16(W) && aligned16(out), FMA_ERR_MISALIGNED, "%s: x, W and out must be 16-byte aligned",
                who);
    return FMA_OK;
}

// a product whose arguments check() has passed
int product(const void* x, int64_t x_rows, const int32_t* row_index, int32_t divisor, const void* W, const void* bias, void* out,
            const uint32_t* counts, const uint32_t* offsets, int64_t R, int64_t max_rows, int64_t E, int64_t N, int64_t K,
            int swiglu, const uint32_t* taken, int dtype, hipStream_t st) {
    if (E == 0 || R == 0) return FMA_OK;
    Args a{};
    a.x = (const uint16_t*)x;
    a.row_index = row_index;
    a.W = (const uint16_t*)W;
    a.bias = (const uint16_t*)bias;
    a.out = (uint16_t*)out;
    a.counts = counts;
    a.offsets = offsets;
    a.E = (uint32_t)E;
    a.N = (uint32_t)N;
    a.K = (uint32_t)K;
    a.divisor = (uint32_t)divisor;
    a.x_rows = row_index ? (uint32_t)x_rows : 0u;
    a.taken = taken;
    const int64_t groups = R < E ? R : E;  // no more experts than rows can have rows
    const bool w = wide(R, E), glu = swiglu != 0;
    if (dtype == FMA_BF16) return w ? launch<ElemBf16, 64>(a, glu, R, groups, max_rows, st) : launch<ElemBf16, 32>(a, glu, R, groups, max_rows, st);
    return w ? launch<ElemF16, 64>(a, glu, R, groups, max_rows, st) : launch<ElemF16, 32>(a, glu, R, groups, max_rows, st);
}

// The expert path of one token (decode.hip)
bool takes_one_token(int64_t T, int64_t top_k) { return T == 1 && top_k <= (int64_t)kMostChoices; }
int one_token(const void* x, const void* logits, const void* W1, const void* bias1, const void* W2, const void* bias2, void* act, void* y,
              int64_t E, int64_t H, int64_t I, int64_t top_k, int dtype, hipStream_t st) {
    Args up{}, down{};
    up.x = (const uint16_t*)x;
    up.W = (const uint16_t*)W1;
    up.bias = (const uint16_t*)bias1;
    up.out = (uint16_t*)act;
    up.N = (uint32_t)(2 * I);
    up.K = (uint32_t)H;
    down.x = (const uint16_t*)act;
    down.W = (const uint16_t*)W2;
    down.bias = (const uint16_t*)bias2;
    down.out = (uint16_t*)y;
    down.N = (uint32_t)H;
    down.K = (uint32_t)I;
    up.E = down.E = (uint32_t)E;
    up.divisor = down.divisor = 1;
    const uint16_t* l = (const uint16_t*)logits;
    const uint32_t k = (uint32_t)top_k;
    if (dtype == FMA_BF16) return E <= 64 ? launch_one_token<ElemBf16, RouterBf16, 4>(up, down, l, k, st) : launch_one_token<ElemBf16, RouterBf16, 16>(up, down, l, k, st);
    return E <= 64 ? launch_one_token<ElemF16, RouterF16, 4>(up, down, l, k, st) : launch_one_token<ElemF16, RouterF16, 16>(up, down, l, k, st);
}

}  // namespace thin
}  // namespace gemm
}  // namespace fmahip

extern "C" {

int fma_grouped_gemm_thin(const void* x, int64_t x_rows, const int32_t* row_index, int32_t divisor, const void* W,
                          const void* bias, void* out, const uint32_t* counts, const uint32_t* offsets, int64_t R, int64_t E,
                          int64_t N, int64_t K, int swiglu, int dtype, void* stream) {
    using namespace fmahip::gemm;
    const int rc = thin::check("grouped_gemm_thin", x, x_rows, row_index, divisor, W, out, counts, offsets, R, E, N, K, swiglu, dtype);
    if (rc) return rc;
    return thin::product(x, x_rows, row_index, divisor, W, bias, out, counts, offsets, R, 0, E, N, K, swiglu, nullptr, dtype,
                         (hipStream_t)stream);
}

int64_t fma_thin_swiglu_experts_workspace_bytes(int64_t R, int64_t I) {
    return R < 0 || I < 0 ? 0 : (2 * R * I + 255) / 256 * 256 + 16;  // the activation, the tile kernel's word
}

int fma_thin_swiglu_experts(const void* x, int64_t x_rows, const int32_t* row_index, int32_t divisor, const void* W1,
                            const void* bias1, const void* W2, const void* bias2, void* out, const uint32_t* counts,
                            const uint32_t* offsets, int64_t R, int64_t max_rows, int64_t E, int64_t H, int64_t I,
                            void* workspace, int64_t workspace_bytes, int dtype, void* stream) {
    using namespace fmahip;
    using namespace fmahip::gemm;
    const char* who = "thin_swiglu_experts";
    FMA_REQUIRE((workspace != nullptr && aligned16(workspace)) || E == 0 || R == 0, FMA_ERR_MISALIGNED,
                "%s: the workspace must be 16-byte aligned", who);
    FMA_REQUIRE(workspace_bytes >= fma_thin_swiglu_experts_workspace_bytes(R, I) || E == 0 || R == 0, FMA_ERR_WORKSPACE_TOO_SMALL,
                "%s: workspace of %lld bytes is smaller than the %lld needed", who, (long long)workspace_bytes,
                (long long)fma_thin_swiglu_experts_workspace_bytes(R, I));
    void* act = workspace;
    uint32_t* taken = (uint32_t*)((uint8_t*)workspace + (2 * R * I + 255) / 256 * 256);
    int rc = thin::check(who, x, x_rows, row_index, divisor, W1, act, counts, offsets, R, E, 2 * I, H, 1, dtype);
    if (!rc) rc = thin::check(who, act, R, nullptr, 1, W2, out, counts, offsets, R, E, H, I, 0, dtype);
    if (rc || E == 0 || R == 0) return rc;
    // Where an expert can take more than four passes, the tile kernel is enqueued in front of both products. Few experts with many
    // rows each are its case, and how many there are is known on the device only: it decides, once, and whichever kernel the
    // products do not fall to ends at once. A bias that it cannot address leaves them here.
    // Whole layer, us: the tile kernel / this kernel alone / the choice (k 8, all tokens on the same 8, 16 or 32 experts, or evenly):
    //   hidden 4096, I 1536, E 128, 256 tokens:   8: 237 / 337 / 248   16: 253 / 386 / 265   32: 396 / 465 / 411   even: 978 / 870 / 872
    //   hidden 4096, I 1536, E 128, 512 tokens:   8: 235 / 386 / 244   16: 387 / 443 / 396   32: 417 / 506 / 427   even: 999 / 943 / 945
    //   hidden 2048, I 768, E 256, 1024 tokens:   8: 178 / 280 / 189   16: 206 / 302 / 214   32: 267 / 315 / 277   even: 596 / 568 / 574
    //   hidden 2048, I 768, E 256, 192 tokens:    8: 151 / 140 / 176   16: 166 / 161 / 176   32: 161 / 186 / 173   even: 578 / 467 / 473
    // One or two experts in every token's choice and the rest even stay here (1.1 passes per expert): 1025 / 916 / 916 in the first
    // line. Up to four passes this kernel takes at most 1.09 times the tile kernel's time on any of these routings (16 experts, E 64, 256
    // tokens).
    const uint32_t pass_bits = thin::wide(R, E) ? 6u : 5u;
    const bool bias_ok = ((reinterpret_cast<uintptr_t>(bias1) | reinterpret_cast<uintptr_t>(bias2)) & 3u) == 0;
    if (max_rows <= (4ll << pass_bits) || !bias_ok) taken = nullptr;
    hipStream_t st = (hipStream_t)stream;
    if (taken)
        rc = ragged::up_projection(who, x, x_rows, row_index, divisor, W1, bias1, nullptr, act, counts, E, 2 * I, H, 1, dtype, st,
                                   taken, pass_bits);
    if (!rc) rc = thin::product(x, x_rows, row_index, divisor, W1, bias1, act, counts, offsets, R, max_rows, E, 2 * I, H, 1, taken, dtype,
                               st);
    if (!rc && taken)
        rc = ragged::up_projection(who, act, R, nullptr, 1, W2, bias2, out, nullptr, counts, E, H, I, 0, dtype, st, taken, 0);
    return rc ? rc : thin::product(act, R, nullptr, 1, W2, bias2, out, counts, offsets, R, max_rows, E, H, I, 0, taken, dtype, st);
}

}  // extern "C"
