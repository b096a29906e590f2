// The choice and the second pass of a split reduction (the kernel: ragged_kernel.h).
#include <algorithm>
#include <cmath>

#include "ragged_kernel.h"

namespace fmahip {
namespace gemm {
namespace ragged {

// ---- split reduction ---------------------------------------------------------------------------------------------
// A launch with fewer tiles than compute units leaves the others idle for the whole reduction: the second projection of 800 tokens on
// 8 experts (2048 x 8192) is 64 tiles of 128 K steps, 184 us. With the reduction in three parts (192 units of 44 steps, fp32 sums to
// memory and one pass over them) it takes 94 us. More of the same, 8 groups, randomly routed (unsplit -> parts):
//   NT 2048 x 8192, 150 / 256 / 400 / 512 rows a group       157 -> 86 us (3), 172 -> 106 us (3), 175 -> 121 us (2), 193 -> 149 us (2)
//   NT 4096 x 14336, 100 / 200 / 600 rows                    265 -> 191 us (2), 330 -> 227 us (2), 605 -> 571 us (2)
//   NN 2048 x 16384, 150 / 256 / 400 / 512 rows              234 -> 129 us (4), 276 -> 175 us (3), 291 -> 214 us (2), 332 -> 247 us (2)
//   NN 4096 x 28672, 100 / 256 rows                          380 -> 320 us (2), 619 -> 440 us (4)
//
// How many parts: the number with the least predicted time, rounds of tiles times (K steps + a tile's fixed cost) or the
// weights at the rate they stream, plus the traffic of the sums. The row counts lie in device memory, so the number of tiles
// is the expected one for evenly loaded groups. Parts have at least kSplitMinSteps steps, the sums at most kSplitMaxBytes (they
// stay in the last-level cache), and a split has to promise a twentieth less than none. Groups of few rows run the three-stage
// loop, whose steps are shorter, without a split on half-width tiles in the NT layout: NT 4096 x 14336 on 8 groups of 24 rows
// streams its weights in 175 us as it is and would take 197 us in two parts.
// Tall tiles (TALL in ragged_kernel.h): a round takes 1.6 to 2.0 us per K step of its tiles, most when every compute unit is busy and
// streams weights of its own, and a partial last round costs what rounds_of there says. The tiles of a group follow from the spread of a
// random routing (a standard deviation of the root of the mean): 8 groups of 256 or 512 rows are 8 or 16 tiles high, not 12 or 20. That
// ends the split of [8 x 512 rows, 4096 x 14336] (370 us, two parts 432).
// Routings are less even than random ones, too, and what fills the compute units exactly once is worth little if one more row tile spoils
// it: where a group of 2.5 times the mean rows has a second tile, one launch in five (kUneven) is taken to have one. 8 groups of 200 rows,
// 2048 x 8192 and 2048 x 16384 in four parts (256 units) take 101 and 146 us, but with odds of the experts as their rank to the -0.7 (9 row
// tiles) 135 and 216; in three parts 93 and 157, 88 and 149. Over 210 launches (seven shapes of 4 to 32 groups, 24 to 1000 rows a group,
// a random and such an uneven routing, one draw of each) the parts taken cost 1.6 % (random) and 6.4 % (uneven) more than the best number
// would; without the line 1.4 and 9.2 %. A fifth more or less of any constant moves that by less than 1 and 3 %, as another draw does. What the
// constants miss: with few rows the half-width tiles of no split take 0.6 us a step, the whole ones of parts 1.15, so that 8 groups of 24 or 48
// rows, NT 2048 x 8192, run in three parts (69 and 72 us) and not in four (58 and 60).
constexpr double kStepUs = 1.45, kTallStepUs = 1.55, kFullStepUs = 0.4, kThinStepUs[2] = {1.1, 0.75}, kTileSteps = 6.0, kThinRows = 48.0;
constexpr double kTailCost = 0.87, kLoneTailCost = 0.85, kUneven = 0.2, kWeightBytesPerUs = 5.5e6;
constexpr double kReduceUs = 4.0, kReduceBytesPerUs = 4.5e6, kSplitGain[2] = {0.9, 0.95};  // [tall]
constexpr uint32_t kSplitMinSteps = 24;
constexpr int64_t kSplitMaxBytes = 256ll << 20;
SplitPlan plan_split(int64_t R, int64_t E, int64_t N, int64_t K, bool b_kc, bool tall) {
    const uint32_t all = (uint32_t)((K + BK - 1) / BK);
    SplitPlan best{1u, all};
    // (the sizes for which every tile takes the matrix-instruction path)
    if (R < 1 || E < 1 || N < 8 || N % 8 || N >= (1 << 23) || K % 8 || K >= (1 << 21) || R > 0x7fffffffll) return best;
    if (all < 2 * kSplitMinSteps) return best;
    const int cus = num_compute_units() > 0 ? num_compute_units() : 256;
    const double active = (double)(R < E ? R : E), mean = (double)R / active;
    const bool thin = mean <= kThinRows;
    double row_tiles = active * (mean < BM / 2 ? 1.0 : mean / BM + 0.5);
    if (tall) {
        // about a boundary b of kTallM rows, the share of the groups past it is that of a normal distribution
        const double b = std::max(1.0, std::floor(mean / kTallM + 0.5));
        const double past = 0.5 * std::erfc((b * kTallM - mean) / std::sqrt(2.0 * mean));
        row_tiles = active * (b + past);
    }
    const double columns = (double)((N + BN - 1) / BN);
    const double weights_us = active * N * K * 2.0 / kWeightBytesPerUs;
    auto us_of = [&](double tiles, uint32_t parts, uint32_t steps) {
        const bool narrow = thin && b_kc && 2.0 * tiles <= cus;
        const double units = tiles * parts * (parts == 1 && narrow ? 2.0 : 1.0);
        double rounds = std::ceil(units / cus - 1e-9);
        const double whole = std::floor(units / cus), rest = units - whole * cus;
        double step_us = thin ? kThinStepUs[b_kc] : kStepUs;
        if (tall && !thin) {
            const bool in_parts = parts == 1 && rest > 0.5 && 2.0 * rest <= cus && (whole > 0.0 || !b_kc);
            if (in_parts) rounds = whole + (whole > 0.0 ? kTailCost : kLoneTailCost);
            step_us = kTallStepUs + (in_parts ? kFullStepUs : kFullStepUs * std::min(1.0, units / cus));
        }
        const double products = rounds * (steps + kTileSteps) * step_us;
        const double sums = parts > 1 ? kReduceUs + (double)R * N * (8.0 * parts + 2.0) / kReduceBytesPerUs : 0.0;
        return std::max(products, weights_us) + sums;
    };
    // tall: between the two numbers of row tiles about the expected one, by how likely they are
    const double low = tall ? std::floor(row_tiles) : row_tiles, uneven = tall && !thin && mean * 2.5 > kTallM ? kUneven : 0.0;
    const double more = std::max(row_tiles - low, uneven);
    auto us = [&](uint32_t parts, uint32_t steps) {
        const double t = us_of(low * columns, parts, steps);
        return more > 0.0 ? (1.0 - more) * t + more * us_of((low + 1.0) * columns, parts, steps) : t;
    };
    double best_us = us(1, all) * kSplitGain[tall];
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

int launch_split_reduce(const Args& args, bool bf16, hipStream_t st) {
    const dim3 grid((args.rows + kReduceRows - 1) / kReduceRows), block(kReduceThreads);
    if (bf16 && args.bias) hipLaunchKernelGGL((split_reduce_kernel<ElemBf16, true>), grid, block, 0, st, args);
    else if (bf16) hipLaunchKernelGGL((split_reduce_kernel<ElemBf16, false>), grid, block, 0, st, args);
    else if (args.bias) hipLaunchKernelGGL((split_reduce_kernel<ElemF16, true>), grid, block, 0, st, args);
    else hipLaunchKernelGGL((split_reduce_kernel<ElemF16, false>), grid, block, 0, st, args);
    return launch_status("grouped_gemm_ragged(reduce)");
}

}  // namespace ragged
}  // namespace gemm
}  // namespace fmahip
