// Grouped GEMM for fp32 operands: D_e = alpha * op(A_e) op(B_e) on the fp32 matrix instruction (v_mfma_f32_32x32x2_f32,
// 157 TFLOP/s peak: one sixteenth of the bf16 rate, so a large product is bound by the matrix pipe long before memory, and a small
// one, which an fp32 layer mostly is, by the number of tiles and the latency of a K step).
// Four wavefronts (2 x 2) on output tiles of 128 x 128 with 16-wide K steps, or, where those are too few to fill the compute units,
// 64 x 64 with 32-wide steps: four times the tiles and half the steps. Operands of any M, N, K and either storage order (rows past a
// group's edge and K past its end read as zero) are fetched two K steps ahead into registers, four consecutive k of a row at a time
// (one 16-byte load where the reduction is contiguous and a multiple of 4), and staged in LDS as [row][k] with rows padded by 4 floats,
// double-buffered with one barrier per K step: 16-byte LDS accesses without bank conflicts in either storage order. The instruction
// multiplies two k values at a time (lane half h supplies one of them); since the order of a sum's terms is free, half h takes one
// half of the step's k, so a lane's values of a fragment are contiguous in LDS.
// Workgroups are persistent and find their tiles in a per-workgroup prefix table of the groups' tile counts, like the
// 16-bit kernel.
// Against 128 x 128 tiles alone, fetched and staged element by element (us; layer of hidden 256, I 512, E 8, k 2, 512 tokens): up 30 ->
// 17, down 50 -> 18, input gradients 102 -> 38 and 31 -> 13, weight gradients 23 -> 16 and 22 -> 11; hidden 2048, I 4096, 4096 tokens
// (large tiles): 2660 -> 2377, 1521 -> 1379, 3415 -> 3030, 1533 -> 1398, 2680 -> 2669, 1346 -> 1339 (116 TFLOP/s).
#include <type_traits>

#include "common.h"
#include "grouped_gemm_f32.h"

namespace fmahip {
namespace gemm_f32 {
namespace {

typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(16))) float f32x16;

constexpr int kThreads = 256;

struct Args {
    const float* A;
    const float* B;
    float* D;
    const uint32_t* M_arr;
    const uint32_t* N_arr;
    const uint32_t* K_arr;
    uint32_t E;
    float alpha;
};

// The group table: first tile and operand offsets of every group
struct Table {
    uint32_t tile_start[FMA_MAX_GROUPS + 1];
    uint64_t off_a[FMA_MAX_GROUPS], off_b[FMA_MAX_GROUPS], off_d[FMA_MAX_GROUPS];
};

// Tiles of S x S outputs, K steps of BK. An operand tile is S rows of BK / 4 quads (four consecutive k), two per thread.
template <int S_, int BK_>
struct Shape {
    static constexpr int S = S_, BK = BK_;
    static constexpr int kPitch = BK + 4;            // floats per LDS row
    static constexpr int kQuads = BK / 4;            // of a row
    static constexpr int kBlocks = S / 64;           // 32 x 32 blocks per wavefront and direction
    static constexpr int kTileFloats = S * kPitch;   // LDS of an operand and stage
    static_assert(S * kQuads == 2 * kThreads, "two quads per thread, operand and K step");
};
using Large = Shape<128, 16>;
using Small = Shape<64, 32>;

// Row and first k of quad g of this thread: consecutive threads walk the operand's contiguous dimension. K_CONTIG: stored [rows, K];
// otherwise stored [K, rows].
template <bool K_CONTIG, typename SH>
__device__ __forceinline__ void quad_of(int g, int tid, uint32_t& row, uint32_t& k) {
    const int q = tid + g * kThreads;
    if constexpr (K_CONTIG) {
        row = q / SH::kQuads;
        k = q % SH::kQuads * 4;
    } else {
        k = q / SH::S * 4;
        row = q % SH::S;
    }
}

// Requests the thread's quads of the operand tile at (row0, k0). Elements outside the operand are requested from
// its first element instead (a valid address: a tile exists only if M, N >= 1, a K step only if K >= 1) and replaced by
// zeros in stage(): nothing here consumes a loaded value, so the loads stay in flight until the data is needed.
// VEC: the quads of a K_CONTIG operand are whole and aligned (K and the operand's offset multiples of 4).
template <bool K_CONTIG, bool VEC, typename SH>
__device__ __forceinline__ void fetch(float4 (&regs)[2], const float* __restrict__ base, uint32_t rows, uint32_t K, uint32_t row0,
                                      uint32_t k0, int tid) {
#pragma unroll
    for (int g = 0; g < 2; ++g) {
        uint32_t r, k;
        quad_of<K_CONTIG, SH>(g, tid, r, k);
        const uint32_t row = row0 + r, kk = k0 + k;
        if constexpr (K_CONTIG && VEC) {
            const bool in = row < rows && kk < K;
            regs[g] = *reinterpret_cast<const float4*>(base + (in ? (uint64_t)row * K + kk : 0u));
        } else {
            float v[4];
#pragma unroll
            for (int x = 0; x < 4; ++x) {
                const bool in = row < rows && kk + x < K;
                const uint64_t idx = K_CONTIG ? (uint64_t)row * K + kk + x : (uint64_t)(kk + x) * rows + row;
                v[x] = base[in ? idx : 0u];
            }
            regs[g] = float4{v[0], v[1], v[2], v[3]};
        }
    }
}

template <bool K_CONTIG, typename SH>
__device__ __forceinline__ void stage(const float4 (&regs)[2], float* __restrict__ tile, uint32_t rows, uint32_t K, uint32_t row0,
                                      uint32_t k0, int tid) {
#pragma unroll
    for (int g = 0; g < 2; ++g) {
        uint32_t r, k;
        quad_of<K_CONTIG, SH>(g, tid, r, k);
        const bool in = row0 + r < rows;
        const uint32_t kk = k0 + k;
        float4 v;
        v.x = in && kk < K ? regs[g].x : 0.0f;
        v.y = in && kk + 1u < K ? regs[g].y : 0.0f;
        v.z = in && kk + 2u < K ? regs[g].z : 0.0f;
        v.w = in && kk + 3u < K ? regs[g].w : 0.0f;
        *reinterpret_cast<float4*>(tile + r * SH::kPitch + k) = v;
    }
}

// The workgroup's tiles. lds: two stages of both operands.
template <bool A_KC, bool B_KC, typename SH>
__device__ __forceinline__ void run(const Args& args, const Table& table, float* __restrict__ lds, uint32_t total) {
    constexpr int S = SH::S, BK = SH::BK, NB = SH::kBlocks, kHalf = BK / 2;
    float* const s_a[2] = {lds, lds + SH::kTileFloats};
    float* const s_b[2] = {lds + 2 * SH::kTileFloats, lds + 3 * SH::kTileFloats};
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave >> 1, wn = wave & 1;  // 2 x 2 wavefronts of S / 2 x S / 2

    for (uint32_t tile = blockIdx.x; tile < total; tile += gridDim.x) {
        // the group of this tile: last e with tile_start[e] <= tile (empty groups share their start with the next)
        uint32_t lo = 0, hi = args.E;
        while (hi - lo > 1) {
            const uint32_t mid = (lo + hi) >> 1;
            if (table.tile_start[mid] <= tile) lo = mid;
            else hi = mid;
        }
        while (table.tile_start[lo + 1] <= tile) ++lo;  // skip groups without tiles
        const uint32_t e = lo;
        const uint32_t Me = args.M_arr[e], Ne = args.N_arr[e], Ke = args.K_arr[e];
        const uint32_t tiles_n = (Ne + S - 1) / S;
        const uint32_t local = tile - table.tile_start[e];
        const uint32_t m0 = (local / tiles_n) * S, n0 = (local % tiles_n) * S;
        const float* Ae = args.A + table.off_a[e];
        const float* Be = args.B + table.off_b[e];
        float* De = args.D + table.off_d[e];
        const bool vec = ((Ke | (A_KC ? (uint32_t)table.off_a[e] : 0u) | (B_KC ? (uint32_t)table.off_b[e] : 0u)) & 3u) == 0;

        f32x16 acc[NB][NB];
#pragma unroll
        for (int i = 0; i < NB; ++i)
#pragma unroll
            for (int j = 0; j < NB; ++j)
#pragma unroll
                for (int x = 0; x < 16; ++x) acc[i][j][x] = 0.0f;

        const uint32_t KT = (Ke + BK - 1) / BK;
        // two register sets: set s holds the operands of the steps with kt % 2 == s, fetched two steps before their use
        float4 ra[2][2], rb[2][2];
        auto compute = [&](int buf) {
            // lane l: row (l % 32) of a 32-row block, one half of the step's k values
            const float* ta = s_a[buf] + (wm * (S / 2) + (lane & 31)) * SH::kPitch + (lane >> 5) * kHalf;
            const float* tb = s_b[buf] + (wn * (S / 2) + (lane & 31)) * SH::kPitch + (lane >> 5) * kHalf;
#pragma unroll
            for (int q = 0; q < kHalf / 4; ++q) {
                float4 fa[NB], fb[NB];
#pragma unroll
                for (int i = 0; i < NB; ++i) {
                    fa[i] = *reinterpret_cast<const float4*>(ta + i * 32 * SH::kPitch + q * 4);
                    fb[i] = *reinterpret_cast<const float4*>(tb + i * 32 * SH::kPitch + q * 4);
                }
#pragma unroll
                for (int x = 0; x < 4; ++x) {
                    // B first: a lane then owns one output row and four consecutive output columns per register quad
#pragma unroll
                    for (int i = 0; i < NB; ++i)
#pragma unroll
                        for (int j = 0; j < NB; ++j)
                            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(reinterpret_cast<const float*>(&fb[j])[x],
                                                                             reinterpret_cast<const float*>(&fa[i])[x], acc[i][j], 0, 0, 0);
                }
            }
        };
        auto k_loop = [&](auto vec_c) __attribute__((always_inline)) {
            constexpr bool VEC = decltype(vec_c)::value;
            fetch<A_KC, VEC, SH>(ra[0], Ae, Me, Ke, m0, 0, tid);
            fetch<B_KC, VEC, SH>(rb[0], Be, Ne, Ke, n0, 0, tid);
            fetch<A_KC, VEC, SH>(ra[1], Ae, Me, Ke, m0, BK, tid);  // past the end of K: zeros
            fetch<B_KC, VEC, SH>(rb[1], Be, Ne, Ke, n0, BK, tid);
            __syncthreads();  // the previous tile is done with the LDS stages
            stage<A_KC, SH>(ra[0], s_a[0], Me, Ke, m0, 0, tid);
            stage<B_KC, SH>(rb[0], s_b[0], Ne, Ke, n0, 0, tid);
            __syncthreads();
            for (uint32_t kt = 0; kt < KT; kt += 2) {
#pragma unroll
                for (int ph = 0; ph < 2; ++ph) {
                    // step kt + ph (a step past the last one multiplies zeros): request step + 2 into the set this step's
                    // operands came from, multiply from stage ph, move step + 1 from its registers to the other stage
                    fetch<A_KC, VEC, SH>(ra[ph], Ae, Me, Ke, m0, (kt + ph + 2) * BK, tid);
                    fetch<B_KC, VEC, SH>(rb[ph], Be, Ne, Ke, n0, (kt + ph + 2) * BK, tid);
                    compute(ph);
                    stage<A_KC, SH>(ra[ph ^ 1], s_a[ph ^ 1], Me, Ke, m0, (kt + ph + 1) * BK, tid);
                    stage<B_KC, SH>(rb[ph ^ 1], s_b[ph ^ 1], Ne, Ke, n0, (kt + ph + 1) * BK, tid);
                    __syncthreads();  // stage ph^1 is complete; stage ph may be overwritten in the next step
                }
            }
        };
        // (two loops, not a look per load: a branch around loads makes the compiler wait for them where it ends)
        if (KT > 0) {
            if (vec && (A_KC || B_KC)) k_loop(std::true_type{});
            else k_loop(std::false_type{});
        }

        // accumulator register 4 q + j of block (i, j'): row m = ... + (lane % 32), column n = ... + 8 q + 4 (lane / 32) + j
        const float alpha = args.alpha;
#pragma unroll
        for (int i = 0; i < NB; ++i) {
            const uint32_t m = m0 + wm * (S / 2) + i * 32 + (lane & 31);
            if (m >= Me) continue;
#pragma unroll
            for (int j = 0; j < NB; ++j) {
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const uint32_t n = n0 + wn * (S / 2) + j * 32 + q * 8 + (lane >> 5) * 4;
                    float* dst = De + (uint64_t)m * Ne + n;
                    if (n + 3 < Ne && (reinterpret_cast<uintptr_t>(dst) & 15u) == 0) {
                        // (one value of a vector type: of four floats the compiler sank the last one's store into the other branch's,
                        // a 12- and a 4-byte store for each of these)
                        *reinterpret_cast<f32x4*>(dst) = f32x4{alpha * acc[i][j][q * 4 + 0], alpha * acc[i][j][q * 4 + 1],
                                                               alpha * acc[i][j][q * 4 + 2], alpha * acc[i][j][q * 4 + 3]};
                    } else {
#pragma unroll
                        for (int x = 0; x < 4; ++x)
                            if (n + x < Ne) dst[x] = alpha * acc[i][j][q * 4 + x];
                    }
                }
            }
        }
    }
}

template <bool A_KC, bool B_KC>
__global__ __launch_bounds__(kThreads) void grouped_gemm_f32_kernel(const Args args) {
    static_assert(Small::kTileFloats <= Large::kTileFloats, "one LDS buffer for both");
    __shared__ __attribute__((aligned(16))) float s_tiles[4 * Large::kTileFloats];
    __shared__ Table table;
    __shared__ uint32_t s_total[2];  // tiles, and whether they are small

    if (threadIdx.x < 64) {
        // wavefront 0: how many large tiles there are, then the prefixes
        const uint32_t lane = threadIdx.x;
        auto tiles_of = [](uint64_t M, uint64_t N, uint32_t S) { return (uint32_t)(((M + S - 1) / S) * ((N + S - 1) / S)); };
        uint32_t n_large = 0, n_small = 0;
        float k_sum = 0.0f;  // of the large tiles' reductions
        for (uint32_t e = lane; e < args.E; e += 64) {
            const uint32_t t = tiles_of(args.M_arr[e], args.N_arr[e], Large::S);
            n_large += t;
            k_sum += (float)t * (float)args.K_arr[e];
            n_small += tiles_of(args.M_arr[e], args.N_arr[e], Small::S);
        }
#pragma unroll
        for (int d = 32; d > 0; d >>= 1) {
            n_large += (uint32_t)__shfl_xor((int)n_large, d, 64);
            n_small += (uint32_t)__shfl_xor((int)n_small, d, 64);
            k_sum += __shfl_xor(k_sum, d, 64);
        }
        // The compute unit with the most tiles ends last. A large tile takes as long as 48 more k of its reduction on top of that, a small
        // one a little less than a third, and of the fixed part not much less than a half: 256 large tiles, one per compute unit, beat 1024
        // small ones by 5 to 20 % over long reductions (39 against 41 us, 19 against 23), 272 lose by a quarter (347 against 256 us); over 7 to
        // 30 rows weight gradients [576, 576] of 8, 64 and 100 experts take 12, 41 and 57 us on large tiles and 14, 63 and 97 on
        // small ones. Over 420 products of all kinds (1 to 200 groups, reductions of 1 to 4096) the tiles taken cost 0.4 % more than the
        // better ones; a third whatever the reduction cost 1.5 %, and up to 1.6 times what large tiles alone had.
        // (every workgroup forms the same sums in the same order: all of them choose alike)
        const uint32_t cus = gridDim.x / 2u;
        const float k_mean = k_sum / (float)(n_large > 0u ? n_large : 1u);
        const bool small = (float)((n_small + cus - 1) / cus) * (20.0f + 0.31f * k_mean) < (float)((n_large + cus - 1) / cus) * (48.0f + k_mean);
        uint32_t tiles = 0;
        uint64_t oa = 0, ob = 0, od = 0;
        for (uint32_t base = 0; base < args.E; base += 64) {
            const uint32_t e = base + lane;
            const bool in = e < args.E;
            const uint64_t M = in ? args.M_arr[e] : 0u, N = in ? args.N_arr[e] : 0u, K = in ? args.K_arr[e] : 0u;
            const uint32_t t = tiles_of(M, N, small ? Small::S : Large::S);
            const uint32_t it = wave_inclusive_scan<uint32_t>(t);
            const uint64_t ia = wave_inclusive_scan<uint64_t>(M * K), ib = wave_inclusive_scan<uint64_t>(K * N);
            const uint64_t id = wave_inclusive_scan<uint64_t>(M * N);
            if (in) {
                table.tile_start[e] = tiles + it - t;
                table.off_a[e] = oa + ia - M * K;
                table.off_b[e] = ob + ib - K * N;
                table.off_d[e] = od + id - M * N;
            }
            tiles += __shfl(it, 63, 64);
            oa += __shfl(ia, 63, 64);
            ob += __shfl(ib, 63, 64);
            od += __shfl(id, 63, 64);
        }
        if (lane == 0) {
            table.tile_start[args.E] = tiles;
            s_total[0] = tiles;
            s_total[1] = small ? 1u : 0u;
        }
    }
    __syncthreads();
    if (s_total[1]) run<A_KC, B_KC, Small>(args, table, s_tiles, s_total[0]);
    else run<A_KC, B_KC, Large>(args, table, s_tiles, s_total[0]);
}

}  // namespace

int launch(const void* A, const void* B, void* D, const uint32_t* M_arr, const uint32_t* N_arr, const uint32_t* K_arr,
           int64_t E, bool a_kc, bool b_kc, float alpha, hipStream_t st) {
    Args args;
    args.A = (const float*)A;
    args.B = (const float*)B;
    args.D = (float*)D;
    args.M_arr = M_arr;
    args.N_arr = N_arr;
    args.K_arr = K_arr;
    args.E = (uint32_t)E;
    args.alpha = alpha;
    const int cus = num_compute_units() > 0 ? num_compute_units() : 256;
    const dim3 grid((uint32_t)(2 * cus)), block(kThreads);
    if (a_kc && b_kc) hipLaunchKernelGGL((grouped_gemm_f32_kernel<true, true>), grid, block, 0, st, args);
    else if (a_kc) hipLaunchKernelGGL((grouped_gemm_f32_kernel<true, false>), grid, block, 0, st, args);
    else if (b_kc) hipLaunchKernelGGL((grouped_gemm_f32_kernel<false, true>), grid, block, 0, st, args);
    else hipLaunchKernelGGL((grouped_gemm_f32_kernel<false, false>), grid, block, 0, st, args);
    return launch_status("grouped_gemm (fp32)");
}

}  // namespace gemm_f32
}  // namespace fmahip
