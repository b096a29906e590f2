// Grouped GEMM for launches whose groups differ in ONE dimension (every grouped GEMM of an MoE layer: rows per expert
// in forward and input gradient, reduction length per expert in the weight gradient) for gfx950: bf16 or fp16 operands,
// fp32 accumulation on the matrix cores, optional SwiGLU epilogue. The tile kernel of grouped_gemm.hip (256x256x64
// tiles, eight wavefronts, two LDS stages filled by direct global -> LDS loads, the same LDS layouts) with another
// matrix instruction and a different tile boundary:
//
//  * The products are 16x16x32 instructions (v_mfma_f32_16x16x32), not 32x32x16: the same arithmetic rate per
//    instruction cycle, but the part holds a higher clock on them. Measured on N(0,1) operands: a loop of nothing but
//    matrix instructions sustains 0.79 of the peak rate against 0.70, and this kernel ran 3.5 to 6 % faster on the
//    Mixtral-shape layer's GEMMs than the same kernel on 32x32x16. A wavefront's 128 x 64 sub-tile is 8 x 4 blocks; a K
//    step is two 32-wide slices, each worked through in four phases of two row blocks (see the K loop).
//  * With two dimensions known on the host, a group's operand offsets follow from one 32-bit prefix of the varying
//    dimension, so the group table takes 10 bytes per group instead of 30. The LDS that frees (16 KB) is a staging
//    buffer of its own for the epilogue, which therefore no longer needs a piece of an operand stage.
//  * The operand loads run as ONE stream over the tile sequence: the load slots of a tile's last two K steps carry the
//    first two K steps of the NEXT tile (the loaders of both tiles are kept, a scalar select picks one per step), so that
//    when a tile's K loop ends the next tile's first step is already in LDS and its second on the way. The tile boundary
//    is then the epilogue alone: no loader set-up, no burst of 16 loads per wavefront competing with the 16 stores for the
//    compute unit's one address path, no wait for first operands, no barrier. (Nothing more is requested while it lasts, from the
//    last step's loads to where the next tile's first step has freed its stage.)
//  * The epilogue's stores stay outstanding across the start of the next tile: they are issued after that tile's first
//    loads, and loads and stores of a wavefront complete in issue order, so the first K step waits for "all but the
//    stores and its own newest loads" (an exact count) and the second for everything older than its own loads.
//  * A K step has two barriers. Behind the first, in the middle of its fifth phase, the step's LDS stage is free (all its fragments have been
//    read) and the loads of step kt + 2 begin; the second, in the middle of the eighth, is where step kt + 1 has to have landed, and
//    leaves the four loads behind the first outstanding. One barrier for both, as there was, waits for every load in flight, so that
//    once a step nothing is on its way and the latency of an L2 miss is paid in full; a compute unit has no more than 32 KB of
//    misses in flight (60 GB/s from HBM for one alone, 114 from the last-level cache, with 32 KB as with 128), so what the stream needs
//    is to be continuous. Products, one barrier and an L2 prefetch of the lines shared -> two
//    barriers and none, us: hidden 4096, I 1536, E 128, 512 rows an expert 1415 -> 1332, 789 -> 756 (up, down), input gradients 1397 ->
//    1350, weight gradients 1735 -> 1694, 902 -> 866; 256 rows 901 -> 840, 479 -> 449 (up with the activation 889 -> 800); 128 rows 807 ->
//    734 (up); hidden 2048, I 1408, E 64, 4096 rows 2360 -> 2296, 1242 -> 1198, input gradient 2284 -> 2236; hidden 4096, I 14336, E 8,
//    4096 rows 5640 -> 5650, 2981 -> 2862, input gradient of the first projection 5920 -> 5867 (there the matrix instructions' power is the
//    bound: all-zero operands 4657 -> 4310, 5107 -> 4620). What it costs: launches of a tile or two per workgroup 0.3 us (input gradient
//    [8 x 256 rows, 4096 x 64] 13.7 -> 14.0), gathered weight gradients over few rows, whose second loads wait for the index behind the
//    second barrier, 1.5 to 2.7 % ([8 x 128 rows, 2048 x 2048] 25.7 -> 26.3, [128 x 128, 3072 x 4096] 845 -> 865; [128 x 512] 1655 -> 1633).
//  * A K loop always runs an even number of steps (a step of zeros is appended to an odd reduction length), so every tile
//    starts in LDS stage 0 and the loop body stays two straight-line steps.
//  * Tiles that break the pattern (groups of few rows on their three-stage loop, groups without reduction, groups
//    that need the element-wise path) start cold: the tile before them lets its last two load slots fetch nothing and
//    drains, and they issue their first loads themselves, followed by as many stores outside every buffer as an epilogue
//    issues, so that the waits of the K loop are the same constants in both cases.
//  * Two kinds of kernels read one operand through an index instead of a packed copy (GATHER): the forward product takes
//    the rows of A as rows row_index[i] / divisor of the token matrix (a table of the tile's 256 entries in LDS, four
//    per-lane offsets per K step), the weight gradient takes the reduction rows of B the same way (eight entries per
//    wavefront and K step, requested two steps ahead). Both give the bits of the packed kernel on a gathered copy.
//  * Tall tiles (TALL; rows vary, A with its reduction contiguous, at most 256 groups, whose shorter table leaves the LDS): a tile may
//    have 32 rows more, one 16-row block per wavefront in a 4 KB stage of its own. A K step is bound by the delivery of its
//    operands, above all of B (a tile of 8 rows takes 88 % of a full one's time), so what counts is how many tiles stream a
//    panel of B: experts of 256 or 512 +- 20 rows, as an even routing makes them, take one or two tiles instead of every other one
//    a nearly empty one more. A group gets as few tiles as 288 rows allow, of which as few as its rows need are tall (a tall
//    step costs 6 % more loads and 12 % more matrix instructions), in launches where that saves rounds of tiles (most_rows), by the
//    sizes in device memory. Same sums in the same order: same bits. Products of evenly
//    routed layers, 256-row tiles -> tall (us): hidden 4096, I 1536, E 128, k 8, 4096 tokens 984 -> 945, 541 -> 500 (up, down), input
//    gradients 951 -> 852, 595 -> 522; 8192 tokens 1570 -> 1432, 858 -> 801, 1536 -> 1416, 924 -> 806; hidden 4096, I 14336, E 8,
//    k 2, 4096 tokens 1600 -> 1510, 1004 -> 749, 1996 -> 1460, 900 -> 842; hidden 2048, I 8192, 1021 tokens 228 -> 159 (up); rows that
//    leave the number of tiles as it is (94 to 156 an expert) 0.99 to 1.01 of the time.
//  * The last, partial round of tiles of a tall kernel is cut into 2 or 4 parts of their columns where there are workgroups for them: the
//    loads of B shrink with the columns, and the round takes 0.8 to 0.9 of a whole one's time. Products of 384 tiles (hidden 2880,
//    I 2880, E 32, k 4, 2000 tokens) 191 -> 179 us (down), 331 -> 314 us (input gradient); of 320 (hidden 2048, I 8192, E 8, k 2, 5000
//    tokens) 393 -> 364 us.
#pragma once

#include "gemm_parts.h"

namespace fmahip {
namespace gemm {
namespace ragged {

constexpr int kBwdAhead = 2;        // passes of the SwiGLU-gradient epilogue whose h values are requested ahead
constexpr uint32_t kStreamOutSteps = 16;  // weight-gradient tiles of at most this many K steps store with the non-temporal hint

constexpr int NWM = 2, NWN = 4, NW = NWM * NWN, NT = NW * 64;
constexpr int WM = BM / NWM, WN = BN / NWN;  // 128 x 64 per wavefront
constexpr int RB = WM / 16, CB = WN / 16;    // 8 x 4 accumulator blocks of 16 x 16 (the 16x16x32 matrix instruction)
constexpr int kTallM = 288;                  // rows of a tall tile: 256, and one more 16-row block per wavefront
constexpr uint32_t kTallGroups = 256;        // groups a launch of the tall kernels may have (their table is that much shorter)
constexpr int kRowLoads = 5;                 // loads of A rows per wavefront and K step of a tall tile (otherwise four)
constexpr int kExtraBytes = (kTallM - BM) * kRowBytes;  // LDS of the rows past 256, per stage
// The three-stage K loop: groups of at most 64 rows, and without a bias of at most kShortRows where the reduction has kShortSteps K steps
// and more (with a bias and both forms of the loop the plain kernel of tall tiles runs out of registers). Such a group has one row tile, whose
// panels of B no other workgroup reads: a stream of the weights, with one more K step in flight than two stages hold. What it pays is that
// its tiles start cold, which short reductions feel. Groups of 65 to 128 rows, two stages / three, us: [8 x 96 rows, 28672 x 4096] 429 / 407, [8 x 100,
// 2048 x 2048] 38.2 / 36.8, input gradient [16 x 100, 2048 x 2048] 33.4 / 32.1, SwiGLU gradient [64 x 96, 1408 x 2048] 102.2 / 100.7, [64 x 96, 2816 x
// 2048] gathered 189 / 190, [128 x 96, 3072 x 4096] 683 / 658 (which repeats to 4 %). Below the line: 24 steps [128 x 128, 4096 x 1536] 367 / 372,
// [8 x 100, 2048 x 1536] 31.9 / 30.6; 16 steps, SwiGLU gradient [64 x 96, 1408 x 1024] 59.9 / 62.0; 8 steps [128 x 96, 3072 x 512] 109 / 112. Groups of up to
// 64 rows fetch 64 rows of A a step and not 128: with one form of the loop for all, SwiGLU gradients of [64 x 32 rows, 1408 x 2048] took 91.8 us
// instead of 89.5, of [16 x 32, 1024 x 2048] 29.0 instead of 27.8, the input gradient [64 x 32, 1408 x 2048] 75.0 instead of 73.2, the rest up to 1 %
// more. B with the non-temporal hint: weights from memory 3 to 5 % faster ([128 x 48, 3072 x 4096] 638 -> 619), weights that the last-level cache
// holds from the pass before up to 37 % slower ([8 x 48, 4096 x 2048] 27 -> 35, [16 x 40, 2048 x 2048] 27 -> 37); on all tiles 4 to 17 % slower
// where row tiles share a panel. Not taken.
constexpr uint32_t kShortRows = 128, kShortSteps = 32;
constexpr int kStageBytes = 2048;            // epilogue staging per wavefront: 16 rows of 128 bytes or 32 rows of 64

struct Args {
    const uint16_t* A;
    const uint16_t* B;
    uint16_t* D;            // plain: output; swiglu: pre-activation h (may be NULL)
    uint16_t* ACT;          // swiglu only: activation output
    const uint32_t* sizes;  // E values of the varying dimension
    const uint16_t* bias;   // BIAS kernels: [E, n] added to the rounded product before anything else
    const uint16_t* h_in;   // EPI_SWIGLU_BWD: the packed pre-activation [rows, 2 n] whose gradient goes to D
    // GATHER kernels, rows vary: row i of the packed A operand is row row_index[i] / divisor of A, which has a_rows rows.
    // GATHER kernels, reduction varies (weight gradient): reduction row i of the packed B operand is row
    // row_index[i] / divisor of B, which has a_rows rows of n elements.
    const int32_t* row_index;
    uint32_t divisor, a_rows;
    uint32_t E;
    uint32_t m, n, k;  // the dimensions all groups share (the varying one is ignored)
    float alpha;
    // fma_grouped_gemm (per-group M, N and K arrays in device memory): when n_dev is set, the shared dimensions are the
    // first entries of the arrays, and the kernel runs only if the launch has its form (see the top of the kernel)
    const uint32_t* m_dev;
    const uint32_t* n_dev;
    const uint32_t* k_dev;
    // EPI_SPLIT: every tile is computed `splits` times, each time over split_steps K steps (an even number, so that only the
    // last part can end inside a step or on an odd one); part s of packed row r goes to partial[(s * rows + r) * n ..]
    float* partial;
    uint32_t splits, split_steps, rows;
    // not NULL: the kernel runs only if *taken, which it decides (takes_many_passes) and writes first if pass_bits is not 0;
    // otherwise the streaming kernel behind it computes the product (thin_experts.hip)
    uint32_t* taken;
    uint32_t pass_bits;
};

// s_waitcnt immediate: vmcnt(vm), and lgkmcnt(0) too if lgkm0 (expcnt untouched)
constexpr int waitcnt_imm(int vm, bool lgkm0) {
    return (vm & 15) | ((vm >> 4) << 14) | (7 << 4) | ((lgkm0 ? 0 : 15) << 8);
}

// The per-tile part of a loader's state (everything else depends on lane, wavefront and the shared dimensions only)
template <bool KC>
struct Feed {
    const uint16_t* base0;
    const uint16_t* base1;  // second row range of a split [row][k] tile
    uint32_t extent;        // [row][k] tile: valid bytes from a base; [k][out] tile: reduction length
    uint32_t ldb;           // row pitch of the operand in bytes
    uint32_t col_bytes;     // [k][out] tile: byte offset of the tile's first column inside a row
};


// The `rest` tiles left after the whole rounds of `g` workgroups are computed in 1, 2 or 4 (the logarithm is returned) parts of their
// columns, as many as there are workgroups for.
__device__ __forceinline__ uint32_t parts_of_tail(uint32_t rest, uint32_t g) {
    return rest * 4u <= g ? 2u : (rest * 2u <= g ? 1u : 0u);
}

// The time of `units` tiles on `g` workgroups in rounds of 256-row tiles, `tall` of them with rows past 256: such a tile takes a seventh
// more (8 groups of about 300 rows, 2048 x 8192: 165 us, with one or more of them 186), the last, partial round 0.87 of a
// whole one in parts of its columns and on its own 0.85 (NN, 64 tiles of 2048 x 16384: 345 -> 278 us, 327 -> 279). In the NT layout a launch of at
// most half as many tiles as workgroups is never cut. Over 118 launches (twelve shapes, 200 to 2048 rows a group, randomly routed) the height taken
// costs 0.6 % more than the better of the two; 256 rows always 5.7 %, 288 wherever a group has more than 256 rows 2.2 %. Without parts of the
// last round they take 0.8 % longer.
template <bool PARTS, bool B_KC>
__device__ __forceinline__ float rounds_of(uint32_t units, uint32_t tall, uint32_t g) {
    const uint32_t whole = units / g, rest = units - whole * g;
    float last = rest ? 1.0f : 0.0f;
    if (PARTS && rest && parts_of_tail(rest, g)) last = whole ? 0.87f : (B_KC ? 1.0f : 0.85f);
    return (float)whole + last + 0.14f * (float)((tall + g - 1) / g);
}

// Names an accumulator value as one 16-register value (no instruction, no ordering).
__device__ __forceinline__ void anchor_value(f32x16& c) { asm("" : "+v"(c)); }

template <typename EL, bool A_KC, bool B_KC, int EPI, bool VARY_K, bool BIAS, bool GATHER_ANY, bool TALL>
__global__ __launch_bounds__(NT) void ragged_gemm_kernel(const Args args) {
    // GATHER: the rows of A are picked through row_index (forward); kGatherK: the reduction rows of B are (weight gradient)
    constexpr bool GATHER = GATHER_ANY && !VARY_K;
    constexpr bool kGatherK = GATHER_ANY && VARY_K;
    // kGlu: a forward SwiGLU epilogue (the tile holds 128 "up" and 128 "gate" columns of the product)
    constexpr bool kGlu = EPI == EPI_SWIGLU || EPI == EPI_SWIGLU_ACT;
    static_assert(!kGlu || (A_KC && B_KC && !VARY_K), "the SwiGLU epilogue exists for the NT layout only");
    static_assert(EPI != EPI_SWIGLU_BWD || (A_KC && !B_KC && !VARY_K && !BIAS && !GATHER_ANY),
                  "the SwiGLU-gradient epilogue exists for the input-gradient (NN) layout only");
    // kSplit: fp32 sums over a part of the reduction, added up by split_reduce_kernel
    constexpr bool kSplit = EPI == EPI_SPLIT;
    static_assert(!kSplit || (A_KC && !VARY_K && !BIAS && !GATHER_ANY), "the reduction is split in the NT and NN layouts only");
    static_assert(!TALL || (A_KC && !VARY_K), "tall tiles exist where the rows vary and A has its reduction contiguous");
    static_assert(!BIAS || (A_KC && B_KC && !VARY_K), "the bias term exists for the forward (NT) layout only");
    static_assert(!GATHER || (A_KC && B_KC), "rows are gathered in the forward (NT) layout only");
    static_assert(!kGatherK || (!A_KC && !B_KC && EPI == EPI_PLAIN), "reduction rows are gathered in the weight-gradient (TN) layout only");

    // one array per stage and operand: distinct LDS objects let the compiler see that a direct-to-LDS load
    // into one stage cannot alias the fragment reads of the other, so it does not wait for the load first
    __shared__ __attribute__((aligned(1024))) uint8_t s_a0[kTileBytes];
    __shared__ __attribute__((aligned(1024))) uint8_t s_b0[kTileBytes];
    __shared__ __attribute__((aligned(1024))) uint8_t s_a1[kTileBytes];
    __shared__ __attribute__((aligned(1024))) uint8_t s_b1[kTileBytes];
    // TALL: rows 256 .. 287 of the A tile, per stage
    __shared__ __attribute__((aligned(TALL ? 1024 : 16))) uint8_t s_x0[TALL ? kExtraBytes : 16];
    __shared__ __attribute__((aligned(TALL ? 1024 : 16))) uint8_t s_x1[TALL ? kExtraBytes : 16];
    __shared__ __attribute__((aligned(1024))) uint8_t s_stage[NW * kStageBytes];
    // BIAS: per wavefront, the bias values of its own 64 columns (plain) or 32 "up" | 32 "gate" columns
    constexpr int kBiasBytes = 128;
    __shared__ __attribute__((aligned(256))) uint8_t s_bias[BIAS ? NW * kBiasBytes : 16];
    // GATHER: the row_index entries of the rows of a tile, for the tile of round r in half r % 2. Filled by
    // direct-to-LDS loads and read in assembly: the compiler never sees an access to it.
    constexpr uint32_t kMostRows = TALL ? kTallM : BM;  // of a tile
    __shared__ __attribute__((aligned(256))) uint32_t s_rows[GATHER ? 2 * kMostRows : 4];
    // kGatherK: row_index entries on their way from one tile's last two steps (or a cold start) to the next tile's first two:
    // per LDS stage and wavefront the 64 dwords of one direct-to-LDS load. Read in assembly only.
    __shared__ __attribute__((aligned(256))) uint32_t s_gk[kGatherK ? 2 * NW * 64 : 4];
    // The group table, one LDS object: first tile of the group at position p of the tile sequence, exclusive prefix of the
    // varying dimension over the groups, and which group is at position p.
    constexpr uint32_t kMostGroups = TALL ? kTallGroups : FMA_MAX_GROUPS;
    __shared__ uint32_t s_table[2 * (kMostGroups + 1) + kMostGroups / 2];
    uint32_t* const s_tile_start = s_table;
    uint32_t* const s_prefix = s_table + (kMostGroups + 1);
    uint16_t* const s_order = reinterpret_cast<uint16_t*>(s_table + 2 * (kMostGroups + 1));

    const uint32_t tid = threadIdx.x;
    const uint32_t lane = tid & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t wm = wave / NWN;
    const uint32_t wn = wave % NWN;
    const uint32_t E = args.E;

    if constexpr (A_KC && B_KC && !VARY_K && (EPI == EPI_PLAIN || EPI == EPI_SWIGLU_ACT)) {
        if (args.taken) {
            uint32_t take;
            if (args.pass_bits) {
                take = takes_many_passes(args.sizes, E, args.pass_bits, lane) ? 1u : 0u;
                if (blockIdx.x == 0 && tid == 0) *args.taken = take;
            } else {
                take = *args.taken;
            }
            if (!take) return;
        }
    }

    // The dimensions all groups share. Called with per-group arrays of all three dimensions (fma_grouped_gemm), the kernel
    // first looks whether the launch has its form: rows vary -> N and K the same for every group; reduction varies -> M and
    // N the same and K not (when all three are the same the rows-vary kernel runs). If not, it leaves the launch to the
    // kernel launched beside it: the three kernels of fma_grouped_gemm agree on one of them without a word to the host.
    uint32_t dim_m = args.m, dim_n = args.n, dim_k = args.k;
    if (args.n_dev) {
        typedef const __attribute__((address_space(4))) uint32_t* const_dim_ptr;
        const const_dim_ptr ma = (const_dim_ptr)args.m_dev, na = (const_dim_ptr)args.n_dev, ka = (const_dim_ptr)args.k_dev;
        dim_m = ma[0];
        dim_n = na[0];
        dim_k = ka[0];
        bool m_differs = false, n_differs = false, k_differs = false;
        for (uint32_t e = tid; e < E; e += NT) {
            m_differs = m_differs || args.m_dev[e] != dim_m;
            n_differs = n_differs || args.n_dev[e] != dim_n;
            k_differs = k_differs || args.k_dev[e] != dim_k;
        }
        const bool m_same = !__syncthreads_or(m_differs), n_same = !__syncthreads_or(n_differs), k_same = !__syncthreads_or(k_differs);
        const bool mine = VARY_K ? (m_same && n_same && !k_same) : (n_same && k_same);
        if (!mine) return;
    }

    // The compiler orders LDS accesses behind direct-to-LDS loads in flight per LDS object: an access to an object that
    // some load has written waits for the loads into THAT object only, an access to an object no load has ever written
    // waits for all of them. The group table is read while the next tile's operand loads are in flight, so it gets
    // one load that fetches nothing, here, to be known as an object of its own.
    {
        const __amdgpu_buffer_rsrc_t nowhere = make_rsrc(args.A, 0u);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(nowhere, (lds_void*)s_table, 4, kOutOfRange, 0, 0, 0);
        __builtin_amdgcn_s_waitcnt(waitcnt_imm(0, false));
        __syncthreads();
    }

    // The size array is read through the constant address space: with a wavefront-uniform index that is a scalar load
    // (nothing writes the array while the kernel runs), not a vector load that every tile would wait for.
    typedef const __attribute__((address_space(4))) uint32_t* const_u32_ptr;
    const const_u32_ptr sizes = (const_u32_ptr)args.sizes;
    auto group_m = [&](uint32_t e) { return VARY_K ? dim_m : sizes[e]; };
    auto group_k = [&](uint32_t e) { return VARY_K ? sizes[e] : dim_k; };
    const uint32_t Ne = dim_n;
    constexpr bool kCanNarrow = A_KC && B_KC && !kSplit;
    // kTail: the tiles of the last round may be cut into column parts (not those of a split reduction, which fills the round already)
    constexpr bool kTail = TALL && !kSplit;
    constexpr uint32_t kTileN = kGlu ? BN / 2 : BN;  // columns of the tile grid one tile covers
    const uint32_t n_span = kGlu ? Ne / 2 : Ne;      // columns the tile grid runs over
    bool narrow = false;
    uint32_t most_rows = kMostRows;  // rows of a tile of this launch (TALL: decided below)
    auto row_tiles = [&](uint32_t m) -> uint32_t { return (m + most_rows - 1) / most_rows; };
    // how many of a group's tiles have rows past 256
    auto tall_tiles = [&](uint32_t m, uint32_t tiles) -> uint32_t {
        return m > tiles * (uint32_t)BM ? (m - tiles * (uint32_t)BM + (uint32_t)(kTallM - BM) - 1) / (uint32_t)(kTallM - BM) : 0u;
    };
    auto tiles_of = [&](uint32_t m) -> uint32_t {
        if (m == 0 || Ne == 0) return 0;
        const uint32_t width = (kCanNarrow && narrow && m <= 64u) ? kTileN / 2 : kTileN;
        return row_tiles(m) * ((n_span + width - 1) / width);
    };

    // ---- order of the groups in the tile sequence: by K steps per tile, longest first (see grouped_gemm.hip) ----
    {
        uint32_t* const key = reinterpret_cast<uint32_t*>(s_a0);  // K steps per tile of group e; 0 if it has no tiles
        const uint32_t key0 = tiles_of(group_m(0)) ? (group_k(0) + BK - 1) / BK : 0u;
        bool differs = false;
        for (uint32_t e = tid; e < E; e += NT) {
            const uint32_t k = tiles_of(group_m(e)) ? (group_k(e) + BK - 1) / BK : 0u;
            key[e] = k;
            differs = differs || k != key0;
        }
        if (__syncthreads_or(differs)) {
            for (uint32_t e = tid; e < E; e += NT) {
                const uint32_t mine = key[e];
                uint32_t rank = 0;
                for (uint32_t j = 0; j < E; ++j) {
                    const uint32_t other = key[j];
                    rank += (other > mine || (other == mine && j < e)) ? 1u : 0u;
                }
                s_order[rank] = (uint16_t)e;
            }
        } else {
            for (uint32_t e = tid; e < E; e += NT) s_order[e] = (uint16_t)e;
        }
        __syncthreads();
    }

    if constexpr (TALL || kCanNarrow) {
        // (every wavefront sums by itself: no barrier, and no atomics, which the compiler makes a loop over the lanes)
        uint32_t few = 0, sums[3] = {0u, 0u, 0u};  // groups of at most 64 rows; tiles of 256 rows, tiles of up to 288, tall ones of these
        for (uint32_t e = lane; e < E; e += 64u) {
            const uint32_t m = group_m(e), tiles = (m + (uint32_t)kTallM - 1) / (uint32_t)kTallM;
            few += m > 0u && m <= 64u ? 1u : 0u;
            sums[0] += (m + (uint32_t)BM - 1) / (uint32_t)BM;
            sums[1] += tiles;
            sums[2] += tall_tiles(m, tiles);
        }
#pragma unroll
        for (int d = 32; d > 0; d >>= 1) {
            few += (uint32_t)__shfl_xor((int)few, d, 64);
#pragma unroll
            for (int i = 0; i < 3; ++i) sums[i] += (uint32_t)__shfl_xor((int)sums[i], d, 64);
        }
        const uint32_t columns = (n_span + kTileN - 1) / kTileN, g = gridDim.x;
        if constexpr (TALL) {
            // Tiles of up to 288 rows where they save more rounds than their longer K steps cost. 256-row tiles / tall ones wherever a
            // group has more than 256 rows, us, randomly routed: 2048 x 8192, E 8, 300, 600 and 800 rows a group (one round either way:
            // not taken) 165 / 186, 171 / 196, 181 / 208, 1024 rows (two rounds / one) 309 / 205; 2880 x 2880, E 32, 300 rows (three /
            // three) 179 / 204, 256 rows 194 / 159; 4096 x 1536, E 128, 256 rows (12 / 9) 516 / 479; 2048 x 1408, E 64, 300 rows 135 / 146.
            const uint32_t per = columns * (kSplit ? args.splits : 1u);
            const float low = rounds_of<kTail, B_KC>(uniform(sums[0]) * per, 0u, g);
            const float high = rounds_of<kTail, B_KC>(uniform(sums[1]) * per, uniform(sums[2]) * per, g);
            most_rows = uniform(high < low ? (uint32_t)kTallM : (uint32_t)BM);
        }
        if constexpr (kCanNarrow) {
            // half-width column tiles for groups of at most 64 rows when that fills the workgroups better (grouped_gemm.hip)
            const uint32_t t_small = uniform(few) * columns, t_other = uniform(sums[most_rows == (uint32_t)BM ? 0 : 1]) * columns - t_small;
            const uint32_t rounds = (t_small + t_other + g - 1) / g;
            const uint32_t half_rounds = (2 * t_small + g - 1) / g;
            narrow = t_other == 0 ? half_rounds * 10u <= 2u * rounds * 9u : (t_small + t_other) * 2u <= g;
        }
    }

    // ---- group table, built by wavefront 0: exclusive prefix of tiles over the order above, exclusive prefix of the
    // varying dimension over the groups as they lie in memory ----
    if (wave == 0) {
        uint32_t carry_t = 0, carry_s = 0;
        for (uint32_t base = 0; base < E; base += 64) {
            const uint32_t e = base + lane;
            uint32_t sz = 0, t = 0;
            if (e < E) {
                sz = sizes[e];
                t = tiles_of(group_m(s_order[e]));  // the group at position e of the tile sequence
            }
            const uint32_t it = wave_inclusive_scan<uint32_t>(t);
            const uint32_t is = wave_inclusive_scan<uint32_t>(sz);
            if (e < E) {
                s_tile_start[e] = carry_t + it - t;
                s_prefix[e] = carry_s + is - sz;
            }
            carry_t += __shfl(it, 63, 64);
            carry_s += __shfl(is, 63, 64);
        }
        if (lane == 0) {
            s_tile_start[E] = carry_t;
            s_prefix[E] = carry_s;
        }
    }
    __syncthreads();
    const uint32_t total_tiles = s_tile_start[E];
    // the last, partial round: its tiles in `tail_parts` parts of their columns
    const uint32_t tail_first = total_tiles - total_tiles % gridDim.x;
    const uint32_t tail_shift = kTail && !narrow ? parts_of_tail(total_tiles - tail_first, gridDim.x) : 0u;

    // first tile row of B fragment j (16 rows) of this wavefront
    auto b_frag_row = [&](int j) -> uint32_t {
        if constexpr (kGlu) {
            return j < CB / 2 ? wn * (WN / 2) + j * 16 : BN / 2 + wn * (WN / 2) + (j - CB / 2) * 16;
        } else {
            return wn * WN + j * 16;
        }
    };
    // per-lane LDS byte offsets of this wavefront's fragments for k slice 0 of the two 32-wide slices of a K step
    // (slice 1 adds a constant). A fragment is 16 rows: lane l holds row l % 16, k 8 (l / 16) .. + 7 of the slice.
    uint32_t a_off[RB], b_off[CB];
#pragma unroll
    for (int i = 0; i < RB; ++i) {
        const uint32_t r0 = wm * WM + i * 16;
        a_off[i] = A_KC ? r0 * kRowBytes : mc_frag_off16(r0, lane);
    }
#pragma unroll
    for (int j = 0; j < CB; ++j) {
        const uint32_t r0 = b_frag_row(j);
        b_off[j] = B_KC ? r0 * kRowBytes : mc_frag_off16(r0, lane);
    }
    uint32_t kc_slice[2];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) kc_slice[ks] = kc_off(lane & 15u, (uint32_t)ks * 4u + (lane >> 4));
    const uint32_t x_off = wm * 16 * kRowBytes;    // TALL: this wavefront's row block of the rows past 256
    constexpr uint32_t kSliceT = 32 * kTRowBytes;  // from slice 0 to slice 1 in a [k][out] tile

    // workgroup id -> position in the round of gridDim.x tiles: workgroups of one XCD take 32 neighbours
    const uint32_t grid = gridDim.x;
    const uint32_t per_xcd = grid / kXcds;
    const uint32_t slot = (grid % kXcds == 0) ? (blockIdx.x % kXcds) * per_xcd + blockIdx.x / kXcds : blockIdx.x;

    // Everything that identifies one output tile; the same in every lane.
    struct Tile {
        bool valid, fast;
        uint32_t Me, Ke, m0, n0, n_lim;  // n_lim: first column past the tile (kTileN columns wide, or half of that)
        uint32_t rows;                   // rows of the tile inside the group
        uint32_t e;                      // the group
        uint32_t row0;                   // first packed row (reduction row, if the reduction varies) of the group
        uint64_t off_a, off_b, off_d;
        uint32_t ks, part;    // kSplit: first K element of the tile's part of the reduction, and which part
    };
    auto lookup = [&](uint32_t round) -> Tile {
        Tile t{};
        uint32_t v = round * grid + ((round & 1u) ? grid - 1u - slot : slot);
        const uint32_t total_units = kSplit ? total_tiles * args.splits : tail_first + ((total_tiles - tail_first) << tail_shift);
        if ((uint64_t)round * grid >= total_units || v >= total_units) return t;
        if constexpr (kSplit) {
            // part by part: neighbours in the sequence share operand panels as they do without a split
            t.part = v / total_tiles;
            t.ks = t.part * args.split_steps * (uint32_t)BK;
            v -= t.part * total_tiles;
        }
        uint32_t column_part = 0, parts_shift = 0;
        if constexpr (kTail) {
            if (v >= tail_first) {
                parts_shift = tail_shift;
                column_part = (v - tail_first) & ((1u << tail_shift) - 1u);
                v = tail_first + ((v - tail_first) >> tail_shift);
            }
        }
        // position of the group that holds tile v: the number of groups whose tiles end at or before v. Every lane
        // compares one table entry per 64 groups and a ballot counts them (a binary search would be ten dependent LDS
        // round trips for 1024 groups; this is one per 64 groups, issued back to back).
        uint32_t groups_before = 0;
        for (uint32_t base = 0; base < E; base += 64u) {
            const uint32_t p = base + lane;
            const bool ends_before = p < E && s_tile_start[p + 1] <= v;
            groups_before += (uint32_t)__builtin_popcountll(__ballot(ends_before));
        }
        const uint32_t pos = uniform(groups_before);
        const uint32_t e = uniform((uint32_t)s_order[pos]);
        t.valid = true;
        t.e = e;
        t.Me = group_m(e);
        t.Ke = group_k(e);
        const uint32_t tiles_m = row_tiles(t.Me);
        const uint32_t tile_n = (kCanNarrow && narrow && t.Me <= 64u) ? kTileN / 2 : kTileN;
        const uint32_t tiles_n = (n_span + tile_n - 1) / tile_n;
        const uint32_t local = v - uniform(s_tile_start[pos]);
        const uint32_t band = kGroupM * tiles_n;
        const uint32_t first_m = (local / band) * kGroupM;
        const uint32_t band_m = tiles_m - first_m < (uint32_t)kGroupM ? tiles_m - first_m : (uint32_t)kGroupM;
        const uint32_t mt = first_m + (local % band) % band_m;
        const uint32_t nt = (local % band) / band_m;
        // TALL: the first tiles of the group are 288 rows high, as many as its rows need; the others 256
        const uint32_t past = TALL ? tall_tiles(t.Me, tiles_m) : 0u;
        const uint32_t height = mt < past ? kMostRows : (uint32_t)BM;
        t.m0 = mt * (uint32_t)BM + (mt < past ? mt : past) * (kMostRows - (uint32_t)BM);
        t.rows = t.Me - t.m0 < height ? t.Me - t.m0 : height;
        t.n0 = nt * tile_n;
        t.n_lim = n_span - t.n0 < tile_n ? n_span : t.n0 + tile_n;
        if constexpr (kTail) {
            // (parts past the last column are tiles without columns)
            const uint32_t width = tile_n >> parts_shift, end = t.n_lim;
            t.n0 = t.n0 + column_part * width < end ? t.n0 + column_part * width : end;
            t.n_lim = end - t.n0 < width ? end : t.n0 + width;
        }
        // packed element offsets of the group: the varying dimension's prefix times the other dimension of the operand
        const uint64_t before = uniform(s_prefix[e]);
        t.row0 = (uint32_t)before;
        if constexpr (VARY_K) {
            t.off_a = before * dim_m;
            t.off_b = kGatherK ? 0u : before * Ne;  // gathered: the loads address all of B
            t.off_d = (uint64_t)e * dim_m * Ne;
        } else {
            t.off_a = before * dim_k;
            t.off_b = (uint64_t)e * Ne * dim_k;
            t.off_d = before * Ne;
        }
        // 16-byte accesses need every contiguous dimension a multiple of 8 elements and packed group bases that stayed
        // multiples of 8; loads and stores address a tile with 32-bit byte offsets below 2^31 (grouped_gemm.hip)
        bool fast = (Ne % 8u == 0) && (Ne < (1u << 23)) && (t.off_a % 8u == 0) && (t.off_b % 8u == 0) && (t.off_d % 8u == 0);
        if (A_KC || B_KC) fast = fast && (t.Ke % 8u == 0) && (t.Ke < (1u << 21));
        if (!A_KC) fast = fast && (t.Me % 8u == 0) && (t.Me < (1u << 23));
        if (kGlu) fast = fast && (n_span % 8u == 0);
        t.fast = fast;
        return t;
    };
    auto k_steps = [&](const Tile& t) {
        const uint32_t all = (t.Ke + BK - 1) / BK;
        if constexpr (!kSplit) return all;
        const uint32_t left = all - t.part * args.split_steps;
        return left < args.split_steps ? left : args.split_steps;
    };
    // groups of few rows run a K loop of their own with a third LDS stage; they start cold
    auto is_thin = [&](const Tile& t) {
        if constexpr (BIAS) return A_KC && t.Me <= 64u && k_steps(t) >= 3u;
        return A_KC && t.Me <= kShortRows && k_steps(t) >= (t.Me <= 64u ? 3u : kShortSteps);
    };
    // a tile whose first two K steps can be fetched by the tile before it, and which can fetch the next tile's
    // (gathered reduction rows: their indices are fetched two K steps ahead of the loads, four ahead of the step itself,
    // which looks at most one tile ahead if every tile in the stream has four steps)
    auto streams = [&](const Tile& t) { return t.valid && t.fast && t.Ke > 0 && !is_thin(t) && (!kGatherK || k_steps(t) >= 3u); };

    uint32_t round = 0;  // tiles this workgroup has finished

    // ---- loaders: `cur` feeds the tile being computed, `nxt` the tile after it ----
    LoaderK<NW, false> lk_a;
    LoaderK<NW, kGlu> lk_b;
    LoaderT<NW, true> lt_a, lt_b;
    Feed<A_KC> fa_cur{}, fa_nxt{};
    Feed<B_KC> fb_cur{}, fb_nxt{};
    uint32_t va_cur = 0, va_nxt = 0, vb_cur = 0, vb_nxt = 0;  // the loaders' per-lane offsets (they depend on the pitch)
    // sets a loader object up for tile t and keeps what is specific to the tile
    auto setup_a = [&](const Tile& t, Feed<A_KC>& f, uint32_t& v) {
        if constexpr (GATHER) return;  // nothing per tile: the rows come from the table in s_rows
        const uint16_t* Ae = args.A + t.off_a;
        if constexpr (A_KC) {
            lk_a.setup(Ae + (uint64_t)t.m0 * t.Ke, nullptr, t.rows, t.Ke, wave, lane);
            f = Feed<A_KC>{lk_a.base0, nullptr, lk_a.bytes, lk_a.ldb, 0u};
            v = lk_a.voff;
        } else {
            lt_a.setup(Ae, t.Me, t.Ke, t.m0, wave, lane);
            f = Feed<A_KC>{lt_a.base, nullptr, t.Ke, lt_a.ldb, lt_a.col_bytes};
            v = lt_a.voff;
        }
    };
    auto setup_b = [&](const Tile& t, Feed<B_KC>& f, uint32_t& v) {
        const uint16_t* Be = args.B + t.off_b;
        if constexpr (B_KC) {
            if constexpr (kGlu) {
                // tile rows 0..127: "up" rows n0.. of the weight; rows 128..255: "gate" rows I + n0..
                lk_b.setup(Be + (uint64_t)t.n0 * t.Ke, Be + (uint64_t)(n_span + t.n0) * t.Ke, t.n_lim - t.n0, t.Ke, wave, lane);
            } else {
                lk_b.setup(Be + (uint64_t)t.n0 * t.Ke, nullptr, t.n_lim - t.n0, t.Ke, wave, lane);
            }
            f = Feed<B_KC>{lk_b.base0, lk_b.base1, lk_b.bytes, lk_b.ldb, 0u};
            v = lk_b.voff;
        } else {
            lt_b.setup(Be, Ne, t.Ke, t.n0, wave, lane, kTail ? t.n_lim - t.n0 : (uint32_t)BN);
            f = Feed<B_KC>{lt_b.base, nullptr, t.Ke, lt_b.ldb, lt_b.col_bytes};
            v = kGatherK ? t.row0 : lt_b.voff;  // gathered: where the group's entries of row_index begin (same in every lane)
        }
    };
    // points a loader object at a feed (what depends on lane and wavefront only stays as the last setup left it)
    // (kSplit: the same in every lane, which the compiler does not see in the NT kernels: without this it wraps every load in a loop
    // over the distinct descriptors it fears)
    auto same = [](auto f) __attribute__((always_inline)) {
        if constexpr (kSplit) {
            f.base0 = reinterpret_cast<const uint16_t*>(uniform((uint64_t)(uintptr_t)f.base0));
            f.extent = uniform(f.extent);
            f.ldb = uniform(f.ldb);
        }
        return f;
    };
    auto aim_a = [&](const Feed<A_KC>& any, uint32_t v) {
        if constexpr (GATHER) return;
        const Feed<A_KC> f = same(any);
        if constexpr (A_KC) { lk_a.base0 = f.base0; lk_a.bytes = f.extent; lk_a.ldb = f.ldb; lk_a.kdim = f.ldb / 2u; lk_a.voff = v; }
        else { lt_a.base = f.base0; lt_a.kdim = f.extent; lt_a.ldb = f.ldb; lt_a.col_bytes = f.col_bytes; lt_a.voff = v; }
    };
    auto aim_b = [&](const Feed<B_KC>& any, uint32_t v) {
        const Feed<B_KC> f = same(any);
        if constexpr (B_KC) { lk_b.base0 = f.base0; lk_b.base1 = f.base1; lk_b.bytes = f.extent; lk_b.ldb = f.ldb; lk_b.kdim = f.ldb / 2u; lk_b.voff = v; }
        else { lt_b.base = f.base0; lt_b.kdim = f.extent; lt_b.ldb = f.ldb; lt_b.col_bytes = f.col_bytes; lt_b.voff = v; }
    };

    // ---- GATHER: the A operand's rows are rows of args.A picked through args.row_index ----
    // The tile of round r keeps the row_index entries of its rows in half r % 2 of s_rows. A wavefront's four load
    // instructions of a K step fetch tile rows g_row, g_row + 64, + 128, + 192 of this lane (TALL: and a fifth row
    // 256 + g_row % 32): table entries, divided by the divisor, times the row pitch. Entries past the group's rows read as zero (row 0 of A: rows never stored).
    const uint32_t g_full = GATHER ? args.a_rows * dim_k * 2u : 0u;  // bytes of A (below 2^31)
    const uint32_t g_ldb = dim_k * 2u;
    const uint32_t g_row = logical_row(wave * 8u + (lane >> 3));
    const uint32_t g_chunk = (lane & 7u) ^ (g_row & 7u);
    // The row an entry n of row_index names, n / divisor, or a number no row has if the entry is negative: for n < 2^31 the
    // high word of n * floor((2^32 - 1) / divisor) is the quotient or one less (any divisor from 1 on, no branch).
    const uint32_t g_magic = GATHER_ANY ? 0xffffffffu / args.divisor : 0u;
    auto g_source_row = [&](uint32_t n) -> uint32_t {
        uint32_t q = __umulhi(n, g_magic);
        q += (n - q * args.divisor >= args.divisor) ? 1u : 0u;
        return q | (n & 0x80000000u);
    };
    uint32_t g_bytes_nxt = 0;  // bytes of A the loads for the next tile may read: all of it, or nothing when nothing follows
    // per-lane offsets of the loads of a K step of the tile in table half `half` (the step's k0 goes into the
    // instruction's scalar offset)
    auto g_tile_offsets = [&](uint32_t half, uint32_t (&v)[kRowLoads]) {
        uint32_t n4[4], n[kRowLoads];
        const uint32_t table = lds_address(reinterpret_cast<const uint8_t*>(s_rows)) + half * (kMostRows * 4u);
        lds_read4_stride64_quiet(table + g_row * 4u, n4);
#pragma unroll
        for (int i = 0; i < 4; ++i) n[i] = n4[i];
        if constexpr (TALL) n[4] = lds_read1_quiet(table + (256u + (g_row & 31u)) * 4u);
#pragma unroll
        for (int i = 0; i < (TALL ? 5 : 4); ++i) {
            // an entry that names no row of A (negative, or past the last row) reads as a row of zeros
            const uint32_t src = g_source_row(n[i]);
            v[i] = src < args.a_rows ? src * g_ldb + g_chunk * 16u : kOutOfRange;
        }
    };
    // last, partial K step: chunks past the end of K are pushed out of range, which zero-fills them
    auto g_clip = [&](uint32_t k0, uint32_t (&v)[kRowLoads]) {
        const bool past = k0 + (uint32_t)BK > dim_k && k0 + g_chunk * 8u >= dim_k;
#pragma unroll
        for (int i = 0; i < (TALL ? 5 : 4); ++i) v[i] = past ? kOutOfRange : v[i];
    };
    auto g_offsets = [&](uint32_t half, uint32_t k0, uint32_t (&v)[kRowLoads]) {
        g_tile_offsets(half, v);
        g_clip(k0, v);
    };
    uint32_t g_kept[kRowLoads] = {};  // g_tile_offsets of the tile the full-tile K loop is loading from
    // the table of tile t into half `half`: 32 (TALL: 36) entries per wavefront, in assembly (one load per wavefront)
    auto g_issue_table = [&](const Tile& t, uint32_t half) {
        if constexpr (GATHER) {
            const bool real = t.valid && t.Me > t.m0;
            const uint32_t rows = real ? t.rows : 0u;
            constexpr uint32_t kEach = kMostRows / NW;
            const u32x4 rs = make_rsrc_words(reinterpret_cast<const uint16_t*>(args.row_index + (real ? (uint64_t)t.row0 + t.m0 : 0u)),
                                             rows * 4u);
            const uint32_t to = lds_address(reinterpret_cast<const uint8_t*>(s_rows)) + half * (kMostRows * 4u) + wave * (kEach * 4u);
            if (lane < kEach) buffer_load_lds_quiet_b32(rs, (wave * kEach + lane) * 4u, 0u, to);
        }
    };
    static_assert(!GATHER_ANY || 32 / NW == 4, "four load instructions per wavefront and K step");

    // ---- kGatherK: the reduction rows of the B operand are rows of args.B picked through args.row_index ----
    // A wavefront's four load instructions of a K step fetch the step's reduction rows 8 wave + 2 i + (lane >> 5), i = 0..3
    // (the packed loader's are 16 i + 2 wave + (lane >> 5)): eight consecutive entries of row_index per wavefront and step.
    // They land where the packed loader puts the same rows: rows 2 s and 2 s + 1 of the step lie in kilobyte s of the stage
    // either way, so the LDS image, the fragment reads and the order of the sums are those of the packed kernel.
    // The eight entries are one vector load per wavefront and step (lane l: entry l % 8; a position past the end of
    // row_index reads as 0), issued two steps ahead of the loads that use them, behind the step's own loads: a step's loads
    // for K step kt + 2 go out with the entries requested in step kt - 2, which the second barrier of step kt has seen arrive
    // (loads complete in issue order). Inside a tile the entries travel in a register (gk_ring[s]: requested in the latest
    // step that ran in LDS stage s). Across a tile boundary they travel through LDS (s_gk, a direct-to-LDS load read back
    // in assembly): a register loaded in one tile and used in the next makes the compiler, which cannot count the
    // epilogue's stores, wait for everything in flight at the top of the tile.
    const __amdgpu_buffer_rsrc_t gk_index = make_rsrc(reinterpret_cast<const uint16_t*>(args.row_index),
                                                      kGatherK ? uniform(s_prefix[E]) * 4u : 0u);
    const uint32_t gk_bytes = kGatherK ? args.a_rows * Ne * 2u : 0u;  // bytes of B (below 2^31)
    const uint32_t gk_half = lane >> 5;
    // the 16-byte chunk of a row this lane loads, swizzled as the packed loader does it for the row's place in the step;
    // instruction i: ^ 128 (i & 1)
    const uint32_t gk_chunk = ((lane & 31u) ^ (4u * gk_half) ^ (2u * (wave & 1u))) << 4;
    uint32_t gk_v[4] = {0u, 0u, 0u, 0u};
    // this lane's entry of the eight that begin at position `first` of row_index. pinned: the request may not be issued
    // ahead of anything that precedes it in the program (the empty statement the lane's offset passes through is ordered
    // behind every load before it): the step waits count on the request being the newest load of its step
    auto gk_request = [&](uint32_t first, bool pinned) __attribute__((always_inline)) -> uint32_t {
        uint32_t mine = (lane & 7u) * 4u;
        if (pinned) asm volatile("" : "+v"(mine));
        return __builtin_amdgcn_raw_buffer_load_b32(gk_index, mine, first * 4u, 0);
    };
    // the same request into this wavefront's dwords of LDS stage `slot` of s_gk, and the entry read back from there
    auto gk_request_lds = [&](uint32_t first, int slot, bool pinned) __attribute__((always_inline)) {
        uint32_t mine = (lane & 7u) * 4u;
        if (pinned) asm volatile("" : "+v"(mine));
        __builtin_amdgcn_raw_ptr_buffer_load_lds(gk_index, (lds_void*)(s_gk + (slot * NW + wave) * 64), 4, mine, first * 4u, 0, 0);
    };
    auto gk_from_lds = [&](int slot) __attribute__((always_inline)) -> uint32_t {
        return lds_read1_quiet(lds_address(reinterpret_cast<const uint8_t*>(s_gk)) + (((uint32_t)slot * NW + wave) * 64u + lane) * 4u);
    };
    // per-lane offsets of the four loads of the K step at k0 of a group with `limit` reduction rows, from the entries n
    // (lane l holds entry l % 8): every lane forms the byte offset of its entry's row, then picks, per instruction, the
    // offset of one of the instruction's two rows from the lane that holds it, and adds its chunk.
    auto gk_offsets = [&](uint32_t k0, uint32_t limit, uint32_t n, uint32_t (&v)[4]) {
        // an entry that names no row of B (negative, or past the last row) reads as a row of zeros, and so does a
        // reduction row past the group's end
        uint32_t q = g_source_row(n);
        q = k0 + wave * 8u + (lane & 7u) < limit ? q : 0xffffffffu;
        const uint32_t off = q < args.a_rows ? q * (Ne * 2u) : kOutOfRange;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t even = (uint32_t)__builtin_amdgcn_readlane((int)off, 2 * i);
            const uint32_t odd = (uint32_t)__builtin_amdgcn_readlane((int)off, 2 * i + 1);
            v[i] = (gk_half ? odd : even) + (gk_chunk ^ (128u * ((uint32_t)i & 1u)));
        }
    };

    constexpr int kLoads = 32 / NW;                // load instructions per wavefront, operand and K step
    constexpr uint32_t kStepLoads = 2 * kLoads;    // per wavefront and K step
    constexpr uint32_t kColdLoads = kStepLoads + (TALL ? 1 : 0);  // ... of a cold start, which always fetches the rows past 256
    // store instructions per wavefront and tile (the epilogue issues a fixed number; that of a tile with rows past 256 a few
    // more, which makes the wait that counts them wait for the oldest few as well)
    constexpr uint32_t kTileStores = EPI == EPI_PLAIN        ? WM * WN * 2 / 1024
                                     : EPI == EPI_SWIGLU_BWD ? 2 * (WM * WN * 2 / 1024)  // two columns written per column
                                     : kSplit                ? WM * WN * 4 / 1024
                                                             : (EPI == EPI_SWIGLU ? WM * WN * 2 / 1024 : 0) + WM * WN / 1024;

    // loads of one K step of the CURRENT loaders' aim into `stage` (compiler-visible: placed by the scheduling hints)
    // (i0_c, i1_c: which of the kLoads instructions)
    auto issue_a = [&](int stage, uint32_t k0, auto i0_c, auto i1_c) __attribute__((always_inline)) {
        constexpr int I0 = decltype(i0_c)::value, I1 = decltype(i1_c)::value;
        if constexpr (A_KC) lk_a.template issue_range<I0, I1>(stage ? s_a1 : s_a0, k0);
        else lt_a.template issue_range<I0, I1>(stage ? s_a1 : s_a0, k0);
    };
    // GATHER: the same four loads through the row table in half `half`; `bytes`: how much of A they may read
    // kept: take the offsets from g_kept (the caller has set it for that tile) instead of reading the table
    // (instruction 4: the rows past 256)
    auto issue_a_gathered = [&](int stage, uint32_t k0, uint32_t half, uint32_t bytes, bool kept, auto i0_c, auto i1_c)
                                __attribute__((always_inline)) {
        constexpr int I0 = decltype(i0_c)::value, I1 = decltype(i1_c)::value;
        uint32_t v[kRowLoads];
        if (kept) {
#pragma unroll
            for (int i = 0; i < (TALL ? 5 : 4); ++i) v[i] = g_kept[i];
            g_clip(k0, v);
        } else {
            g_offsets(half, k0, v);
        }
        const __amdgpu_buffer_rsrc_t r = make_rsrc(args.A, uniform(bytes));
        uint8_t* tile = stage ? s_a1 : s_a0;
#pragma unroll
        for (int i = I0; i < I1; ++i)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_void*)(i < 4 ? tile + (i * NW + wave) * 1024 : (stage ? s_x1 : s_x0) + (wave & 3u) * 1024),
                                                     16, v[i], k0 * 2u, 0, 0);
    };
    // TALL: the rows past 256, one instruction per wavefront (outside the tile's rows: zeros)
    auto issue_x = [&](int stage, uint32_t k0) __attribute__((always_inline)) {
        if constexpr (TALL && !GATHER) lk_a.issue_extra(stage ? s_x1 : s_x0, k0);
    };
    auto issue_b = [&](int stage, uint32_t k0, auto i0_c, auto i1_c) __attribute__((always_inline)) {
        constexpr int I0 = decltype(i0_c)::value, I1 = decltype(i1_c)::value;
        if constexpr (kGatherK) {
            // (gk_v: the offsets of the step's four loads, formed by the caller from the entries requested two steps ago)
            const __amdgpu_buffer_rsrc_t r = make_rsrc(lt_b.base, gk_bytes - lt_b.col_bytes);
            uint8_t* tile = stage ? s_b1 : s_b0;
#pragma unroll
            for (int i = I0; i < I1; ++i)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_void*)(tile + (wave * 4 + i) * 1024), 16, gk_v[i], 0u, 0, 0);
        } else if constexpr (B_KC) lk_b.template issue_range<I0, I1>(stage ? s_b1 : s_b0, k0);
        else lt_b.template issue_range<I0, I1>(stage ? s_b1 : s_b0, k0);
    };
    // ... and written in assembly, for a cold start
    auto issue_quiet = [&](int stage, uint32_t k0) {
        if constexpr (GATHER) {
            uint32_t v[kRowLoads];
            g_offsets(round & 1u, k0, v);
            const u32x4 r = make_rsrc_words(args.A, g_full);
            const uint32_t lds0 = lds_address(stage ? s_a1 : s_a0) + wave * 1024u;
#pragma unroll
            for (int i = 0; i < 4; ++i) buffer_load_lds_quiet(r, v[i], k0 * 2u, lds0 + (uint32_t)(i * NW) * 1024u);
            if constexpr (TALL) buffer_load_lds_quiet(r, v[4], k0 * 2u, lds_address(stage ? s_x1 : s_x0) + (wave & 3u) * 1024u);
        } else if constexpr (A_KC) {
            lk_a.issue_quiet(stage ? s_a1 : s_a0, k0);
            if constexpr (TALL) lk_a.issue_quiet_extra(stage ? s_x1 : s_x0, k0);
        } else lt_a.issue_quiet(stage ? s_a1 : s_a0, k0);
        if constexpr (kGatherK) {
            uint32_t v[4];
            gk_offsets(k0, lt_b.kdim, gk_request(vb_cur + k0 + wave * 8u, false), v);
            const u32x4 r = make_rsrc_words(lt_b.base, gk_bytes - lt_b.col_bytes);
            const uint32_t lds0 = lds_address(stage ? s_b1 : s_b0) + wave * 4096u;
#pragma unroll
            for (int i = 0; i < 4; ++i) buffer_load_lds_quiet(r, v[i], 0u, lds0 + (uint32_t)i * 1024u);
        } else if constexpr (B_KC) lk_b.issue_quiet(stage ? s_b1 : s_b0, k0);
        else lt_b.issue_quiet(stage ? s_b1 : s_b0, k0);
    };

    Tile cur = lookup(0), nxt = lookup(1);
    // GATHER: the second tile's rows (the first tile fetches its own in its cold start; from then on every tile
    // fetches those of the tile after next, before its epilogue)
    g_issue_table(nxt, 1u);
    bool streamed = false;  // the first two K steps of `cur` were fetched by the tile before it
    while (cur.valid) {
        const uint32_t Me = cur.Me, Ke = cur.Ke, m0 = cur.m0, n0 = cur.n0, n_lim = cur.n_lim;
        const uint64_t off_d = cur.off_d;
        const bool has_extra = TALL && cur.rows > (uint32_t)BM;  // rows past 256

        if (!streamed) {
            if (!cur.fast) {
                if constexpr (EPI == EPI_PLAIN && !kGatherK) {  // (the gathered entry point admits only sizes without such tiles)
                    scalar_tile<EL, A_KC, B_KC>(args.A + cur.off_a, args.B + cur.off_b, args.D + off_d, Me, Ne, Ke, m0, m0 + cur.rows,
                                                n0, n_lim, args.alpha, NT);
                }
                cur = nxt;
                nxt = lookup(round + 2);
                ++round;
                continue;
            }
            setup_a(cur, fa_cur, va_cur);
            setup_b(cur, fb_cur, vb_cur);
        }
        if (GATHER && !streamed) {
            // a tile that starts cold fetches its own rows and waits for them (and for everything else in flight)
            g_issue_table(cur, round & 1u);
            __builtin_amdgcn_s_waitcnt(waitcnt_imm(0, false));
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
        }
        const uint32_t KT = k_steps(cur);
        const uint32_t KT2 = (KT + 1u) & ~1u;  // steps of the K loop: an odd count gets a step of zeros
        const bool thin = is_thin(cur);
        // kGatherK: where in row_index the entries of this wavefront for K step `abs_step` of the load stream begin: a step
        // of this tile, or, past its end, of the next (vb_cur, vb_nxt: where the two groups' entries begin)
        auto gk_first = [&](uint32_t abs_step) __attribute__((always_inline)) -> uint32_t {
            const bool of_next = abs_step >= KT2;
            return (of_next ? vb_nxt + (abs_step - KT2) * (uint32_t)BK : vb_cur + abs_step * (uint32_t)BK) + wave * 8u;
        };
        uint32_t gk_ring[2] = {0u, 0u};
        // the next tile's first two K steps ride on this tile's last two load slots
        const bool stream_next = streams(cur) && streams(nxt);
        if (stream_next) {
            setup_a(nxt, fa_nxt, va_nxt);
            setup_b(nxt, fb_nxt, vb_nxt);
        } else {
            // a feed that fetches nothing: every load of it zero-fills
            if constexpr (!GATHER) {
                fa_nxt = fa_cur;
                fa_nxt.extent = 0u;
                va_nxt = va_cur;
            }
            fb_nxt = fb_cur;
            fb_nxt.extent = 0u;
            vb_nxt = vb_cur;
        }
        const bool extra_near = has_extra || (stream_next && nxt.rows > (uint32_t)BM);
        g_bytes_nxt = stream_next ? g_full : 0u;
        // (the set-ups above left the loader objects aimed at the last tile set up)
        aim_a(fa_cur, va_cur);
        aim_b(fb_cur, vb_cur);

        // The CB column blocks of a row block are one 16-register value (block j in elements 4 j ..), and every matrix
        // instruction's result is named as part of that value again (anchor_value): the result then stays in the register
        // quadruple its addend came from. The compiler has no tied-operand form of the 4-register instruction; as 32 separate
        // quadruples the results wandered through the register file and the allocator spilled 3 to 40 registers.
        // (TALL: one more row block, the wavefront's share of the rows past 256)
        constexpr int RBX = TALL ? RB + 1 : RB;
        f32x16 acc[RBX];
#pragma unroll
        for (int i = 0; i < RBX; ++i)
#pragma unroll
            for (int x = 0; x < 16; ++x) acc[i][x] = 0.0f;
        auto mfma_block = [&](f32x16& c, int j, typename EL::frag b, typename EL::frag a) __attribute__((always_inline)) {
            f32x4 q = {c[4 * j], c[4 * j + 1], c[4 * j + 2], c[4 * j + 3]};
            q = EL::mfma16(b, a, q);
            c[4 * j] = q[0];
            c[4 * j + 1] = q[1];
            c[4 * j + 2] = q[2];
            c[4 * j + 3] = q[3];
            anchor_value(c);
        };

        // MFMA operand fragments of one 32-wide k slice: the A fragments of two row blocks (a "pair"), in four buffers (full
        // tiles read them two phases ahead and hold three pairs across the step's barrier; the other versions use two), and
        // the B fragments of the four column blocks. A phase is one pair times the four column blocks, column block by
        // column block. In the last phase of a slice every B fragment is replaced by the next slice's as soon as its two
        // matrix instructions have been issued (one set of B registers).
        // The K loop exists in five versions, for wavefronts whose first FA = 8, 4, 2, 1 or 0 row blocks (of 16 rows)
        // hold rows of the group, and TALL in a sixth, FA = 9, for tiles with rows past 256: the ninth block joins the last
        // pair of each slice.
        typename EL::frag fa[4][2], fx, fb[CB];
        // A fragments of pair `pair` of slice ks into buffer buf
        auto load_a = [&](auto fa_c, int stage, int ks, int pair, int buf) __attribute__((always_inline)) {
            constexpr int FA = decltype(fa_c)::value;
            constexpr int AB = FA < 2 ? FA : 2;
            const uint8_t* ta = stage ? s_a1 : s_a0;
#pragma unroll
            for (int i = 0; i < AB; ++i) {
                const int b = pair * 2 + i;
                if constexpr (A_KC) fa[buf][i] = __builtin_bit_cast(typename EL::frag, read_kc_frag(ta + a_off[b] + kc_slice[ks]));
                else fa[buf][i] = __builtin_bit_cast(typename EL::frag, read_tr_frag(ta + a_off[b] + ks * kSliceT));
            }
        };
        auto load_x = [&](int stage, int ks) __attribute__((always_inline)) {
            fx = __builtin_bit_cast(typename EL::frag, read_kc_frag((stage ? s_x1 : s_x0) + x_off + kc_slice[ks]));
        };
        auto load_b = [&](int stage, int ks, int j) __attribute__((always_inline)) {
            const uint8_t* tb = stage ? s_b1 : s_b0;
            if constexpr (B_KC) fb[j] = __builtin_bit_cast(typename EL::frag, read_kc_frag(tb + b_off[j] + kc_slice[ks]));
            else fb[j] = __builtin_bit_cast(typename EL::frag, read_tr_frag(tb + b_off[j] + ks * kSliceT));
        };
        // pair `pair` from A buffer abuf times the B fragments j0 .. j1 - 1; reload: each B fragment is then read anew from slice
        // next_ks of stage next_stage; reload or nine: the ninth row block joins
        auto mma = [&](auto fa_c, int pair, int abuf, bool reload, int next_stage, int next_ks, int j0 = 0, int j1 = CB, bool nine = false) __attribute__((always_inline)) {
            constexpr int FA = decltype(fa_c)::value;
            constexpr int AB = FA < 2 ? FA : 2;
            if constexpr (FA > 0) {
#pragma unroll
                for (int j = j0; j < j1; ++j) {
#pragma unroll
                    for (int i = 0; i < AB; ++i)
                        mfma_block(acc[pair * 2 + i], j, fb[j], fa[abuf][i]);
                    if constexpr (FA > RB) {
                        if (reload || nine) mfma_block(acc[RB], j, fb[j], fx);
                    }
                    if (reload) load_b(next_stage, next_ks, j);
                }
            }
        };

        // ---- one K step ----
        // WAIT: the s_waitcnt immediate in front of the second barrier. The loads issued after the first barrier are those of step
        // kt + 2: of this tile, or, in the last two steps, steps 0 and 1 of the next tile (or nothing).
        // SRC: which tile the loads issued in the step belong to: 0 the current one, 1 the next one (the loaders are aimed
        // by the caller in both cases), 2 decided here (first steps of a tile, and the versions for tiles with few rows), 3 the same
        // in a step that fetches no rows past 256.
        auto step = [&](auto fa_c, auto wait_c, auto src_c, int stage, uint32_t kt) __attribute__((always_inline)) {
            constexpr int FA = decltype(fa_c)::value;
            constexpr int SRC = decltype(src_c)::value;
            constexpr int AB = FA < 2 ? FA : 2;       // row blocks per phase
            constexpr int PP = FA >= RB ? RB / 2 : (FA >= 2 ? FA / 2 : 1);  // phases per k slice
            constexpr int X = FA > RB ? 1 : 0;        // the ninth row block
            // The rows past 256 are fetched where the tile has them and in the steps whose loads may be for the next tile. The version
            // for no columns looks whether this tile or the next has any; it has no matrix instructions to place loads between, as
            // the others have: a branch in front of their ninth load would leave the other eight in a block of their own.
            constexpr bool kLoadX = TALL && (FA > RB || FA == 0 || SRC == 1 || SRC == 2);
            constexpr bool kEither = SRC >= 2;
            constexpr int NPH = 2 * PP;               // phases of the step
            constexpr int kReadsA = (A_KC ? 1 : 2) * AB, kReadsB = (B_KC ? 1 : 2);  // LDS reads per pair, per B fragment
            // On entry A buffer 0 and the B registers hold the fragments of the first phase.
            typedef std::integral_constant<int, 0> I0_;
            typedef std::integral_constant<int, 1> I1_;
            typedef std::integral_constant<int, 3> I3_;
            typedef std::integral_constant<int, kLoads> IN_;
            static_assert(kLoads == 4, "a step's loads are placed for four per operand");
            // the A loads [i0, i1) of the step's load slot
            auto issue_a_part = [&](uint32_t k0, auto i0_c, auto i1_c) __attribute__((always_inline)) {
                if constexpr (GATHER) {
                    const bool of_next = SRC == 1 || (kEither && kt + 2u >= KT2);
                    issue_a_gathered(stage, k0, (of_next ? round + 1u : round) & 1u, of_next ? g_bytes_nxt : g_full, !kEither, i0_c, i1_c);
                } else {
                    issue_a(stage, k0, i0_c, i1_c);
                }
            };
            auto issue_x_part = [&](uint32_t k0) __attribute__((always_inline)) {
                if constexpr (kLoadX) {
                    if (FA == 0 && !extra_near) return;
                    if constexpr (GATHER) issue_a_part(k0, std::integral_constant<int, 4>{}, std::integral_constant<int, 5>{});
                    else issue_x(stage, k0);
                }
            };
            // The operand whose loads go out behind the first barrier, and the other one, behind the second: B and A (A first: the input
            // gradients 2 to 6 % slower, 512 rows an expert and up; the rest within 1 %, both ways). Gathered reduction rows: A and B,
            // whose entries of row_index have landed at the second barrier only.
            auto issue_first = [&](uint32_t k0, auto i0_c, auto i1_c) __attribute__((always_inline)) {
                if constexpr (kGatherK) issue_a_part(k0, i0_c, i1_c);
                else issue_b(stage, k0, i0_c, i1_c);
            };
            auto issue_second = [&](uint32_t k0) __attribute__((always_inline)) {
                if constexpr (kGatherK) issue_b(stage, k0, I0_{}, IN_{});
                else issue_a_part(k0, I0_{}, IN_{});
            };
            // first barrier: every LDS read of this stage has returned, in every wavefront; the loads of step kt + 2 may fill it
            auto free_stage = [&]() __attribute__((always_inline)) {
                __builtin_amdgcn_s_waitcnt(waitcnt_imm(63, true));
                __builtin_amdgcn_s_barrier();
                asm volatile("" ::: "memory");
            };
            // second barrier: every load of step kt + 1 has landed
            auto next_landed = [&]() __attribute__((always_inline)) {
                __builtin_amdgcn_s_waitcnt(decltype(wait_c)::value);
                __builtin_amdgcn_s_barrier();
                asm volatile("" ::: "memory");
            };
            // kGatherK: the entries for this step's loads were requested two steps ago: by a step of this tile into a register,
            // or, for a tile's first two steps (SRC == 2 in a full tile), by the tile before or the cold start into LDS; the
            // versions for tiles with few rows do not know at compile time which of their steps are the last two and use LDS
            // throughout
            auto gk_step_offsets = [&](uint32_t k0) __attribute__((always_inline)) {
                if constexpr (kGatherK) {
                    constexpr bool kFromLds = FA != RB || kEither;
                    gk_offsets(k0, lt_b.kdim, kFromLds ? gk_from_lds(stage) : gk_ring[stage], gk_v);
                }
            };
            // ... and the entries for the loads of step kt + 2 (K step kt + 4 of the stream) are requested as the step's last
            // load: into LDS by a full tile's last two steps (SRC == 1)
            auto gk_step_request = [&]() __attribute__((always_inline)) {
                if constexpr (kGatherK) {
                    constexpr bool kToLds = FA != RB || SRC == 1;
                    if constexpr (kToLds) gk_request_lds(gk_first(kt + 4u), stage, true);
                    else gk_ring[stage] = gk_request(gk_first(kt + 4u), true);
                }
            };
            // what the loads issued in this step fetch: the K offset (returned) and, decided here (kEither), whether the
            // loaders aim at the current tile's operands or the next one's
            auto aim_loads = [&]() __attribute__((always_inline)) -> uint32_t {
                uint32_t k0;
                if constexpr (SRC == 0) {
                    k0 = (kt + 2u) * (uint32_t)BK;
                    if constexpr (kSplit) k0 += cur.ks;
                } else if constexpr (SRC == 1) {
                    k0 = (kt + 2u - KT2) * (uint32_t)BK;
                    if constexpr (kSplit) k0 += nxt.ks;
                } else {
                    const bool of_next = kt + 2u >= KT2;
                    k0 = (of_next ? kt + 2u - KT2 : kt + 2u) * (uint32_t)BK;
                    if constexpr (kSplit) k0 += of_next ? nxt.ks : cur.ks;
                    if constexpr (!GATHER)
                        aim_a(Feed<A_KC>{of_next ? fa_nxt.base0 : fa_cur.base0, nullptr, of_next ? fa_nxt.extent : fa_cur.extent,
                                         of_next ? fa_nxt.ldb : fa_cur.ldb, of_next ? fa_nxt.col_bytes : fa_cur.col_bytes},
                              of_next ? va_nxt : va_cur);
                    aim_b(Feed<B_KC>{of_next ? fb_nxt.base0 : fb_cur.base0, of_next ? fb_nxt.base1 : fb_cur.base1,
                                     of_next ? fb_nxt.extent : fb_cur.extent, of_next ? fb_nxt.ldb : fb_cur.ldb,
                                     of_next ? fb_nxt.col_bytes : fb_cur.col_bytes},
                          of_next ? vb_nxt : vb_cur);
                }
                return k0;
            };
            if constexpr (FA >= RB) {
                // Full tiles: the first barrier comes after four and a half of the eight phases, with the A fragments of the last
                // three phases already in registers (four A buffers), and the loads go out a few a phase: eight wavefronts that leave a
                // barrier together otherwise queue 72 loads on the one address path at once. Both barriers lie in the middle of a
                // phase, where the reads they wait for have had half a phase to return and the matrix instructions behind them need
                // nothing from LDS (at the phases' ends, and 2 + 2 loads: 0 to 5 % slower on large tiles, 1 % faster on a few others).
                // A fragments are read two phases ahead (phase p's pair sits in buffer p % 4): phase 0 reads those of phases 1
                // (the step before could not: they are behind its barrier) and 2, phase 4 those of 6 and 7 first thing
                load_a(fa_c, stage, 0, 1, 1);
#pragma unroll
                for (int ph = 0; ph < 4; ++ph) {
                    load_a(fa_c, stage, (ph + 2) / PP, (ph + 2) % PP, (ph + 2) & 3);
                    if (X && ph == 1) load_x(stage, 0);
                    mma(fa_c, ph, ph, ph == 3, stage, 1);
                    if (ph == 3) {
                        __builtin_amdgcn_sched_group_barrier(0x100, kReadsA, 0);
#pragma unroll
                        for (int j = 0; j < CB; ++j) {
                            __builtin_amdgcn_sched_group_barrier(0x008, AB + X, 0);
                            __builtin_amdgcn_sched_group_barrier(0x100, kReadsB, 0);
                        }
                    } else {
                        if (ph == 0) interleave3<0, AB * CB, 2 * kReadsA, 0>();
                        else if (ph == 1) interleave3<0, AB * CB, kReadsA + X, 0>();
                        else interleave3<0, AB * CB, kReadsA, 0>();
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
                load_a(fa_c, stage, 1, 2, 2);
                load_a(fa_c, stage, 1, 3, 3);
                if (X) load_x(stage, 1);
                mma(fa_c, 0, 0, false, stage, 1, 0, CB / 2);
                __builtin_amdgcn_sched_group_barrier(0x100, 2 * kReadsA + X, 0);
                __builtin_amdgcn_sched_group_barrier(0x008, AB * CB / 2, 0);
                __builtin_amdgcn_sched_barrier(0);
                free_stage();
                const uint32_t k0 = aim_loads();
                issue_first(k0, I0_{}, I1_{});
                mma(fa_c, 0, 0, false, stage, 1, CB / 2, CB);
                spread_mfma_vmem<0, AB * CB / 2, 1>();
                __builtin_amdgcn_sched_barrier(0);
                issue_first(k0, I1_{}, I3_{});
                mma(fa_c, 1, 1, false, stage, 1);
                spread_mfma_vmem<0, AB * CB, 2>();
                __builtin_amdgcn_sched_barrier(0);
                issue_first(k0, I3_{}, IN_{});
                mma(fa_c, 2, 2, false, stage, 1);
                spread_mfma_vmem<0, AB * CB, 1>();
                __builtin_amdgcn_sched_barrier(0);
                mma(fa_c, 3, 3, false, stage ^ 1, 0, 0, CB / 2, true);
                __builtin_amdgcn_sched_barrier(0);
                next_landed();
                load_a(fa_c, stage ^ 1, 0, 0, 0);
                load_b(stage ^ 1, 0, 0);
                load_b(stage ^ 1, 0, 1);
                gk_step_offsets(k0);
                issue_second(k0);
                issue_x_part(k0);
                gk_step_request();
                mma(fa_c, 3, 3, true, stage ^ 1, 0, CB / 2, CB);
                __builtin_amdgcn_sched_group_barrier(0x100, kReadsA + 2 * kReadsB, 0);
#pragma unroll
                for (int j = 0; j < CB / 2; ++j) {
#pragma unroll
                    for (int i = 0; i < AB + X; ++i) {
                        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                        if (j * (AB + X) + i < kLoads + (kLoadX ? 1 : 0) + (kGatherK ? 1 : 0)) __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
                    }
                    __builtin_amdgcn_sched_group_barrier(0x100, kReadsB, 0);
                }
            } else {
#pragma unroll
                for (int ph = 0; ph < NPH - 1; ++ph) {
                    const bool last_of_slice = ph == PP - 1;
                    load_a(fa_c, stage, (ph + 1) / PP, (ph + 1) % PP, (ph + 1) & 1);
                    mma(fa_c, ph % PP, ph & 1, last_of_slice, stage, 1);
                    if constexpr (FA > 0) {
                        if (last_of_slice) {
                            // the A reads, then per column block its matrix instructions and the read of its next fragment
                            __builtin_amdgcn_sched_group_barrier(0x100, kReadsA, 0);
#pragma unroll
                            for (int j = 0; j < CB; ++j) {
                                __builtin_amdgcn_sched_group_barrier(0x008, AB, 0);
                                __builtin_amdgcn_sched_group_barrier(0x100, kReadsB, 0);
                            }
                        } else {
                            interleave3<0, AB * CB, kReadsA, 0>();
                        }
                        // nothing moves from one phase into another: reads issued earlier would hold their registers longer
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
                free_stage();
                const uint32_t k0 = aim_loads();
                issue_first(k0, I0_{}, IN_{});
                next_landed();
                load_a(fa_c, stage ^ 1, 0, 0, 0);
                gk_step_offsets(k0);
                issue_second(k0);
                issue_x_part(k0);
                gk_step_request();
                mma(fa_c, PP - 1, 1, true, stage ^ 1, 0);
                if constexpr (FA > 0) {
                    // the A reads; per column block its matrix instructions, followed by a load, and the read of the block's next
                    // fragment
                    __builtin_amdgcn_sched_group_barrier(0x100, kReadsA, 0);
#pragma unroll
                    for (int j = 0; j < CB; ++j) {
                        __builtin_amdgcn_sched_group_barrier(0x008, AB, 0);
                        __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
                        __builtin_amdgcn_sched_group_barrier(0x100, kReadsB, 0);
                    }
                    if constexpr (kLoadX) __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
                    if constexpr (kGatherK) __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
                }
            }
        };
        // What the second barrier of a step waits for: all but the four loads behind the first barrier; in a tile's first step the
        // stores of the previous epilogue (or the cold start's stand-ins) and the one load of the bias values are newer than the
        // loads waited for as well, from the second on they are older.
        // (kGatherK: and the request for row_index entries that follows every step's loads. In a tile's first step that
        // request is older than the stores, and a cold start issues none behind the loads waited for: the count stays the one of
        // the cold start, which only waits for more in a streamed tile. A step forms the offsets of its gathered loads behind its second
        // barrier, from the request before the last one, which that wait has seen arrive.)
        using WaitStep = std::integral_constant<int, waitcnt_imm(kLoads + (kGatherK ? 1 : 0), false)>;
        using WaitFirst = std::integral_constant<int, waitcnt_imm(kLoads + (int)kTileStores + (BIAS ? 1 : 0), false)>;

        // BIAS: the bias values of this wavefront's columns of the tile into its 128 bytes of LDS: one load by 32 lanes
        // (every wavefront issues it, so that all count the same loads), complete (loads and stores complete in issue
        // order) long before the epilogue reads them. Columns past the end zero-fill.
        auto issue_bias = [&]() {
            if constexpr (BIAS) {
                const uint16_t* row = args.bias + (uint64_t)cur.e * Ne;
                const u32x4 rs = make_rsrc_words(row, Ne * 2u);
                const uint32_t to = lds_address(s_bias) + wave * (uint32_t)kBiasBytes;
                // plain: columns n0 + wn*64 + 2*lane; swiglu: lanes 0..15 the 32 "up" columns, lanes 16..31 the "gate" ones
                const uint32_t col = EPI == EPI_PLAIN ? n0 + wn * WN + 2u * lane
                                                      : n0 + wn * (WN / 2) + 2u * (lane & 15u) + (lane >= 16u ? n_span : 0u);
                if (lane < 32u) buffer_load_lds_quiet_b32(rs, col * 2u, 0u, to);
            }
        };
        Tile nn{};  // the tile after next
        const uint32_t tile_rows = cur.rows;
        const uint32_t wave_rows = tile_rows > wm * WM ? tile_rows - wm * WM : 0u;
        const bool has_columns = n0 + wn * (kGlu ? WN / 2 : WN) < n_lim;
        const uint32_t row_blocks = has_columns ? uniform((wave_rows + 15u) / 16u) : 0u;  // of 16 rows
        if (thin) {
            // three LDS stages in the space that a tile of at most 64 rows leaves unused, or of at most 128 rows and the epilogue's
            // staging buffer; cold start
            constexpr int kMostA = BIAS ? 1 : 2;  // loads of A per wavefront and step, 64 rows each: one up to 64 rows
            const uint8_t* const a_at[3] = {s_a0, s_a1, kMostA == 1 ? s_a0 + 8192 : s_stage};
            const uint8_t* const b_lo[3] = {s_b0, s_b1, s_a0 + 16384};
            const uint8_t* const b_hi[3] = {s_b0 + 16384, s_b1 + 16384, s_a1 + 16384};
            auto issue_thin = [&](auto a_loads_c, int st, uint32_t k0) __attribute__((always_inline)) {
                constexpr int kThinA = decltype(a_loads_c)::value;
                if constexpr (GATHER) {
                    uint32_t v[kRowLoads];
                    g_offsets(round & 1u, k0, v);
#pragma unroll
                    for (int i = 0; i < kThinA; ++i)
                        buffer_load_lds_quiet(make_rsrc_words(args.A, g_full), v[i], k0 * 2u, lds_address(a_at[st]) + (uint32_t)(i * NW) * 1024u + wave * 1024u);
                } else if constexpr (A_KC) lk_a.template issue_quiet_first_rows<kThinA>(lds_address(a_at[st]), k0);
                if constexpr (B_KC) lk_b.issue_quiet_halves(lds_address(b_lo[st]), lds_address(b_hi[st]), k0);
                else lt_b.issue_quiet_halves(lds_address(b_lo[st]), lds_address(b_hi[st]), k0);
            };
            issue_bias();
            const uint32_t k_first = kSplit ? cur.ks : 0u;
            auto thin_start = [&](auto a_loads_c) __attribute__((always_inline)) {
                issue_thin(a_loads_c, 0, k_first);
                issue_thin(a_loads_c, 1, k_first + BK);
                __builtin_amdgcn_s_waitcnt(waitcnt_imm(decltype(a_loads_c)::value + kLoads, true));
                __builtin_amdgcn_s_barrier();
                asm volatile("" ::: "memory");
                issue_thin(a_loads_c, 2, k_first + 2 * BK);
            };
            auto thin_loop = [&](auto a_loads_c, auto fa_c) __attribute__((always_inline)) {
                constexpr int FA = decltype(fa_c)::value;
                auto thin_step = [&](int st, uint32_t kt) {
                    if constexpr (FA > 0) {
#pragma unroll
                        for (int ks = 0; ks < 2; ++ks) {
                            typename EL::frag ta[FA], tb[CB];
#pragma unroll
                            for (int i = 0; i < FA; ++i)
                                ta[i] = __builtin_bit_cast(typename EL::frag, read_kc_frag(a_at[st] + a_off[i] + kc_slice[ks]));
#pragma unroll
                            for (int j = 0; j < CB; ++j) {
                                if constexpr (B_KC) {
                                    const uint8_t* half = b_frag_row(j) < 128u ? b_lo[st] + b_off[j] : b_hi[st] + (b_off[j] - 128u * kRowBytes);
                                    tb[j] = __builtin_bit_cast(typename EL::frag, read_kc_frag(half + kc_slice[ks]));
                                } else {
                                    const uint8_t* half = ks == 0 ? b_lo[st] : b_hi[st];  // k rows 0..31 and 32..63 of the step
                                    tb[j] = __builtin_bit_cast(typename EL::frag, read_tr_frag(half + b_off[j]));
                                }
                            }
#pragma unroll
                            for (int i = 0; i < FA; ++i)
#pragma unroll
                                for (int j = 0; j < CB; ++j) mfma_block(acc[i], j, tb[j], ta[i]);
                        }
                    }
                    // (and every LDS read of this stage has returned: the compiler moves matrix instructions, and the waits for their
                    // fragments with them, past the barrier, behind which the other wavefronts' loads fill the stage again)
                    __builtin_amdgcn_s_waitcnt(waitcnt_imm(decltype(a_loads_c)::value + kLoads, true));
                    __builtin_amdgcn_s_barrier();
                    asm volatile("" ::: "memory");
                    issue_thin(a_loads_c, st, k_first + (kt + 3) * BK);
                };
                uint32_t kt = 0;
                for (; kt + 2 < KT; kt += 3) {
                    thin_step(0, kt);
                    thin_step(1, kt + 1);
                    thin_step(2, kt + 2);
                }
                if (kt < KT) thin_step(0, kt);
                if (kt + 1 < KT) thin_step(1, kt + 1);
            };
            using One = std::integral_constant<int, 1>;
            using Most = std::integral_constant<int, kMostA>;
            // (more than 64 rows: more than four row blocks, all of one row of wavefronts)
            if (kMostA > 1 && Me > 64u) {
                thin_start(Most{});
                if (row_blocks > 0) thin_loop(Most{}, std::integral_constant<int, 4 * kMostA>{});
                else thin_loop(Most{}, std::integral_constant<int, 0>{});
            } else {
                thin_start(One{});
                if (row_blocks > 2) thin_loop(One{}, std::integral_constant<int, 4>{});
                else if (row_blocks == 2) thin_loop(One{}, std::integral_constant<int, 2>{});
                else if (row_blocks == 1) thin_loop(One{}, std::integral_constant<int, 1>{});
                else thin_loop(One{}, std::integral_constant<int, 0>{});
            }
            __builtin_amdgcn_s_waitcnt(waitcnt_imm(0, true));
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
        } else if (KT > 0) {
            if (!streamed) {
                // cold start: the first two K steps, then as many stores outside every buffer as an epilogue issues
                // (kGatherK: the entries for the loads of steps 0 and 1 first, so that everything the waits below leave
                // outstanding is what they count; a streamed tile has them from the last two steps of the tile before it)
                if constexpr (kGatherK) {
                    gk_request_lds(gk_first(2u), 0, false);
                    gk_request_lds(gk_first(3u), 1, false);
                }
                issue_quiet(0, kSplit ? cur.ks : 0u);
                issue_quiet(1, (kSplit ? cur.ks : 0u) + BK);
                const __amdgpu_buffer_rsrc_t nowhere = make_rsrc(args.D, 0u);
#pragma unroll
                for (uint32_t i = 0; i < kTileStores; ++i)  // (distinct offsets: identical stores would be merged into one)
                    store_tile16<false>(nowhere, kOutOfRange + i * 16u, uint4{0u, 0u, 0u, 0u});
                // the first step's loads have landed; the second step's, and the stand-in stores, may be out
                __builtin_amdgcn_s_waitcnt(waitcnt_imm((int)(kColdLoads + kTileStores), false));
                __builtin_amdgcn_s_barrier();
                asm volatile("" ::: "memory");
            }
            issue_bias();
            using SrcCur = std::integral_constant<int, 0>;
            using SrcNext = std::integral_constant<int, 1>;
            using SrcEither = std::integral_constant<int, 2>;
            using SrcEitherLow = std::integral_constant<int, 3>;
            auto k_loop = [&](auto fa_c) {
                constexpr int FA = decltype(fa_c)::value;
                load_a(fa_c, 0, 0, 0, 0);
                if constexpr (FA > 0) {
#pragma unroll
                    for (int j = 0; j < CB; ++j) load_b(0, 0, j);
                }
                step(fa_c, WaitFirst{}, SrcEither{}, 0, 0);
                step(fa_c, WaitStep{}, SrcEither{}, 1, 1);
                if constexpr (FA >= RB) {
                    // full tiles: the steps in the middle load from the current tile and the last two from the next, each
                    // with the loaders aimed once, so that the loop body carries no selects
                    if (KT2 > 2u) {
                        aim_a(fa_cur, va_cur);
                        aim_b(fb_cur, vb_cur);
                        if constexpr (GATHER) g_tile_offsets(round & 1u, g_kept);
                        uint32_t kt = 2;
                        for (; kt + 2u < KT2; kt += 2) {  // two steps per iteration without a branch between them
                            step(fa_c, WaitStep{}, SrcCur{}, 0, kt);
                            step(fa_c, WaitStep{}, SrcCur{}, 1, kt + 1);
                        }
                        aim_a(fa_nxt, va_nxt);
                        aim_b(fb_nxt, vb_nxt);
                        if constexpr (GATHER) g_tile_offsets((round + 1u) & 1u, g_kept);
                        step(fa_c, WaitStep{}, SrcNext{}, 0, kt);
                        step(fa_c, WaitStep{}, SrcNext{}, 1, kt + 1);
                    }
                } else {
                    uint32_t kt = 2;
                    if constexpr (TALL && FA > 0) {
                        // (a tile of few rows has none past 256: they are fetched for the next one, in the last two steps)
                        for (; kt + 2u < KT2; kt += 2) {
                            step(fa_c, WaitStep{}, SrcEitherLow{}, 0, kt);
                            step(fa_c, WaitStep{}, SrcEitherLow{}, 1, kt + 1);
                        }
                    }
                    for (; kt < KT2; kt += 2) {
                        step(fa_c, WaitStep{}, SrcEither{}, 0, kt);
                        step(fa_c, WaitStep{}, SrcEither{}, 1, kt + 1);
                    }
                }
            };
            static_assert(RB == 8, "the versions below are for eight row blocks per wavefront");
            if constexpr (TALL) {
                if (has_extra && has_columns) k_loop(std::integral_constant<int, RB + 1>{});
            }
            if (has_extra && has_columns) {}
            else if (row_blocks > 4) k_loop(std::integral_constant<int, 8>{});
            else if (row_blocks > 2) k_loop(std::integral_constant<int, 4>{});
            else if (row_blocks == 2) k_loop(std::integral_constant<int, 2>{});
            else if (row_blocks == 1) k_loop(std::integral_constant<int, 1>{});
            else k_loop(std::integral_constant<int, 0>{});
            if (!stream_next) {
                // nothing rides behind this tile: its last two load slots zero-filled the stages; they must have landed,
                // and every wavefront must be past its last read, before anyone starts cold
                __builtin_amdgcn_s_waitcnt(waitcnt_imm(0, true));
                __builtin_amdgcn_s_barrier();
                asm volatile("" ::: "memory");
            }
        }

        if (BIAS && KT == 0) {  // a group without reduction: the result is the bias
            issue_bias();
            __builtin_amdgcn_s_waitcnt(waitcnt_imm(0, false));
        }
        // the tile after next is looked up here: scalar work beside an epilogue that is bound by the store path
        nn = lookup(round + 2);
        // GATHER: its rows go where this tile's were (no load of this tile is left to be issued). The load is older than
        // this tile's stores, so the first wait of the next tile covers it.
        g_issue_table(nn, round & 1u);

        // ---- epilogue: through this wavefront's 2 KB of the staging buffer, 16 rows of 128 bytes at a time ----
        // A lane holds row (lane & 15), columns (lane >> 4)*4 + 0..3 of each 16x16 accumulator block.
        // (the lane id is made opaque so that the per-lane address arithmetic is redone per tile, not hoisted out of the
        // tile loop where it would occupy registers throughout the K loop)
        uint32_t el = lane;
        asm volatile("" : "+v"(el));
        const uint32_t img = lds_address(s_stage) + wave * (uint32_t)kStageBytes;
        if (EPI == EPI_PLAIN && args.alpha != 1.0f) {
            const float alpha = args.alpha;
#pragma unroll
            for (int i = 0; i < RBX; ++i) acc[i] *= alpha;
        }
        // Tiles with a short reduction write much per flop (a weight gradient over ~500 rows: 8 K steps per 128 KB tile):
        // their stores carry the non-temporal hint (+4 to 5 % there); for long reductions plain stores are faster by 0 to 1 %
        const bool stream_out = VARY_K && KT <= kStreamOutSteps;
        // BIAS: the four groups of four columns this lane holds of every row block, as fp32
        float bias_f[CB][4];
        if constexpr (BIAS) {
            uint32_t at[4];
            uint2 raw[4];
            const uint32_t mine = lds_address(s_bias) + wave * (uint32_t)kBiasBytes;
            // plain: 64 columns; swiglu: 32 "up" columns (j = 0, 1), then 32 "gate" columns
#pragma unroll
            for (int j = 0; j < CB; ++j) at[j] = mine + ((uint32_t)j * 16u + (el >> 4) * 4u) * 2u;
            lds_read4x8_quiet(at, raw);
#pragma unroll
            for (int j = 0; j < CB; ++j) {
                const uint2 r = raw[j];
                bias_f[j][0] = EL::from_bits((uint16_t)(r.x & 0xffffu));
                bias_f[j][1] = EL::from_bits((uint16_t)(r.x >> 16));
                bias_f[j][2] = EL::from_bits((uint16_t)(r.y & 0xffffu));
                bias_f[j][3] = EL::from_bits((uint16_t)(r.y >> 16));
            }
        }
        // the value that is stored (plain) or activated (swiglu): the rounded product, plus the bias rounded again, which is
        // what the product followed by a separate bias pass gives
        auto with_bias = [&](float product, int j, int x) -> float {
            if constexpr (BIAS) return EL::round(product) + bias_f[j][x];
            else return product;
        };
        // EPI_SWIGLU_BWD: the h values of the eight passes (16 rows each) of this wavefront's sub-tile: [pass][row 0/1][up, gate]
        u32x4 bwd_h[EPI == EPI_SWIGLU_BWD ? RBX : 1][2][2];
        // first row, inside the group, of this wavefront's row block i
        auto block_row = [&](int i) -> uint32_t { return i < RB ? m0 + wm * WM + (uint32_t)i * 16u : m0 + (uint32_t)BM + wm * 16u; };
        // byte offset of this lane's piece of row `r` (0 or 1: rows lane / 8 and 8 + lane / 8 of the pass) from the pass's
        // first row and the wavefront's first column, or out of range
        auto bwd_offset = [&](int r, uint32_t cols_valid) -> uint32_t {
            const uint32_t c16 = el & 7u;
            const uint32_t row = (uint32_t)r * 8u + (el >> 3);
            return c16 * 8u < cols_valid ? row * (Ne * 4u) + c16 * 16u : kOutOfRange;
        };
        auto bwd_rows = [&](int pass) -> uint32_t {  // rows of the pass inside the group
            const uint32_t r0 = block_row(pass);
            if (pass == RB && !has_extra) return 0u;
            return r0 < Me ? (Me - r0 < 16u ? Me - r0 : 16u) : 0u;
        };
        auto bwd_origin = [&](int pass, uint32_t col0) -> uint64_t {  // element offset of the pass's first row and column
            return ((uint64_t)cur.row0 + block_row(pass)) * (2ull * Ne) + col0;
        };
        // h is read once and its gradient written once, in whole 128-byte lines: both carry the non-temporal hint, which
        // keeps them from displacing the operand panels in the L2 (+3 % on the Mixtral shape, +2 % large-E, +0.5 % fine-grained)
        constexpr int kStreamAux = 2;
        auto bwd_request = [&](int pass, uint32_t col0, uint32_t cols_valid) {
            if constexpr (EPI == EPI_SWIGLU_BWD) {
                const __amdgpu_buffer_rsrc_t rs = make_rsrc(args.h_in + bwd_origin(pass, col0), bwd_rows(pass) * (Ne * 4u));
#pragma unroll
                for (int r = 0; r < 2; ++r) {
                    const uint32_t off = bwd_offset(r, cols_valid);
                    bwd_h[pass][r][0] = __builtin_amdgcn_raw_buffer_load_b128(rs, (int)off, 0, kStreamAux);
                    bwd_h[pass][r][1] = __builtin_amdgcn_raw_buffer_load_b128(rs, (int)off, (int)(Ne * 2u), kStreamAux);
                }
            }
        };
        auto bwd_finish = [&](int pass, uint32_t col0, uint32_t cols_valid) {
            if constexpr (EPI == EPI_SWIGLU_BWD) {
                const uint32_t c16 = el & 7u;
                u32x4 dy[2];
                stage_get2_quiet(img, stage_off<WN * 2>(el >> 3, c16), stage_off<WN * 2>(8u + (el >> 3), c16), dy[0], dy[1]);
                const u32x4 rs = make_rsrc_words(args.D + bwd_origin(pass, col0), bwd_rows(pass) * (Ne * 4u));
#pragma unroll
                for (int r = 0; r < 2; ++r) {
                    u32x4 du, dg;
#pragma unroll
                    for (int x = 0; x < 4; ++x) {
                        float gu[2], gg[2];
#pragma unroll
                        for (int hlf = 0; hlf < 2; ++hlf) {
                            const int sh = hlf * 16;
                            const float d = EL::from_bits((uint16_t)(dy[r][x] >> sh));
                            const float u = EL::from_bits((uint16_t)(bwd_h[pass][r][0][x] >> sh));
                            const float g = EL::from_bits((uint16_t)(bwd_h[pass][r][1][x] >> sh));
                            swiglu_b<typename EL::act_t>(g, u, d, gg[hlf], gu[hlf]);
                        }
                        du[x] = EL::pack2(gu[0], gu[1]);
                        dg[x] = EL::pack2(gg[0], gg[1]);
                    }
                    // The "gate" half's column offset goes into the per-lane offset, not into the instruction's scalar
                    // offset: a 16-byte store with a scalar-register offset whose first data register the next VALU
                    // instruction overwrites lost that dword in some lanes on this part, and the compiler leaves no wait state
                    // there (it does for stores with a constant scalar offset, as every other store of this library has).
                    const uint32_t off = bwd_offset(r, cols_valid);
                    const uint32_t off_gate = off == kOutOfRange ? kOutOfRange : off + Ne * 2u;
                    // (in assembly: the next tile's first wait counts these stores, so their number must be exactly this)
                    store_tile16_quiet_nt(rs, off, du);
                    store_tile16_quiet_nt(rs, off_gate, dg);
                }
            }
        };
        const uint32_t put_row = el & 15u, put_col = (el >> 4) * 4u;  // this lane's place in a 16 x 16 block
        uint32_t ypack[2][2][2];  // swiglu: the activation of two row blocks, which share one image: [block][column block][2]
        auto put_block = [&](int i) __attribute__((always_inline)) {
            const uint32_t r0 = block_row(i);  // first output row of this block
            const uint32_t rows_valid = r0 < Me ? (Me - r0 < 16u ? Me - r0 : 16u) : 0u;
            if constexpr (kSplit) {
                // the sums as they are: a lane's four consecutive columns of every 16 x 16 block, 64 bytes per row and block
                const uint32_t col0 = n0 + wn * WN;
                const uint32_t cols_valid = col0 < n_lim ? n_lim - col0 : 0u;
                float* const origin = args.partial + ((uint64_t)cur.part * args.rows + cur.row0 + r0) * Ne + col0;
                const __amdgpu_buffer_rsrc_t rs = make_rsrc(reinterpret_cast<const uint16_t*>(origin), rows_valid * (Ne * 4u));
#pragma unroll
                for (int j = 0; j < CB; ++j) {
                    const uint32_t col = j * 16 + put_col;
                    const uint32_t off = col < cols_valid ? put_row * (Ne * 4u) + col * 4u : kOutOfRange + (uint32_t)j * 16u;
                    const f32x16& c = acc[i];
                    store_tile16<false>(rs, off, uint4{__float_as_uint(c[4 * j]), __float_as_uint(c[4 * j + 1]),
                                                       __float_as_uint(c[4 * j + 2]), __float_as_uint(c[4 * j + 3])});
                }
            } else if constexpr (EPI == EPI_PLAIN || EPI == EPI_SWIGLU_BWD) {
                const uint32_t col0 = n0 + wn * WN;
                const uint32_t cols_valid = col0 < n_lim ? n_lim - col0 : 0u;
                uint2 w[CB];
#pragma unroll
                for (int j = 0; j < CB; ++j) {
                    const f32x16& c = acc[i];
                    w[j].x = EL::pack2(with_bias(c[4 * j + 0], j, 0), with_bias(c[4 * j + 1], j, 1));
                    w[j].y = EL::pack2(with_bias(c[4 * j + 2], j, 2), with_bias(c[4 * j + 3], j, 3));
                }
                if constexpr (EPI == EPI_PLAIN) {
#pragma unroll
                    for (int j = 0; j < CB; ++j) stage_put_quiet<WN * 2>(img, put_row, j * 16 + put_col, w[j]);
                    stage_flush_quiet<WN * 2, 16>(img, args.D + off_d + (uint64_t)r0 * Ne + col0, Ne, rows_valid, cols_valid, el,
                                                  stream_out);
                } else {
                    // The product (rounded) is the gradient of the activation; h and its gradient are [rows, 2 Ne] with "up" in
                    // columns 0.., "gate" in columns Ne... A pass is 16 rows x 64 columns: a lane takes 8 columns of two rows,
                    // fetches the 8 up and 8 gate values of each (requested two passes ahead), and stores both gradients.
                    constexpr int kAhead = kBwdAhead;
                    if (i == 0) {
#pragma unroll
                        for (int a = 0; a < kAhead; ++a) bwd_request(a, col0, cols_valid);
                    }
#pragma unroll
                    for (int j = 0; j < CB; ++j) stage_put_quiet<WN * 2>(img, put_row, j * 16 + put_col, w[j]);
                    bwd_finish(i, col0, cols_valid);
                    if (i + kAhead < RBX) bwd_request(i + kAhead, col0, cols_valid);
                }
            } else {
                // first the rounded pre-activation (32 "up" columns | 32 "gate" columns per row) of this row block, then,
                // after every second block, the activation of both
                constexpr int HB = WN * 2;
                constexpr int YB = WN;
                static_assert(CB == 4, "two up blocks and two gate blocks per wavefront and row block");
                const uint32_t col0 = n0 + wn * (WN / 2);
                const uint32_t cols_valid = col0 < n_lim ? n_lim - col0 : 0u;
                uint2 wu[2], wg[2];
#pragma unroll
                for (int jj = 0; jj < 2; ++jj) {
                    float u[4], g[4], y[4];
#pragma unroll
                    for (int x = 0; x < 4; ++x) {
                        u[x] = EL::round(with_bias(acc[i][4 * jj + x], jj, x));
                        g[x] = EL::round(with_bias(acc[i][4 * (2 + jj) + x], 2 + jj, x));
                        y[x] = u[x] * g[x] * sigmoid_for<typename EL::act_t>(g[x]);
                    }
                    ypack[i & 1][jj][0] = EL::pack2(y[0], y[1]);
                    ypack[i & 1][jj][1] = EL::pack2(y[2], y[3]);
                    if constexpr (EPI == EPI_SWIGLU) {
                        wu[jj].x = EL::pack2(u[0], u[1]);
                        wu[jj].y = EL::pack2(u[2], u[3]);
                        wg[jj].x = EL::pack2(g[0], g[1]);
                        wg[jj].y = EL::pack2(g[2], g[3]);
                    }
                }
                if constexpr (EPI == EPI_SWIGLU) {
#pragma unroll
                    for (int jj = 0; jj < 2; ++jj) {
                        stage_put_quiet<HB>(img, put_row, jj * 16 + put_col, wu[jj]);
                        stage_put_quiet<HB>(img, put_row, WN / 2 + jj * 16 + put_col, wg[jj]);
                    }
                    stage_flush_split_quiet<HB, 16, WN / 2>(img, args.D + off_d + (uint64_t)r0 * Ne + col0, Ne, rows_valid, cols_valid,
                                                            n_span, el);
                }
                // (the ninth block goes alone: the second half of its image is past its rows)
                if ((i & 1) || i == RB) {
                    const uint32_t row0 = i == RB ? r0 : r0 - 16u;  // first row of the pair of blocks
                    const uint32_t rows_pair = i == RB ? rows_valid : (row0 < Me ? (Me - row0 < 32u ? Me - row0 : 32u) : 0u);
#pragma unroll
                    for (int b = 0; b < (i == RB ? 1 : 2); ++b)
#pragma unroll
                        for (int jj = 0; jj < 2; ++jj) {
                            uint2 wy;
                            wy.x = ypack[b][jj][0];
                            wy.y = ypack[b][jj][1];
                            stage_put_quiet<YB>(img, b * 16 + put_row, jj * 16 + put_col, wy);
                        }
                    stage_flush_quiet<YB, 32>(img, args.ACT + off_d / 2 + (uint64_t)row0 * n_span + col0, n_span, rows_pair, cols_valid, el);
                }
            }
        };
#pragma unroll
        for (int i = 0; i < RB; ++i) put_block(i);
        if constexpr (TALL) {
            if (has_extra) put_block(RB);
        }

        // ---- on to the next tile ----
        streamed = stream_next;
        if (stream_next) {
            if constexpr (!GATHER) {
                fa_cur = fa_nxt;
                va_cur = va_nxt;
            }
            fb_cur = fb_nxt;
            vb_cur = vb_nxt;
        }
        cur = nxt;
        nxt = nn;
        ++round;
    }
}

template <typename EL, bool A_KC, bool B_KC, int EPI, bool VARY_K, bool BIAS, bool GATHER, bool TALL>
int launch(const Args& args, hipStream_t st) {
    int cus = num_compute_units();
    if (cus <= 0) cus = 256;
    hipLaunchKernelGGL((ragged_gemm_kernel<EL, A_KC, B_KC, EPI, VARY_K, BIAS, GATHER, TALL>), dim3((uint32_t)cus), dim3(NT), 0, st,
                       args);
    return launch_status("grouped_gemm_ragged");
}

// the forward (NT) kernels by epilogue, bias and gather
template <typename EL, int EPI, bool TALL>
int launch_forward_as(const Args& args, hipStream_t st) {
    const bool bias = args.bias != nullptr, gather = args.row_index != nullptr;
    if (bias && gather) return launch<EL, true, true, EPI, false, true, true, TALL>(args, st);
    if (bias) return launch<EL, true, true, EPI, false, true, false, TALL>(args, st);
    if (gather) return launch<EL, true, true, EPI, false, false, true, TALL>(args, st);
    return launch<EL, true, true, EPI, false, false, false, TALL>(args, st);
}

// The launches with varying rows and A's reduction contiguous, for at most kTallGroups groups (grouped_gemm_ragged_tall.hip).
// epi: EPI_PLAIN, EPI_SWIGLU, EPI_SWIGLU_ACT with B's reduction contiguous and any bias and gather; without them EPI_PLAIN and
// EPI_SPLIT in both layouts of B, and EPI_SWIGLU_BWD with B stored [reduction, out].
int launch_tall(const Args& args, int epi, bool b_kc, bool bf16, hipStream_t st);

// The parts of a split reduction (ragged_split.hip)
struct SplitPlan {
    uint32_t splits, steps;  // parts and K steps of each (even; the last part takes what is left); splits 1: no split
};
SplitPlan plan_split(int64_t R, int64_t E, int64_t N, int64_t K, bool b_kc, bool tall);
int launch_split_reduce(const Args& args, bool bf16, hipStream_t st);

}  // namespace ragged
}  // namespace gemm
}  // namespace fmahip
