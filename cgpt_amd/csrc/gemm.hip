// Dense contraction kernels for gfx950 (CDNA4): C[M,N] (+)= op(A)·op(B), 16-bit or
// fp32 inputs, fp32 accumulation on the matrix cores.
//
// One kernel family serves the three contractions of a linear layer
// (reference: src/ops/linear.cu:634-667, src/ops/backward/linear_backward.cu:268-285,
// where cuBLASLt does this work):
//   forward  Y  = X·Wᵀ      A[M,K] k-contiguous, B[N,K] k-contiguous
//   dX       dX = dY·W      A[M,K] k-contiguous, B[K,N] n-contiguous
//   dW       dW = dYᵀ·X     A[K,M] m-contiguous, B[K,N] n-contiguous
//
// Design
//   * 256 threads = 4 wavefronts in a 2x2 grid; a block owns a BM x BN tile of C
//     and walks K in tiles of 64, two MFMA steps each. Each wavefront owns (BM/2) x (BN/2) and issues
//     v_mfma_f32_16x16x32 (bf16 or f16): per flop that form moves half the accumulator
//     data of the 32x32x16 one, which counts on a chip whose clock is power-limited.
//   * The kernel is persistent: one block per CU slot walks its share of the work items
//     (output tile x K slice). The 8 XCDs (blocks are dealt round-robin to them) each take
//     a contiguous eighth of the items, ordered in groups of 8 tile-rows, so that the
//     tiles in flight on one XCD share A and B panels in that XCD's L2 (2 tile-rows for
//     the kernel whose epilogue reads and writes whole rows of a wider matrix).
//   * Operand tiles go global -> LDS with buffer_load ... lds (no staging registers, no
//     LDS stores, one loop-invariant per-lane offset) into a ring of LDS slots of one operand's
//     K tile each. A K tile takes 128 bytes of every row of a k-contiguous operand, whole cache lines: in
//     tiles of 64 bytes the path from L2 to LDS carries two thirds as much (0.25 instead of 0.17 us per 16 KiB
//     and CU), and that, not the matrix cores, was what a K step cost: 0.29 us per 128 x 128 tile, 0.23 now.
//     Forward [2048, 4096] x [4096, 4096] 77 -> 60 us, [32768, 1024] x [4096, 1024] 242 -> 227, dX 218 -> 205.
//     LDS rows cannot be padded that way; a chunk swizzle keeps the fragment reads conflict-free.
//   * Operands that are not k-contiguous in memory (dX's weight, both dW operands) sit
//     in LDS as they are in memory and are transposed by the LDS read itself
//     (ds_read_b64_tr_b16): no transpose pass over HBM, no VALU shuffles.
//   * The K loop is a software pipeline with one barrier per K tile whose issue order is
//     pinned in the source: every MFMA is followed by its share of the fragment reads (of the next step, into
//     registers of their own) and of the loads, and the
//     loop has no data-dependent branch (edges are clamped or zero-filled by the buffer
//     range check, never predicated).
//   * MFMA is issued as (B-fragment, A-fragment), so a lane ends up holding four
//     consecutive n for one m per accumulator; each wavefront stages its part of the
//     finished tile in a private piece of LDS and writes it out row by row (256
//     contiguous bytes per row), with bias / residual / old C added in fp32 and one
//     rounding to the dtype. The next item's first K tiles are requested meanwhile.
//   * dW has few output tiles and K = rows (32768): K is split into slices (work items),
//     fp32 partial tiles go to scratch and a second kernel adds them in slice order
//     (deterministic), applying accumulate and the dtype conversion.
//
// Operands whose rows are not whole aligned 16-byte chunks are copied to padded rows first;
// C may have any width and alignment (a store per element). fp32 storage takes the same kernels
// with v_mfma_f32_16x16x4_f32 and K steps of 16. Operands beyond 32-bit offsets, and unaligned ones
// of a caller that owns the arena or whose padded copies the arena has no room for, run on a general fp32 matrix-core kernel
// (v_mfma_f32_32x32x2_f32, register-staged operand tiles) with the same semantics.
#include "gemm_small.hpp"
#include "gemm_tiles.hpp"

#include <algorithm>
#include <cmath>
#include <cstdlib>

namespace cgptx {
namespace {

// LDS is a ring of slots of one operand's K tile each (two K steps: 128 bytes along K per row or column), A and B in turn:
// four slots hold the K tile being multiplied and the next one, the rest what is in flight beyond them. 256x256 blocks
// own a CU (5 x 32 KiB), 128x128 blocks run two per CU (5 x 16 KiB each) or, where there is no second one for a CU, one
// with 9 slots (two K tiles more in flight).
constexpr int kLdsSlots = 5, kDeepSlots = 9;
constexpr int kSteps = 2;  // K steps (of one MFMA each per 16 x 16 block) of a K tile

template <typename T, int BM, int BN, bool A_K, bool B_K, int SLOTS>
struct TileLayout {
    using ATile = std::conditional_t<A_K, KTile<T, BM, kSteps>, NTile<T, BM, kSteps>>;
    using BTile = std::conditional_t<B_K, KTile<T, BN, kSteps>, NTile<T, BN, kSteps>>;
    static constexpr int kSlot = ATile::kElems;  // elements
    static_assert(ATile::kElems == BTile::kElems, "both operands' tiles take any slot");
    static constexpr int kSlots = SLOTS;
    static constexpr int kSmemBytes = kSlots * kSlot * static_cast<int>(sizeof(T));
};

// Stores a lane's 16 bytes at voffset + soffset of a buffer. The sum is taken in the vector register: behind a 16-byte store
// with a scalar offset the compiler lets the very next instruction overwrite the data registers, and on this chip the store
// has then not always read them (128 x 128 tiles, two wavefronts a SIMD: the first four bytes of some hundred stores in a
// [32768, 768] result were the next value's). Without one it keeps the distance.
__device__ __forceinline__ void store_chunk(const u32x4& data, __amdgpu_buffer_rsrc_t rsrc, int voffset, int soffset) {
    __builtin_amdgcn_raw_buffer_store_b128(data, rsrc, voffset + soffset, 0, 0);
}

// One workgroup per CU slot walks its share of the work items (output tile x K slice) one after
// the other: the first K tiles of the next item are requested before the epilogue of the current
// one, whose stores then drain under the next item's MFMAs.
// SEGMENTED: A is stored [M, K] in up to three column segments (separate buffers along K).
// RESIDUAL: the epilogue adds a residual to a 16-bit result and nothing else (the output
// projections of a transformer block); a kernel of its own, so that each kernel carries one
// straight-line epilogue besides the general one.
// SWIGLU: B is the concatenated [gate; up] weight ([2·inter, K]) and C the concatenated [gate | up]
// activation; the kernel also writes silu(gate)·up. A tile's 256 columns are 128 gate columns and
// the 128 up columns of the same indices, interleaved in units of 64 so that each wavefront holds
// gate and up of its 64 indices in the same lanes: the B rows of an LDS tile are
// [gate 0-63 | up 0-63 | gate 64-127 | up 64-127] (one unit per load instruction of a wavefront,
// so only the scalar offsets of the loads change), and the epilogue computes the product from the
// rounded gate and up values, as the separate operator would from memory.
template <typename T, int BM, int BN, bool A_K, bool B_K, bool SPLIT, bool SEGMENTED, bool RESIDUAL = false,
          bool SWIGLU = false, bool GRAD = false, int SLOTS = kLdsSlots>
__global__ __launch_bounds__(kThreads) void gemm_mfma_kernel(KernelArgs p) {
    static_assert(!GRAD || (A_K && !B_K && !SPLIT && !SEGMENTED && !RESIDUAL && !SWIGLU && BN == 256),
                  "the SwiGLU gradient epilogue belongs to the plain input-gradient kernel with 256-wide tiles");
    static_assert(!SEGMENTED || (A_K && !SPLIT), "segments along K are read by the unsplit kernels only");
    static_assert(!RESIDUAL || (!SPLIT && !SEGMENTED), "the residual epilogue belongs to plain unsplit kernels");
    static_assert(!SWIGLU || (A_K && B_K && !SPLIT && !SEGMENTED && !RESIDUAL && BN == 256),
                  "the SwiGLU epilogue belongs to the plain forward kernel with 256-wide tiles");
    using frag_t = typename Mfma<T>::frag;
    using Layout = TileLayout<T, BM, BN, A_K, B_K, SLOTS>;
    using ATile = typename Layout::ATile;
    using BTile = typename Layout::BTile;
    static_assert(BM == BN, "the epilogue staging assumes square tiles");
    constexpr int WM = BM / 2, WN = BN / 2;
    constexpr int TM = WM / 16, TN = WN / 16;  // 16 x 16 MFMA blocks of a wavefront's part
    extern __shared__ __align__(1024) unsigned char smem_raw[];
    T* smem = reinterpret_cast<T*>(smem_raw);
    // Operand tile o of an item (o even: A's K tile o/2, odd: B's) lives in slot o % kSlots.
    constexpr int kSlot = Layout::kSlot;
    constexpr int kSlots = Layout::kSlots;
    constexpr int kAhead = (kSlots - 1) / 2;  // K tiles between the one being multiplied and the one being requested
    static_assert(kSlots % 2 == 1 && kSlots >= 5, "an odd number of slots: first steps request A, second steps B");
    constexpr unsigned int kSlotBytes = kSlot * sizeof(T);

    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int wm = wave >> 1, wn = wave & 1;

    // Work items are numbered slice-major (all tiles of K slice 0, then of slice 1, ...), tiles in
    // groups of 1 << group_rows_log2 tile-rows, down the rows first. Blocks are dealt round-robin to the 8
    // XCDs, so XCD x takes the x-th eighth of the items and its blocks walk it side by side: the
    // items in flight on one XCD are neighbours and share A and B panels in that XCD's L2.
    const int tiles = p.tiles_m * p.tiles_n;
    const int items = tiles * p.slices;
    const int per_xcd = (items + kXcds - 1) / kXcds;
    const int item_stride = gridDim.x / kXcds;
    const int item_end = min(items, static_cast<int>(blockIdx.x % kXcds + 1) * per_xcd);
    int item = static_cast<int>(blockIdx.x % kXcds) * per_xcd + static_cast<int>(blockIdx.x / kXcds);
    if (item >= item_end) return;

    struct Item {
        int m0, n0, slice, kt_begin, kt_end;
    };
    auto locate = [&](int index) __attribute__((always_inline)) {
        // Integer divisions by run-time values cost some thirty scalar instructions each, with
        // nothing to hide them between two items: unsplit launches skip the first, the second is a
        // multiplication by a reciprocal the host prepared, the third a shift in all but the last,
        // ragged group of tile rows.
        Item w;
        w.slice = p.slices == 1 ? 0 : index / tiles;
        const int logical = index - w.slice * tiles;
        const int group_rows = 1 << p.group_rows_log2;
        const int group_size = p.tiles_n << p.group_rows_log2;
        const int group = p.group_reciprocal != 0u
                              ? static_cast<int>(__umulhi(static_cast<unsigned int>(logical), p.group_reciprocal))
                              : logical / group_size;
        const int first_m = group << p.group_rows_log2;
        const int rows_in_group = min(p.tiles_m - first_m, group_rows);
        const int in_group = logical - group * group_size;
        const int column = rows_in_group == group_rows ? in_group >> p.group_rows_log2 : in_group / rows_in_group;
        w.m0 = (first_m + in_group - column * rows_in_group) * BM;
        w.n0 = column * BN;
        w.kt_begin = w.slice * p.k_tiles_per_slice;
        w.kt_end = min(p.k_tiles, w.kt_begin + p.k_tiles_per_slice);
        return w;
    };

    // The operand sources of the item whose K tiles are being requested. A may be given as up to
    // three column segments in separate buffers. Stored [M, K]: the K range is segmented and the
    // source changes along the K loop (boundaries a_end0 / a_end1). Stored [K, M]: the M range is
    // segmented and the item's rows pick their buffer once.
    ATile a_src, a_src1, a_src2;
    BTile b_src;
    int a_end0 = std::numeric_limits<int>::max(), a_end1 = std::numeric_limits<int>::max();
    int src_begin = 0, src_end = 0;  // K steps of that item
    auto open = [&](const Item& w) __attribute__((always_inline)) {
        const int m0 = w.m0, n0 = w.n0;
        src_begin = w.kt_begin;
        src_end = w.kt_end;
        long b_shift = 0;
        if constexpr (A_K && !SEGMENTED) {
            a_src.init(static_cast<const T*>(p.a) + static_cast<long>(m0) * p.lda, p.lda, p.a_extent - m0, p.k, wave);
        } else if constexpr (A_K) {
            // All three sources are set up unconditionally (absent segments repeat the first and
            // are never selected): conditional set-up would be merged into one piece of code that
            // writes through a pointer, which keeps the sources in memory.
            const int segments = p.a_seg.count;
            const void* ptr0 = segments == 0 ? p.a : p.a_seg.ptr[0];
            const long ld0 = segments == 0 ? p.lda : p.a_seg.ld[0];
            const int cols0 = segments == 0 ? p.k : p.a_seg.cols[0];
            const void* ptr1 = segments > 1 ? p.a_seg.ptr[1] : ptr0;
            const long ld1 = segments > 1 ? p.a_seg.ld[1] : ld0;
            const int cols1 = segments > 1 ? p.a_seg.cols[1] : cols0;
            const void* ptr2 = segments > 2 ? p.a_seg.ptr[2] : ptr0;
            const long ld2 = segments > 2 ? p.a_seg.ld[2] : ld0;
            const int cols2 = segments > 2 ? p.a_seg.cols[2] : cols0;
            a_src.init(static_cast<const T*>(ptr0) + static_cast<long>(m0) * ld0, ld0, p.m - m0, cols0, wave);
            a_src1.init(static_cast<const T*>(ptr1) + static_cast<long>(m0) * ld1, ld1, p.m - m0, cols1, wave);
            a_src2.init(static_cast<const T*>(ptr2) + static_cast<long>(m0) * ld2, ld2, p.m - m0, cols2, wave);
            a_end0 = segments > 1 ? cols0 : std::numeric_limits<int>::max();
            a_end1 = segments > 2 ? cols0 + cols1 : std::numeric_limits<int>::max();
        } else {
            // Stacked products: the tile's rows of C name the product, and the operands move with it.
            long product = 0;
            int local_m0 = m0, rows = p.a_extent;
            if constexpr (!B_K) {
                if (p.batch_rows > 0) {
                    product = m0 / p.batch_rows;
                    local_m0 = m0 - static_cast<int>(product) * p.batch_rows;
                    rows = p.batch_rows;
                    b_shift = product * p.b_batch_stride;
                }
            }
            const T* base = static_cast<const T*>(p.a) + product * p.a_batch_stride;
            long ld = p.lda;
            int first = 0, width = rows;
            if (p.a_seg.count > 0) {
                const SegmentPick pick = pick_segment(p.a_seg, local_m0);
                const long stride = pick.index == 2 ? p.a_seg_batch_stride[2]
                                    : pick.index == 1 ? p.a_seg_batch_stride[1] : p.a_seg_batch_stride[0];
                base = static_cast<const T*>(pick.ptr) + product * stride;
                ld = pick.ld;
                first = pick.first;
                width = pick.cols;
            }
            a_src.init(base + (local_m0 - first), ld, width - (local_m0 - first), p.k, wave);
        }
        if constexpr (SWIGLU) b_src.init(static_cast<const T*>(p.b) + static_cast<long>(n0 / 2) * p.ldb, p.ldb, p.n - n0 / 2, p.k, wave);
        else if constexpr (B_K) b_src.init(static_cast<const T*>(p.b) + static_cast<long>(n0) * p.ldb, p.ldb, p.b_extent - n0, p.b_k, wave);
        else b_src.init(static_cast<const T*>(p.b) + b_shift + n0, p.ldb, p.b_extent - n0, p.b_k, wave);
    };
    // K tiles past the end of the slice are still "loaded" (the loop stays free of data-dependent
    // branches and every wavefront always has the same number of loads in flight), but from an
    // offset beyond the buffer: the range check answers those at once with zeros, no memory traffic. What the last K tile
    // holds past an odd number of K steps is never multiplied.
    // The source of a tile is picked with scalar selects, not branches, so that the loads can be
    // issued one by one between MFMAs.
    auto aim_a = [&](int t, TileCursor& ca) __attribute__((always_inline)) {
        const unsigned int past_end = src_begin + t * kSteps >= src_end ? 0x80000000u : 0u;
        const int k0 = min(src_begin + t * kSteps, src_end - 1) * kBK<T>;
        if constexpr (SEGMENTED) {
            // Values first, then selects: a conditional between the objects' members would select
            // an address and keep all three sources in memory.
            const bool in1 = k0 >= a_end0, in2 = k0 >= a_end1;
            const u32x4 rsrc0 = a_src.rsrc, rsrc1 = a_src1.rsrc, rsrc2 = a_src2.rsrc;
            const int voffset0 = a_src.voffset, voffset1 = a_src1.voffset, voffset2 = a_src2.voffset;
            const unsigned int bytes0 = a_src.group_bytes, bytes1 = a_src1.group_bytes, bytes2 = a_src2.group_bytes;
            const int end0 = a_end0, end1 = a_end1;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const unsigned int w0 = rsrc0[e], w1 = rsrc1[e], w2 = rsrc2[e];
                ca.rsrc[e] = in2 ? w2 : in1 ? w1 : w0;
            }
            ca.voffset = in2 ? voffset2 : in1 ? voffset1 : voffset0;
            const unsigned int group_bytes = in2 ? bytes2 : in1 ? bytes1 : bytes0;
            const int start = in2 ? end1 : in1 ? end0 : 0;
            ca.soffset = (wave * group_bytes + (k0 - start) * static_cast<unsigned int>(sizeof(T))) | past_end;
            ca.step = kWaves * group_bytes;
        } else {
            ca.rsrc = a_src.rsrc;
            ca.voffset = a_src.voffset;
            ca.soffset = a_src.first_offset(k0, wave) | past_end;
            ca.step = kWaves * a_src.group_bytes;
        }
    };
    auto aim_b = [&](int t, TileCursor& cb) __attribute__((always_inline)) {
        const unsigned int past_end = src_begin + t * kSteps >= src_end ? 0x80000000u : 0u;
        const int k0 = min(src_begin + t * kSteps, src_end - 1) * kBK<T>;
        cb.rsrc = b_src.rsrc;
        cb.voffset = b_src.voffset;
        cb.soffset = b_src.first_offset(k0, wave) | past_end;
        cb.step = kWaves * b_src.group_bytes;
        if constexpr (SWIGLU) {
            // Two loads per unit of 64 rows: gate unit, up unit of the same rows (inter rows further), then back and 64
            // rows on.
            const unsigned int up = __builtin_amdgcn_readfirstlane(
                static_cast<unsigned int>(static_cast<long>(p.inter) * p.ldb * static_cast<long>(sizeof(T))));
            cb.step_up = up - cb.step;
            cb.step_back = cb.step - up;
        }
    };
    // Load l of an operand tile into the slot whose LDS address, advanced to this wavefront's first 1 KiB, is
    // slot_lds. One load fills 1 KiB; the wavefronts' loads interleave, so a wavefront's consecutive ones are
    // kWaves KiB apart.
    constexpr int kLoadBytes = 64 * 16;
    constexpr int kLoads = ATile::kLoads;  // per wavefront and operand tile
    static_assert(ATile::kLoads == BTile::kLoads && kSlots * kLoads < 64, "the vmcnt waits count either operand's loads");
    auto issue_a = [&](auto index, unsigned int slot_lds, TileCursor& ca) __attribute__((always_inline)) {
        constexpr int l = decltype(index)::value;
        ca.soffset = load_to_lds<l * kWaves * kLoadBytes>(ca.rsrc, slot_lds, ca.voffset, ca.soffset, ca.step);
    };
    auto issue_b = [&](auto index, unsigned int slot_lds, TileCursor& cb) __attribute__((always_inline)) {
        constexpr int l = decltype(index)::value;
        const unsigned int step = !SWIGLU || l % 2 == 0 ? cb.step : l % 4 == 1 ? cb.step_up : cb.step_back;
        cb.soffset = load_to_lds<l * kWaves * kLoadBytes>(cb.rsrc, slot_lds, cb.voffset, cb.soffset, step);
    };
    const unsigned int lds_wave = lds_address_of(smem) + wave * kLoadBytes;
    TileCursor ca, cb;
    // Requests operand tiles FIRST .. LAST-1 of the opened item into the slots of the same numbers.
    auto request_tiles = [&]<int FIRST, int LAST>() __attribute__((always_inline)) {
        static_for<FIRST, LAST>([&](auto index) {
            constexpr int o = decltype(index)::value;
            if constexpr (o % 2 == 0) {
                aim_a(o / 2, ca);
                static_for<0, kLoads>([&](auto l) { issue_a(l, lds_wave + o * kSlotBytes, ca); });
            } else {
                aim_b(o / 2, cb);
                static_for<0, kLoads>([&](auto l) { issue_b(l, lds_wave + o * kSlotBytes, cb); });
            }
        });
    };

    // Per-lane LDS offsets of the fragments: one per K step for a k-contiguous operand (the block is a
    // scalar offset), one per 16-column block for an n-contiguous one (the swizzle depends on it).
    constexpr int kAOffsets = A_K ? kSteps : TM, kBOffsets = B_K ? kSteps : TN;
    int a_off[kAOffsets], b_off[kBOffsets];
#pragma unroll
    for (int i = 0; i < kAOffsets; ++i) a_off[i] = A_K ? ATile::lane_offset(lane, i) : ATile::lane_offset(lane, wm * WM + i * 16);
#pragma unroll
    for (int j = 0; j < kBOffsets; ++j) b_off[j] = B_K ? BTile::lane_offset(lane, j) : BTile::lane_offset(lane, wn * WN + j * 16);

    // Fragments of the K step being multiplied and of the next one: step s of a K tile is in af[s], bf[s].
    acc_t acc[TM][TN];
    frag_t af[kSteps][TM], bf[kSteps][TN];
    constexpr int kFrags = TM + TN;
    // The F-th fragment in the order of first use (A's block 0, B's blocks, A's other blocks) of K step STEP.
    auto read_frag = [&]<int STEP, int F>(const T* a_tile, const T* b_tile) __attribute__((always_inline)) {
        if constexpr (F >= 1 && F <= TN) {
            constexpr int j = F - 1;
            if constexpr (B_K) bf[STEP][j] = BTile::frag(b_tile, wn * WN + j * 16, b_off[STEP]);
            else bf[STEP][j] = BTile::frag(b_tile + STEP * BTile::kStepElems, b_off[j]);
        } else {
            constexpr int i = F == 0 ? 0 : F - TN;
            if constexpr (A_K) af[STEP][i] = ATile::frag(a_tile, wm * WM + i * 16, a_off[STEP]);
            else af[STEP][i] = ATile::frag(a_tile + STEP * ATile::kStepElems, a_off[i]);
        }
    };

    // Epilogue staging. acc[i][j][e] holds C[m, n] with m = lane%16, n = 4*(lane/16) + e, relative
    // to the 16 x 16 block (i, j) of the wavefront's WM x WN part of the tile. Each wavefront passes
    // its part through a private quarter of the last LDS slot (the only one the first operand tiles of
    // the next item do not fill), 32 rows at a time, and stores it row by row: whole contiguous
    // row segments of C per instruction instead of 32 separate 8-byte pieces, and no workgroup
    // barrier. When bias, residual or the old C are added (or the output is fp32 / a split-K
    // partial) the staging is fp32, half the columns per pass, and rounding to the storage dtype
    // still happens once, after the additions; otherwise the values are rounded in registers and
    // staged in the storage dtype. A staged row is kRowBytes long; its 16-byte chunk c sits at
    // chunk position c ^ sw(row), which spreads both the column-wise writes and the row-wise reads
    // over all banks.
    constexpr bool kIsF32 = std::is_same_v<T, float>;
    static_assert(!kIsF32 || (BM <= 128 && !SEGMENTED && !RESIDUAL && !SWIGLU && !GRAD), "fp32 storage has the plain kernels only");
    constexpr int kRowBytes = WN * 2;  // fp32 values always pass in two halves
    constexpr int kRowChunks = kRowBytes / 16;
    static_assert(32 * kRowBytes * kWaves == static_cast<int>(kSlotBytes), "staging is a quarter slot per wavefront");
    unsigned char* region = smem_raw + (kSlots - 1) * kSlotBytes + wave * (kSlotBytes / kWaves);
    auto sw = [](int row) { return (row / (256 / kRowBytes)) % kRowChunks; };
    const int m_lane = lane & 15, q_lane = lane >> 4;
    // Writes blocks (2r, j0 .. j0+JP-1) and (2r+1, ...) into the wavefront's staging region as element type S.
    auto stage = [&]<typename S, int JP>(int r, int j0) __attribute__((always_inline)) {
        static_assert(JP * 16 * sizeof(S) == kRowBytes, "a pass fills whole staged rows");
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int ii = 0; ii < 2; ++ii) {
            const int row = ii * 16 + m_lane;
            unsigned char* write_row = region + row * kRowBytes;
#pragma unroll
            for (int jj = 0; jj < JP; ++jj) {
                // Read out of the accumulator registers here and now: left to the register allocator,
                // some kernels copy all 256 accumulators to vector registers right after the K loop
                // and spill what does not fit.
                acc_t v;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    float x = acc[2 * r + ii][j0 + jj][e];
                    if constexpr (!kIsF32) asm volatile("v_accvgpr_read_b32 %0, %1" : "=v"(x) : "a"(x));
                    v[e] = x;
                }
                const int byte = (jj * 16 + q_lane * 4) * static_cast<int>(sizeof(S));
                unsigned char* slot = write_row + (((byte / 16) ^ sw(row)) * 16) + byte % 16;
                if constexpr (std::is_same_v<S, float>) *reinterpret_cast<vec_t<float, 4>*>(slot) = v;
                else store_vec<T, 4>(reinterpret_cast<T*>(slot), vec_from_f32<T, 4>(v));
            }
        }
        __builtin_amdgcn_wave_barrier();
    };
    // Stages those blocks, 32 rows, and hands each lane 8 consecutive staged elements at a time:
    // consume(round, row, col, pointer to the 8 elements' first chunk, to the second chunk when S is
    // float), row/col relative to the wavefront's part; in round u the lane gets element
    // q = 64 u + lane of the 32 x (8-element groups per row) grid, row-major.
    auto pass = [&]<typename S, int JP>(int r, int j0, auto&& consume) __attribute__((always_inline)) {
        stage.template operator()<S, JP>(r, j0);
        constexpr int kLanesPerRow = kRowBytes / (8 * static_cast<int>(sizeof(S)));
        constexpr int kChunksPerLane = 8 * static_cast<int>(sizeof(S)) / 16;
        constexpr int kRounds = 32 * kLanesPerRow / kWave;
#pragma unroll
        for (int u = 0; u < kRounds; ++u) {
            const int q = u * kWave + lane;
            const int row = q / kLanesPerRow, part = q % kLanesPerRow;
            const unsigned char* base = region + row * kRowBytes;
            const int first = part * kChunksPerLane;
            consume(u, r * 32 + row, j0 * 16 + part * 8, base + ((first ^ sw(row)) * 16),
                    base + (((first + kChunksPerLane - 1) ^ sw(row)) * 16));
        }
    };
    constexpr int kRowBlocks = WM / 32;  // 32-row blocks of a wavefront's part
    auto request_share = [&](int r) __attribute__((always_inline)) {
        static_for<0, kRowBlocks>([&](auto index) {
            constexpr int block = decltype(index)::value;
            if (r == block)
                request_tiles.template operator()<block * (kSlots - 1) / kRowBlocks, (block + 1) * (kSlots - 1) / kRowBlocks>();
        });
    };
    // Before 32-row block r of the tile is staged and stored, its share of the first K tiles of the next item
    // are requested (if there is one): a burst of requests would hold the wavefront up for as long as
    // the memory system takes to accept them, between the stores it costs nothing.
    auto store_tile = [&](const Item& w, bool request) __attribute__((always_inline)) {
        // C may be given as column segments too: this tile's columns then belong to one of them.
        void* c_base = p.c;
        long c_ld = p.ldc;
        int c_col0 = w.n0, c_cols = p.n;
        if (p.c_seg.count > 0) {
            const SegmentPick pick = pick_segment(p.c_seg, w.n0);
            c_base = const_cast<void*>(pick.ptr);
            c_ld = pick.ld;
            c_col0 = w.n0 - pick.first;
            c_cols = pick.cols;
        }
        const int row0 = w.m0 + wm * WM, col0 = wn * WN;  // of the wavefront's part; columns relative to n0
        // The two fp32-staged cases of the training step get straight-line code as well: split-K
        // partial tiles (nothing added, fp32 out) and a residual added to a 16-bit result. Half the
        // columns are staged per pass; lane l of round u holds 8 consecutive columns (group l%8) of
        // row 8u + l/8.
        constexpr int kGroups = WN / 2 / 8, kRowsF = kWave / kGroups, kRoundsF = 32 / kRowsF;
        const int f_row = lane / kGroups, f_col = (lane % kGroups) * 8;  // f_col within the staged half
        auto read_staged = [&](int u, vec_t<float, 4>& v0, vec_t<float, 4>& v1) __attribute__((always_inline)) {
            const int row = u * kRowsF + f_row;
            const unsigned char* base = region + row * kRowBytes;
            v0 = *reinterpret_cast<const vec_t<float, 4>*>(base + (((f_col / 4) ^ sw(row)) * 16));
            v1 = *reinterpret_cast<const vec_t<float, 4>*>(base + (((f_col / 4 + 1) ^ sw(row)) * 16));
        };
        // The same staged half, dealt out so that every store instruction of fp32 values covers whole cache lines: lane l
        // of round u takes columns 4 (l % 8) .. + 3 and, for its second store, the four columns 32 further on, of row
        // 8u + l/8 (with eight consecutive fp32 columns per lane, each store instruction would write every other 16 bytes
        // of a line, and lines reach memory in parts).
        const int l_col = (lane % kGroups) * 4;  // first column of the lane's first quad within the staged half
        auto read_staged_lines = [&](int u, vec_t<float, 4>& v0, vec_t<float, 4>& v1) __attribute__((always_inline)) {
            const int row = u * kRowsF + f_row;
            const unsigned char* base = region + row * kRowBytes;
            v0 = *reinterpret_cast<const vec_t<float, 4>*>(base + (((l_col / 4) ^ sw(row)) * 16));
            v1 = *reinterpret_cast<const vec_t<float, 4>*>(base + (((l_col / 4 + kGroups) ^ sw(row)) * 16));
        };
        // Descriptor over a wavefront's part of a row-major matrix (see the 16-bit case above).
        auto part_rsrc = [&](const void* origin, long ld, int elem, int rows_left, int cols_left) __attribute__((always_inline)) {
            const long extent = rows_left > 0 && cols_left > 0 ? (static_cast<long>(rows_left - 1) * ld + cols_left) * elem : 0;
            return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(origin), 0, static_cast<int>(extent), 0x00020000);
        };
        const int rows_left = min(WM, p.m - row0);
        if constexpr (SWIGLU) {
            // The wavefront's 128 staged columns are gate g0 .. g0+63 and up g0 .. g0+63. Lane l of
            // round u takes 8 gate and the 8 matching up values of row 8u + l/8 from the staging
            // region, stores both where the concatenated layout wants them, and the product beside.
            const int g0 = w.n0 / 2 + wn * (WN / 2);
            const int cols_left = min(WN / 2, p.inter - g0);
            const T* c_origin = static_cast<const T*>(p.c) + static_cast<long>(row0) * p.ldc + g0;
            const __amdgpu_buffer_rsrc_t gate_rsrc = part_rsrc(c_origin, p.ldc, sizeof(T), rows_left, cols_left);
            const __amdgpu_buffer_rsrc_t up_rsrc = part_rsrc(c_origin + p.inter, p.ldc, sizeof(T), rows_left, cols_left);
            const __amdgpu_buffer_rsrc_t act_rsrc = part_rsrc(static_cast<const T*>(p.act) + static_cast<long>(row0) * p.ld_act + g0,
                                                              p.ld_act, sizeof(T), rows_left, cols_left);
            const int c_row_bytes = static_cast<int>(p.ldc * static_cast<long>(sizeof(T)));
            const int act_row_bytes = static_cast<int>(p.ld_act * static_cast<long>(sizeof(T)));
            const bool live = f_col < cols_left;
            const int c_voffset = live ? f_row * c_row_bytes + f_col * static_cast<int>(sizeof(T)) : std::numeric_limits<int>::min();
            const int act_voffset = live ? f_row * act_row_bytes + f_col * static_cast<int>(sizeof(T)) : std::numeric_limits<int>::min();
#pragma unroll
            for (int r = 0; r < kRowBlocks; ++r) {
                __builtin_amdgcn_sched_barrier(0);
                if (request) request_share(r);
                stage.template operator()<T, TN>(r, 0);
                u32x4 gate[kRoundsF], up[kRoundsF];
#pragma unroll
                for (int u = 0; u < kRoundsF; ++u) {
                    const int row = u * kRowsF + f_row;
                    const unsigned char* base = region + row * kRowBytes;
                    gate[u] = *reinterpret_cast<const u32x4*>(base + (((f_col / 8) ^ sw(row)) * 16));
                    up[u] = *reinterpret_cast<const u32x4*>(base + (((kGroups + f_col / 8) ^ sw(row)) * 16));
                }
#pragma unroll
                for (int u = 0; u < kRoundsF; ++u) {
                    const int row = r * 32 + u * kRowsF;
                    store_chunk(gate[u], gate_rsrc, c_voffset, row * c_row_bytes);
                    store_chunk(up[u], up_rsrc, c_voffset, row * c_row_bytes);
                    const vec_t<float, 8> g = vec_to_f32<T, 8>(__builtin_bit_cast(vec_t<T, 8>, gate[u]));
                    const vec_t<float, 8> v = vec_to_f32<T, 8>(__builtin_bit_cast(vec_t<T, 8>, up[u]));
                    vec_t<float, 8> product;
#pragma unroll
                    for (int e = 0; e < 8; ++e) product[e] = g[e] * (1.0f / (1.0f + __expf(-g[e]))) * v[e];
                    store_chunk(__builtin_bit_cast(u32x4, vec_from_f32<T, 8>(product)), act_rsrc,
                                                           act_voffset, row * act_row_bytes);
                }
            }
            return;
        }
        if constexpr (GRAD) {
            // The contraction is the gradient of silu(gate)·up; what is written is the gradient of
            // [gate | up]: dgate = d·up·s·(1 + gate·(1 - s)), dup = d·gate·s with s = sigmoid(gate),
            // from d rounded to the storage dtype (the bits the separate operator reads) and the
            // forward's saved gate and up. The tile is staged in the storage dtype; lane l of round u
            // holds 8 consecutive columns (chunk l%16) of row 4u + l/16, loads the matching gate and up
            // values one 32-row block ahead and stores both gradients.
            const int g0 = w.n0 + col0;  // first gate column of the wavefront's part
            const int cols_left = min(WN, p.inter - g0);
            const T* out_origin = static_cast<const T*>(p.c) + static_cast<long>(row0) * p.ldc + g0;
            const T* in_origin = static_cast<const T*>(p.saved) + static_cast<long>(row0) * p.ld_saved + g0;
            const __amdgpu_buffer_rsrc_t dgate_rsrc = part_rsrc(out_origin, p.ldc, sizeof(T), rows_left, cols_left);
            const __amdgpu_buffer_rsrc_t dup_rsrc = part_rsrc(out_origin + p.inter, p.ldc, sizeof(T), rows_left, cols_left);
            const __amdgpu_buffer_rsrc_t gate_rsrc = part_rsrc(in_origin, p.ld_saved, sizeof(T), rows_left, cols_left);
            const __amdgpu_buffer_rsrc_t up_rsrc = part_rsrc(in_origin + p.inter, p.ld_saved, sizeof(T), rows_left, cols_left);
            constexpr int kLanesPerRow = kRowBytes / 16, kRowsPerRound = kWave / kLanesPerRow, kRounds = 32 / kRowsPerRound;
            const int lane_row = lane / kLanesPerRow, lane_chunk = lane % kLanesPerRow;
            const int out_row_bytes = static_cast<int>(p.ldc * static_cast<long>(sizeof(T)));
            const int in_row_bytes = static_cast<int>(p.ld_saved * static_cast<long>(sizeof(T)));
            const bool live = lane_chunk * 8 < cols_left;
            const int out_voffset = live ? lane_row * out_row_bytes + lane_chunk * 16 : std::numeric_limits<int>::min();
            const int in_voffset = live ? lane_row * in_row_bytes + lane_chunk * 16 : std::numeric_limits<int>::min();
            u32x4 ahead[2][2][kRounds];
            auto request_saved = [&](int r, u32x4 (&into)[2][kRounds]) __attribute__((always_inline)) {
#pragma unroll
                for (int u = 0; u < kRounds; ++u) {
                    const int soffset = (r * 32 + u * kRowsPerRound) * in_row_bytes;
                    into[0][u] = __builtin_amdgcn_raw_buffer_load_b128(gate_rsrc, in_voffset, soffset, 0);
                    into[1][u] = __builtin_amdgcn_raw_buffer_load_b128(up_rsrc, in_voffset, soffset, 0);
                }
            };
            request_saved(0, ahead[0]);
#pragma unroll
            for (int r = 0; r < kRowBlocks; ++r) {
                __builtin_amdgcn_sched_barrier(0);
                if (request) request_share(r);
                if (r + 1 < kRowBlocks) request_saved(r + 1, ahead[(r + 1) & 1]);
                stage.template operator()<T, TN>(r, 0);
                u32x4 data[kRounds];
#pragma unroll
                for (int u = 0; u < kRounds; ++u) {
                    const int row = u * kRowsPerRound + lane_row;
                    data[u] = *reinterpret_cast<const u32x4*>(region + row * kRowBytes + ((lane_chunk ^ sw(row)) * 16));
                }
#pragma unroll
                for (int u = 0; u < kRounds; ++u) {
                    const vec_t<float, 8> d = vec_to_f32<T, 8>(__builtin_bit_cast(vec_t<T, 8>, data[u]));
                    const vec_t<float, 8> g = vec_to_f32<T, 8>(__builtin_bit_cast(vec_t<T, 8>, ahead[r & 1][0][u]));
                    const vec_t<float, 8> v = vec_to_f32<T, 8>(__builtin_bit_cast(vec_t<T, 8>, ahead[r & 1][1][u]));
                    vec_t<float, 8> dg, du;
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        const float sg = 1.0f / (1.0f + __expf(-g[e]));
                        dg[e] = d[e] * v[e] * (sg * (1.0f + g[e] * (1.0f - sg)));
                        du[e] = d[e] * (g[e] * sg);
                    }
                    const int soffset = (r * 32 + u * kRowsPerRound) * out_row_bytes;
                    store_chunk(__builtin_bit_cast(u32x4, vec_from_f32<T, 8>(dg)), dgate_rsrc, out_voffset, soffset);
                    store_chunk(__builtin_bit_cast(u32x4, vec_from_f32<T, 8>(du)), dup_rsrc, out_voffset, soffset);
                }
            }
            return;
        }
        if constexpr (RESIDUAL) {
            const int cols_left = min(WN, c_cols - (c_col0 + col0));
            const T* out_origin = static_cast<const T*>(c_base) + static_cast<long>(row0) * c_ld + (c_col0 + col0);
            const T* res_origin = static_cast<const T*>(p.residual) + static_cast<long>(row0) * p.ldr + (w.n0 + col0);
            const __amdgpu_buffer_rsrc_t out_rsrc = part_rsrc(out_origin, c_ld, sizeof(T), rows_left, cols_left);
            const __amdgpu_buffer_rsrc_t res_rsrc = part_rsrc(res_origin, p.ldr, sizeof(T), rows_left, cols_left);
            const int out_row_bytes = static_cast<int>(c_ld * static_cast<long>(sizeof(T)));
            const int res_row_bytes = static_cast<int>(p.ldr * static_cast<long>(sizeof(T)));
            // The residual of a 32-row block is requested one block ahead (the first one before
            // anything is staged): its memory round trip passes under the previous block's work.
            u32x4 ahead[2][2][kRoundsF];
            auto request_residual = [&](int r, u32x4 (&into)[2][kRoundsF]) __attribute__((always_inline)) {
#pragma unroll
                for (int half = 0; half < 2; ++half) {
                    const int col = half * (WN / 2) + f_col;
                    const int voffset = col < cols_left ? f_row * res_row_bytes + col * static_cast<int>(sizeof(T))
                                                        : std::numeric_limits<int>::min();
#pragma unroll
                    for (int u = 0; u < kRoundsF; ++u)
                        into[half][u] = __builtin_amdgcn_raw_buffer_load_b128(res_rsrc, voffset, (r * 32 + u * kRowsF) * res_row_bytes, 0);
                }
            };
            request_residual(0, ahead[0]);
#pragma unroll
            for (int r = 0; r < kRowBlocks; ++r) {
                __builtin_amdgcn_sched_barrier(0);
                if (request) request_share(r);
                if (r + 1 < kRowBlocks) request_residual(r + 1, ahead[(r + 1) & 1]);
#pragma unroll
                for (int half = 0; half < 2; ++half) {
                    stage.template operator()<float, TN / 2>(r, half * (TN / 2));
                    const int col = half * (WN / 2) + f_col;
                    const int voffset = col < cols_left ? f_row * out_row_bytes + col * static_cast<int>(sizeof(T))
                                                        : std::numeric_limits<int>::min();
                    vec_t<float, 4> v0[kRoundsF], v1[kRoundsF];
#pragma unroll
                    for (int u = 0; u < kRoundsF; ++u) read_staged(u, v0[u], v1[u]);
#pragma unroll
                    for (int u = 0; u < kRoundsF; ++u) {
                        const vec_t<float, 8> add = vec_to_f32<T, 8>(__builtin_bit_cast(vec_t<T, 8>, ahead[r & 1][half][u]));
                        vec_t<float, 8> sum;
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            sum[e] = v0[u][e] + add[e];
                            sum[4 + e] = v1[u][e] + add[4 + e];
                        }
                        store_chunk(__builtin_bit_cast(u32x4, vec_from_f32<T, 8>(sum)), out_rsrc, voffset,
                                                               (r * 32 + u * kRowsF) * out_row_bytes);
                    }
                }
            }
            return;
        }
        bool plain = false;
        if constexpr (!SPLIT) plain = p.bias == nullptr && p.residual == nullptr && p.addend == nullptr && !p.accumulate && !p.c_f32 && !p.ragged;
        if constexpr (!kIsF32 && !SPLIT) if (plain) {
            // Straight-line code, no per-lane predicates or address arithmetic (with one wavefront per
            // SIMD every branch and every dependent wait is exposed): the stores go through a buffer
            // descriptor over the wavefront's part of C, whose range ends with the last valid row, so
            // rows past the matrix are dropped by the range check; a lane whose columns lie past the
            // matrix gets an offset beyond every range. Lane l of round u holds 16 bytes of row
            // 4u + l/16 (256-byte rows): the row advance is a scalar offset.
            T* part = static_cast<T*>(c_base) + static_cast<long>(row0) * c_ld + (c_col0 + col0);
            const int rows_left = min(WM, p.m - row0), cols_left = min(WN, c_cols - (c_col0 + col0));
            const long extent = rows_left > 0 && cols_left > 0
                                    ? (static_cast<long>(rows_left - 1) * c_ld + cols_left) * static_cast<long>(sizeof(T))
                                    : 0;
            const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(part, 0, static_cast<int>(extent), 0x00020000);
            constexpr int kLanesPerRow = kRowBytes / 16, kRowsPerRound = kWave / kLanesPerRow, kRounds = 32 / kRowsPerRound;
            const int lane_row = lane / kLanesPerRow, lane_chunk = lane % kLanesPerRow;
            const int row_bytes = static_cast<int>(c_ld * static_cast<long>(sizeof(T)));
            const int voffset = lane_chunk * 8 < cols_left ? lane_row * row_bytes + lane_chunk * 16 : std::numeric_limits<int>::min();
#pragma unroll
            for (int r = 0; r < kRowBlocks; ++r) {
                // Accumulators leave their registers block by block: read ahead of their block they
                // would not fit the vector registers.
                __builtin_amdgcn_sched_barrier(0);
                if (request) request_share(r);
                stage.template operator()<T, TN>(r, 0);
                u32x4 data[kRounds];
#pragma unroll
                for (int u = 0; u < kRounds; ++u) {
                    const int row = u * kRowsPerRound + lane_row;
                    data[u] = *reinterpret_cast<const u32x4*>(region + row * kRowBytes + ((lane_chunk ^ sw(row)) * 16));
                }
#pragma unroll
                for (int u = 0; u < kRounds; ++u)
                    store_chunk(data[u], rsrc, voffset, (r * 32 + u * kRowsPerRound) * row_bytes);
            }
            return;
        }
        if constexpr (SPLIT || kIsF32) if (SPLIT || plain) {
            // n rounded up to whole 16-byte chunks of 16-bit storage; plain fp32 results: C itself.
            const int pitch = static_cast<int>(SPLIT ? p.ld_partial : p.ldc), columns = SPLIT ? pitch : p.n;
            const float* origin = static_cast<const float*>(p.c) +
                                  (static_cast<long>(w.slice) * p.m + row0) * pitch + (w.n0 + col0);
            const int cols_left = min(WN, columns - (w.n0 + col0));
            const __amdgpu_buffer_rsrc_t rsrc = part_rsrc(origin, pitch, 4, rows_left, cols_left);
            const int row_bytes = pitch * 4;
#pragma unroll
            for (int r = 0; r < kRowBlocks; ++r) {
                __builtin_amdgcn_sched_barrier(0);
                if (request) request_share(r);
#pragma unroll
                for (int half = 0; half < 2; ++half) {
                    stage.template operator()<float, TN / 2>(r, half * (TN / 2));
                    const int col = half * (WN / 2) + l_col;
                    constexpr int kSecond = kGroups * 4;  // columns between a lane's two quads
                    const int voffset0 = col < cols_left ? f_row * row_bytes + col * 4 : std::numeric_limits<int>::min();
                    const int voffset1 = col + kSecond < cols_left ? f_row * row_bytes + (col + kSecond) * 4 : std::numeric_limits<int>::min();
                    vec_t<float, 4> v0[kRoundsF], v1[kRoundsF];
#pragma unroll
                    for (int u = 0; u < kRoundsF; ++u) read_staged_lines(u, v0[u], v1[u]);
#pragma unroll
                    for (int u = 0; u < kRoundsF; ++u) {
                        const int soffset = (r * 32 + u * kRowsF) * row_bytes;
                        store_chunk(__builtin_bit_cast(u32x4, v0[u]), rsrc, voffset0, soffset);
                        store_chunk(__builtin_bit_cast(u32x4, v1[u]), rsrc, voffset1, soffset);
                    }
                }
            }
            return;
        }
        if (p.ragged) {
            // Rows of C that do not start on 16-byte boundaries: lanes along the columns of a staged half, one element
            // each, so that a store instruction still covers one contiguous piece of a row (or of a few).
            constexpr int kCols = WN / 2, kRowsE = kWave / kCols;
            const int e_row = lane / kCols, e_col = lane % kCols;
#pragma unroll
            for (int r = 0; r < kRowBlocks; ++r) {
                __builtin_amdgcn_sched_barrier(0);
                if (request) request_share(r);
#pragma unroll
                for (int half = 0; half < 2; ++half) {
                    stage.template operator()<float, TN / 2>(r, half * (TN / 2));
                    const int col = half * kCols + e_col, n = w.n0 + col0 + col, c_col = c_col0 + col0 + col;
                    const float bias = p.bias != nullptr && c_col < c_cols ? to_f32(static_cast<const T*>(p.bias)[n]) : 0.0f;
#pragma unroll 4
                    for (int u = 0; u < 32 / kRowsE; ++u) {
                        const int row = u * kRowsE + e_row;
                        float v = *reinterpret_cast<const float*>(region + row * kRowBytes + (((e_col / 4) ^ sw(row)) * 16) + (e_col % 4) * 4);
                        const long m = row0 + r * 32 + row;
                        if (m >= p.m || c_col >= c_cols) continue;
                        if (p.addend != nullptr) v += p.addend[m * p.ld_addend + n];
                        v += bias;
                        if (p.residual != nullptr) v += to_f32(static_cast<const T*>(p.residual)[m * p.ldr + n]);
                        if (p.c_f32) {
                            float* out = static_cast<float*>(c_base) + m * c_ld + c_col;
                            *out = p.accumulate ? v + *out : v;
                        } else {
                            T* out = static_cast<T*>(c_base) + m * c_ld + c_col;
                            *out = from_f32<T>(p.accumulate ? v + to_f32(*out) : v);
                        }
                    }
                }
            }
            return;
        }
#pragma unroll
        for (int r = 0; r < kRowBlocks; ++r) {
            __builtin_amdgcn_sched_barrier(0);
            if (request) request_share(r);
#pragma unroll
            for (int half = 0; half < 2; ++half) {
                pass.template operator()<float, TN / 2>(r, half * (TN / 2), [&](int, int row, int col, const unsigned char* lo,
                                                                              const unsigned char* hi) {
                    const int m = row0 + row, n = w.n0 + col0 + col, c_col = c_col0 + col0 + col;
                    vec_t<float, 4> v0 = *reinterpret_cast<const vec_t<float, 4>*>(lo);
                    vec_t<float, 4> v1 = *reinterpret_cast<const vec_t<float, 4>*>(hi);
                    if (m >= p.m || c_col >= c_cols) return;
                    {
                        if (p.addend != nullptr) {
                            const float* addend = p.addend + static_cast<long>(m) * p.ld_addend + n;
                            v0 += *reinterpret_cast<const vec_t<float, 4>*>(addend);
                            v1 += *reinterpret_cast<const vec_t<float, 4>*>(addend + 4);
                        }
                        if (p.bias != nullptr) {
                            const T* bias = static_cast<const T*>(p.bias) + n;
                            v0 += vec_to_f32<T, 4>(load_vec<T, 4>(bias));
                            v1 += vec_to_f32<T, 4>(load_vec<T, 4>(bias + 4));
                        }
                        if (p.residual != nullptr) {
                            const T* residual = static_cast<const T*>(p.residual) + static_cast<long>(m) * p.ldr + n;
                            v0 += vec_to_f32<T, 4>(load_vec<T, 4>(residual));
                            v1 += vec_to_f32<T, 4>(load_vec<T, 4>(residual + 4));
                        }
                        if (p.c_f32) {
                            float* out = static_cast<float*>(c_base) + static_cast<long>(m) * c_ld + c_col;
                            if (p.accumulate) {
                                v0 += *reinterpret_cast<const vec_t<float, 4>*>(out);
                                v1 += *reinterpret_cast<const vec_t<float, 4>*>(out + 4);
                            }
                            *reinterpret_cast<vec_t<float, 4>*>(out) = v0;
                            *reinterpret_cast<vec_t<float, 4>*>(out + 4) = v1;
                        } else {
                            T* out = static_cast<T*>(c_base) + static_cast<long>(m) * c_ld + c_col;
                            if (p.accumulate) {
                                v0 += vec_to_f32<T, 4>(load_vec<T, 4>(out));
                                v1 += vec_to_f32<T, 4>(load_vec<T, 4>(out + 4));
                            }
                            const vec_t<T, 4> r0 = vec_from_f32<T, 4>(v0), r1 = vec_from_f32<T, 4>(v1);
                            if constexpr (kIsF32) {  // 16-byte accesses
                                store_vec<T, 4>(out, r0);
                                store_vec<T, 4>(out + 4, r1);
                            } else {
                                vec_t<T, 8> packed;
#pragma unroll
                                for (int e = 0; e < 4; ++e) {
                                    packed[e] = r0[e];
                                    packed[4 + e] = r1[e];
                                }
                                store_vec<T, 8>(out, packed);
                            }
                        }
                    }
                });
            }
        }
    };

    // Software pipeline over the K tiles t of an item, two K steps of TM x TN MFMAs each. The fragments of a step are read
    // from LDS while the step before it is multiplied, into registers of their own:
    //   first step   MFMAs ‖ LDS reads of this tile's second-step fragments ‖ the loads of A's K tile t+kAhead (into the slot
    //                of B's K tile t-1)
    //   wait         this wavefront's loads of K tile t+1 have landed and its reads of K tile t are through; barrier:
    //                everybody's have, so K tile t's slots are free
    //   second step  MFMAs ‖ LDS reads of K tile t+1's first-step fragments ‖ the loads of B's K tile t+kAhead (into the slot
    //                of A's K tile t)
    // so LDS latency and one to one and a half K tiles of global latency sit in the shadow of MFMAs, and the workgroup
    // meets once per K tile. With one wavefront per SIMD nothing else hides an instruction that is not next to an MFMA, so
    // every MFMA is followed by its share of the loads and fragment reads and a scheduling fence keeps them there. A
    // wavefront's load instruction keeps it from issuing for about as long as an MFMA runs.
    constexpr int kMfmas = TM * TN;
    constexpr int kReadEvery = kMfmas / kFrags >= 4 ? 3 : 1;  // MFMAs between fragment reads
    static_assert(kReadEvery * kFrags <= kMfmas && kLoads <= kMfmas, "a step has room for the reads and loads it carries");
    // STEP 0: a_tile, b_tile are K tile t's; STEP 1: K tile t+1's. slot_lds: where the step's loads (of K tile `aimed`) go.
    auto multiply_step = [&]<int STEP, bool FIRST>(const T* a_tile, const T* b_tile, unsigned int slot_lds, int aimed) __attribute__((always_inline)) {
        static_for<0, kMfmas>([&](auto index) {
            constexpr int m = decltype(index)::value;
            // Rows one after the other, their columns left to right and right to left alternately:
            // consecutive MFMAs always share an operand (measurably less power on a power-limited chip).
            constexpr int i = m / TN, jj = m % TN, j = (i & 1) ? TN - 1 - jj : jj;
            if constexpr (FIRST && STEP == 0) Mfma<T>::start(acc[i][j], bf[STEP][j], af[STEP][i]);
            else Mfma<T>::run(acc[i][j], bf[STEP][j], af[STEP][i]);
            if constexpr (m % kReadEvery == 0 && m / kReadEvery < kFrags)
                read_frag.template operator()<1 - STEP, m / kReadEvery>(a_tile, b_tile);
            static_for<(m * kLoads) / kMfmas, ((m + 1) * kLoads) / kMfmas>([&](auto l) {
                if constexpr (STEP == 0) issue_a(l, slot_lds, ca);
                else issue_b(l, slot_lds, cb);
            });
            // The next step's cursor, where its scalar arithmetic has MFMAs around it.
            if constexpr (m == kMfmas / 2) {
                if constexpr (STEP == 0) aim_b(aimed, cb);
                else aim_a(aimed + 1, ca);
            }
            __builtin_amdgcn_sched_barrier(0);
        });
    };
    auto slot_after = [](int slot, int by) __attribute__((always_inline)) { return slot + by >= kSlots ? slot + by - kSlots : slot + by; };

    // Per round: multiply an item, request the first K tiles of the next one, store the finished
    // tile (its stores drain under the MFMAs that follow). The sources are opened every round, also
    // when no item is left (then for the last one again, unused): values that are set on every path
    // stay in scalar registers.
    Item current = locate(item);
    open(current);
    request_tiles.template operator()<0, kSlots - 1>();
    while (true) {
        const int steps = current.kt_end - current.kt_begin;
        // Loads and stores retire in the order they were issued: at most the loads of the operand tiles
        // after the first two (and no older store of the previous epilogue) may still be outstanding.
        __builtin_amdgcn_s_waitcnt(vmcnt_immediate((kSlots - 3) * kLoads));
        barrier_only();
        static_for<0, kFrags>([&](auto f) { read_frag.template operator()<0, decltype(f)::value>(smem, smem + kSlot); });
        aim_a(kAhead, ca);
        int slot = 0;  // of A's K tile t; B's is in the one after it
        auto first_step = [&]<bool FIRST>(int t) __attribute__((always_inline)) {
            multiply_step.template operator()<0, FIRST>(smem + slot * kSlot, smem + slot_after(slot, 1) * kSlot,
                                                        lds_wave + slot_after(slot, kSlots - 1) * kSlotBytes, t + kAhead);
        };
        auto second_step = [&](int t) __attribute__((always_inline)) {
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            __builtin_amdgcn_s_waitcnt(vmcnt_immediate((kSlots - 4) * kLoads));
            barrier_only();
            const int next = slot_after(slot, 2);
            multiply_step.template operator()<1, false>(smem + next * kSlot, smem + slot_after(slot, 3) * kSlot,
                                                        lds_wave + slot * kSlotBytes, t + kAhead);
            slot = next;
        };
        // The first K step starts the sums (MFMA with a zero addend): no pass over the 256
        // accumulator registers to clear them. Every item has at least one K step (the host makes
        // K slices non-empty).
        first_step.template operator()<true>(0);
        if (steps > 1) {
            second_step(0);
            int t = 1;
            for (; t * kSteps + 1 < steps; ++t) {
                first_step.template operator()<false>(t);
                second_step(t);
            }
            if (t * kSteps < steps) first_step.template operator()<false>(t);
        }
        // The loads still outstanding are of K tiles past the end (zeros, but they do write LDS):
        // once they have landed and every wavefront has read its last fragments, all slots are free.
        __builtin_amdgcn_s_waitcnt(vmcnt_immediate(0));
        barrier_only();
        item += item_stride;
        const bool more = item < item_end;
        const Item next = locate(more ? item : item_end - 1);
        open(next);
        store_tile(current, more);
        if (!more) break;
        current = next;
    }
}

// C = Σ_slices partial (+ C) (+ bias), four columns per thread, slices in order. n: the partial rows' length, a
// multiple of 4; columns past n_valid (rows of C that are not whole 16-byte chunks) are not stored.
template <typename T>
__global__ __launch_bounds__(kThreads) void splitk_reduce_kernel(void* __restrict__ c,
                                                                const float* __restrict__ partial,
                                                                const T* __restrict__ bias, int m, int n, int n_valid,
                                                                long ldc, int slices, int accumulate, int c_f32,
                                                                int ragged) {
    const long quads = static_cast<long>(m) * (n / 4);
    const long stride = static_cast<long>(m) * n;
    for (long q = static_cast<long>(blockIdx.x) * kThreads + threadIdx.x; q < quads;
         q += static_cast<long>(gridDim.x) * kThreads) {
        const long row = q / (n / 4);
        const int col = static_cast<int>(q - row * (n / 4)) * 4;
        const float* source = partial + row * n + col;
        // Four slices are requested at a time; the additions keep the slices' order.
        vec_t<float, 4> v = *reinterpret_cast<const vec_t<float, 4>*>(source);
        int s = 1;
        for (; s + 4 <= slices; s += 4) {
            vec_t<float, 4> part[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) part[u] = *reinterpret_cast<const vec_t<float, 4>*>(source + (s + u) * stride);
#pragma unroll
            for (int u = 0; u < 4; ++u) v += part[u];
        }
        for (; s < slices; ++s) v += *reinterpret_cast<const vec_t<float, 4>*>(source + s * stride);
        if (ragged) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                if (col + e >= n_valid) continue;
                float x = v[e];
                if (bias != nullptr) x += to_f32(bias[col + e]);
                if (c_f32) {
                    float* out = static_cast<float*>(c) + row * ldc + col + e;
                    *out = accumulate ? x + *out : x;
                } else {
                    T* out = static_cast<T*>(c) + row * ldc + col + e;
                    *out = from_f32<T>(accumulate ? x + to_f32(*out) : x);
                }
            }
            continue;
        }
        if (bias != nullptr) v += vec_to_f32<T, 4>(load_vec<T, 4>(bias + col));
        if (c_f32) {
            float* out = static_cast<float*>(c) + row * ldc + col;
            if (accumulate) v += *reinterpret_cast<const vec_t<float, 4>*>(out);
            *reinterpret_cast<vec_t<float, 4>*>(out) = v;
        } else {
            T* out = static_cast<T*>(c) + row * ldc + col;
            if (accumulate) v += vec_to_f32<T, 4>(load_vec<T, 4>(out));
            store_vec<T, 4>(out, vec_from_f32<T, 4>(v));
        }
    }
}

// Copies a [rows, cols] matrix to rows of `pitch` elements (whole 16-byte chunks), zeros past cols: the streamed kernels
// read whole chunks. One chunk per thread; the source may start anywhere.
template <typename E>
__global__ __launch_bounds__(kThreads) void pad_rows_kernel(E* __restrict__ dst, const E* __restrict__ src, long rows, int cols,
                                                            long ld, int pitch) {
    constexpr int VEC = kVec128<E>;
    const int chunks = pitch / VEC;
    const long total = rows * chunks;
    for (long q = static_cast<long>(blockIdx.x) * kThreads + threadIdx.x; q < total; q += static_cast<long>(gridDim.x) * kThreads) {
        const long row = q / chunks;
        const int col = static_cast<int>(q - row * chunks) * VEC;
        const E* from = src + row * ld + col;
        vec_t<E, VEC> v;
        if (col + VEC <= cols) {
            __builtin_memcpy(&v, from, 16);
        } else {
#pragma unroll
            for (int e = 0; e < VEC; ++e) v[e] = col + e < cols ? from[e] : E{0};
        }
        store_vec<E, VEC>(dst + row * pitch + col, v);
    }
}

// ---- fp32 matrix-core kernel for everything the streamed path does not take ----------------------
// Operands that 32-bit byte offsets do not reach, and unaligned ones that cannot be copied to padded rows because the
// caller owns the arena. Any shape, any alignment, all three operand layouts: a 128 x 128 tile of C per block, K in
// steps of 16; the four wavefronts own 64 x 64 each and multiply with v_mfma_f32_32x32x2_f32 on fp32 operands
// (16-bit storage is widened on the way into LDS, so the products are exact and the sums fp32, as in the streamed
// kernels). Operand tiles go through registers into a K-major LDS layout ([k][m], [k][n]) — the fragment of an
// MFMA step is then 32 consecutive floats per half-wavefront — with the next tile's loads in flight during the
// multiplication; rows, columns and K positions past the matrices read as zeros.
constexpr int kF32Tile = 128;  // rows and columns of C per block
constexpr int kF32K = 16;      // K per LDS stage
constexpr int kF32Pad = 4;
using acc16_t = vec_t<float, 16>;

template <typename T>
__global__ __launch_bounds__(kThreads) void gemm_f32_mfma_kernel(KernelArgs p, int a_k, int b_k) {
    __shared__ float as[2][kF32K][kF32Tile + kF32Pad];
    __shared__ float bs[2][kF32K][kF32Tile + kF32Pad];
    const T* A = static_cast<const T*>(p.a);
    const T* B = static_cast<const T*>(p.b);
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    const int wm = wave >> 1, wn = wave & 1;
    const long m0 = static_cast<long>(blockIdx.y) * kF32Tile, n0 = static_cast<long>(blockIdx.x) * kF32Tile;
    constexpr int kPerThread = kF32Tile * kF32K / kThreads;  // elements of each operand tile a thread moves
    float a_regs[kPerThread], b_regs[kPerThread];
    // Element e of a thread's share: consecutive threads walk the operand's contiguous index.
    auto coordinates = [&](int e, bool k_contiguous, int& row, int& k) {
        const int index = threadIdx.x + e * kThreads;
        if (k_contiguous) {
            row = index / kF32K;
            k = index % kF32K;
        } else {
            k = index / kF32Tile;
            row = index % kF32Tile;
        }
    };
    auto fetch = [&](long k0) {
#pragma unroll
        for (int e = 0; e < kPerThread; ++e) {
            int row, k;
            coordinates(e, a_k != 0, row, k);
            const long m = m0 + row, ka = k0 + k;
            a_regs[e] = (m < p.m && ka < p.k) ? to_f32(a_k ? A[m * p.lda + ka] : A[ka * p.lda + m]) : 0.0f;
            coordinates(e, b_k != 0, row, k);
            const long n = n0 + row, kb = k0 + k;
            b_regs[e] = (n < p.n && n < p.b_extent && kb < p.b_k) ? to_f32(b_k ? B[n * p.ldb + kb] : B[kb * p.ldb + n]) : 0.0f;
        }
    };
    auto deposit = [&](int stage) {
#pragma unroll
        for (int e = 0; e < kPerThread; ++e) {
            int row, k;
            coordinates(e, a_k != 0, row, k);
            as[stage][k][row] = a_regs[e];
            coordinates(e, b_k != 0, row, k);
            bs[stage][k][row] = b_regs[e];
        }
    };
    acc16_t acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = acc16_t(0.0f);
    fetch(0);
    deposit(0);
    __syncthreads();
    int stage = 0;
    for (long k0 = 0; k0 < p.k; k0 += kF32K) {
        const bool more = k0 + kF32K < p.k;
        if (more) fetch(k0 + kF32K);  // in flight during the multiplication below
#pragma unroll
        for (int kk = 0; kk < kF32K; kk += 2) {
            // MFMA step of k = 2: lane l holds row (column) l % 32 at k = l / 32.
            float a[2], b[2];
#pragma unroll
            for (int i = 0; i < 2; ++i) a[i] = as[stage][kk + (lane >> 5)][wm * 64 + i * 32 + (lane & 31)];
#pragma unroll
            for (int j = 0; j < 2; ++j) b[j] = bs[stage][kk + (lane >> 5)][wn * 64 + j * 32 + (lane & 31)];
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i], b[j], acc[i][j], 0, 0, 0);
        }
        if (more) {
            deposit(stage ^ 1);  // nobody reads that stage: the barrier below closed its last use
            __syncthreads();
            stage ^= 1;
        }
    }
    // Register r of a block holds row 8 (r / 4) + 4 (lane / 32) + r % 4 of column lane % 32.
#pragma unroll
    for (int i = 0; i < 2; ++i) {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const long n = n0 + wn * 64 + j * 32 + (lane & 31);
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const long m = m0 + wm * 64 + i * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
                if (m >= p.m || n >= p.n) continue;
                float v = acc[i][j][r];
                if (p.addend != nullptr) v += p.addend[m * p.ld_addend + n];
                if (p.bias != nullptr) v += to_f32(static_cast<const T*>(p.bias)[n]);
                if (p.residual != nullptr) v += to_f32(static_cast<const T*>(p.residual)[m * p.ldr + n]);
                if (p.c_f32) {
                    float* out = static_cast<float*>(p.c) + m * p.ldc + n;
                    *out = p.accumulate ? v + *out : v;
                } else {
                    T* out = static_cast<T*>(p.c) + m * p.ldc + n;
                    *out = from_f32<T>(p.accumulate ? v + to_f32(*out) : v);
                }
            }
        }
    }
}

// ------------------------------------------------------------------- host side
constexpr int blocks_per_unit(int tile) { return tile == 256 ? 1 : 2; }  // resident blocks per CU: what the LDS stages allow


template <typename T, int BM, int BN, bool A_K, bool B_K, bool SPLIT, bool SEGMENTED, bool RESIDUAL = false,
          bool SWIGLU = false, bool GRAD = false, int SLOTS = kLdsSlots>
int launch_mfma(const KernelArgs& p, int slices, hipStream_t stream) {
    const long items = static_cast<long>(p.tiles_m) * p.tiles_n * slices;
    if constexpr (BM == 128 && SLOTS == kLdsSlots) {
        if (items <= compute_units())
            return launch_mfma<T, BM, BN, A_K, B_K, SPLIT, SEGMENTED, RESIDUAL, SWIGLU, GRAD, kDeepSlots>(p, slices, stream);
    }
    constexpr std::size_t smem = TileLayout<T, BM, BN, A_K, B_K, SLOTS>::kSmemBytes;
    auto kernel = gemm_mfma_kernel<T, BM, BN, A_K, B_K, SPLIT, SEGMENTED, RESIDUAL, SWIGLU, GRAD, SLOTS>;
    static bool configured = false;
    if (!configured) {
        CGPTX_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                      hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(smem)));
        configured = true;
    }
    // One block per CU slot (256x256 tiles: one per CU; 128x128: two), a multiple of the XCD count
    // so that every XCD gets the same number of blocks; fewer when there are fewer work items.
    KernelArgs args = p;
    args.slices = slices;
    {
        // x * ceil(2^32 / d) >> 32 == x / d for every x with x * d < 2^32.
        // Tile-rows per L2 locality group. 8 (x 4 tile-columns = the 32 tiles in flight on an XCD) shares operand
        // panels best. The SwiGLU-gradient epilogue moves four times the bytes of a plain one, two loads and two
        // stores of whole [gate | up] rows: there the tiles in flight on an XCD are better spread along the rows
        // (2 tile-rows x all 8 tile-columns of the training shape: 250 -> 212 us per launch; 1, 2 and 4 tile-rows
        // measure the same, every other kernel is at its best with 8).
        args.group_rows_log2 = GRAD ? 1 : 3;
        const unsigned long divisor = (1ul << args.group_rows_log2) * static_cast<unsigned long>(p.tiles_n);
        const unsigned long tiles = static_cast<unsigned long>(p.tiles_m) * static_cast<unsigned long>(p.tiles_n);
        const bool exact = divisor > 1 && tiles * divisor < (1ul << 32);
        args.group_reciprocal = exact ? static_cast<unsigned int>(((1ul << 32) + divisor - 1) / divisor) : 0u;
    }
    const long slots = static_cast<long>(compute_units()) * blocks_per_unit(BM) / kXcds * kXcds;
    const long blocks = std::min<long>((items + kXcds - 1) / kXcds * kXcds, std::max<long>(slots, kXcds));
    hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned int>(blocks)), dim3(kThreads), smem, stream, args);
    CGPTX_LAUNCH_CHECK();
    return CGPTX_OK;
}

template <typename T, int BM, int BN, bool SPLIT>
int launch_layout(const KernelArgs& p, bool a_k, bool b_k, int slices, hipStream_t stream) {
    // A given in segments along K has kernels of its own (the source of a K tile is then picked
    // per tile), and only unsplit ones.
    const bool segmented = a_k && p.a_seg.count > 0;
    if constexpr (!SPLIT && !std::is_same_v<T, float>) {
        if (segmented && b_k) return launch_mfma<T, BM, BN, true, true, false, true>(p, slices, stream);
        if (segmented && !b_k) return launch_mfma<T, BM, BN, true, false, false, true>(p, slices, stream);
    }
    if (segmented) return fail(CGPTX_RUNTIME, "gemm: a segmented operand cannot be split along K");
    if constexpr (!SPLIT && BN == 256) {
        if (p.act != nullptr) return launch_mfma<T, BM, BN, true, true, false, false, false, true>(p, slices, stream);
    }
    if (p.act != nullptr) return fail(CGPTX_RUNTIME, "gemm: the SwiGLU epilogue needs 256-wide unsplit tiles");
    if constexpr (!SPLIT && BN == 256) {
        if (p.saved != nullptr) return launch_mfma<T, BM, BN, true, false, false, false, false, false, true>(p, slices, stream);
    }
    if (p.saved != nullptr) return fail(CGPTX_RUNTIME, "gemm: the SwiGLU gradient epilogue needs 256-wide unsplit tiles");
    if constexpr (!SPLIT && !std::is_same_v<T, float>) {
        if (a_k && b_k && p.bias == nullptr && p.addend == nullptr && !p.c_f32 && !p.ragged) {
            if (p.residual != nullptr && !p.accumulate) return launch_mfma<T, BM, BN, true, true, false, false, true>(p, slices, stream);
            if (p.residual == nullptr && p.accumulate && p.c_seg.count == 0) {
                // C += A·B in the storage dtype is the same epilogue with C as its own residual
                // (every lane reads the elements it later writes, and reads them first).
                KernelArgs self = p;
                self.residual = p.c;
                self.ldr = p.ldc;
                self.accumulate = 0;
                return launch_mfma<T, BM, BN, true, true, false, false, true>(self, slices, stream);
            }
        }
    }
    if (a_k && b_k) return launch_mfma<T, BM, BN, true, true, SPLIT, false>(p, slices, stream);
    if (a_k && !b_k) return launch_mfma<T, BM, BN, true, false, SPLIT, false>(p, slices, stream);
    if (!a_k && !b_k) return launch_mfma<T, BM, BN, false, false, SPLIT, false>(p, slices, stream);
    return fail(CGPTX_RUNTIME, "gemm: unsupported operand layout");
}

// CGPTX_GEMM_TILE=32|64|128|256 pins the tile size (for experiments); anything else = automatic.
int forced_tile() {
    static const int value = [] {
        const char* text = std::getenv("CGPTX_GEMM_TILE");
        if (text == nullptr) return 0;
        const int v = std::atoi(text);
        return (v == 32 || v == 64 || v == 128 || v == 256) ? v : 0;
    }();
    return value;
}

std::size_t round_up(std::size_t v, std::size_t unit) { return (v + unit - 1) / unit * unit; }

// How a call of the streamed kernels is cut: tile edge, K slices per tile and K tiles per slice.
struct Plan {
    int tile = 256;
    int slices = 1;
    int k_tiles_per_slice = 1;
    bool deep = false;  // small tiles: all of a CU's LDS for one workgroup's stages
    std::size_t partial_bytes(const GemmArgs& g) const {
        return slices > 1 ? static_cast<std::size_t>(slices) * g.m * round_up(g.n, 8) * sizeof(float) : 0;
    }
};

// Predicted time of a call in microseconds, from launches measured on random bf16 data inside a graph (operands rotated
// through 64 MB; K tiles of 64 bytes): what a kernel costs before its K loop, plus the K loop of the busiest CU.
//   256: one block per CU, 8.5 us for filling its pipeline and storing its tile, 0.55 per K tile on an idle chip, 0.69 at
//        the power limit of a full one
//   128: two blocks per CU share its matrix cores: 0.29 per K tile and block
//    64: 0.128 per K tile and block, 0.14 where few blocks run, whose first 16 K tiles come in one latency
//    32: 0.07 - 0.1 per K tile (k-contiguous operands stream best), up to one block per CU
// A split along K adds a launch and the partial tiles' way to memory and back. fp32 K tiles hold 16 positions and take about
// as long as the fp32 matrix rate asks (0.93 per K tile of 128 x 128), smaller tiles somewhat longer for their share.
// [M, N] x K: 128 x 768 x 768 32/1 4.8, 64/1 5.1, 128/1 9.7; 1024 x 1024 x 1024 64/1 7.8, 128/1 12.7, 256/1 26; 4096 x 1024 x
// 1024 128/1 14.5, 64/1 19, 256/1 27; 16384 x 1024 x 1024 256/1 34, 128/1 42; 768 x 768 x 8192 128/6 22, 64/3 27 - 30, 256/16
// 30; 2048 x 768 x 50272 256/8 145 - 179, 128/8 184 - 255, 64/2 284 - 371; 16384 x 768 x 32000 256/1 688, 128/1 976; fp32
// 256 x 1024 x 1024 32/1 10, 64/4 15, 128/8 20; 256 x 32000 x 1024 128/1 123, 64/1 149 (tile / slices).
double predicted_us(int tile, long tiles, long slices, long k_tiles, double partial_mb, bool f32, bool a_k, bool b_k, long units) {
    const double kt = static_cast<double>((k_tiles + slices - 1) / slices);
    const double load = static_cast<double>(tiles * slices) / static_cast<double>(units);
    const double blocks = std::ceil(load);
    double time = 0.0;
    if (f32) {
        const double per_tile = tile == 32 ? 0.088 : tile == 64 ? 0.265 : 0.93;
        time = (tile == 32 ? 3.0 : tile == 64 ? 4.0 : 5.0) + kt * per_tile * (tile == 32 ? std::max(1.0, load) : blocks);
    } else if (tile == 256) {
        time = blocks * (8.5 + kt * (0.55 + 0.14 * load / blocks));
    } else if (tile == 128) {
        time = 5.0 + kt * (load < 0.5 ? 0.23 : 0.29 * blocks) + 2.0 * std::max(0.0, std::ceil(blocks / 2.0) - 1.0);
    } else if (tile == 64) {
        time = load <= 1.0 ? 3.8 + 0.02 * std::min(kt, 16.0) + std::max(0.0, kt - 16.0) * (!a_k && load < 0.6 ? 0.095 : 0.135)
                           : 3.8 + kt * 0.128 * blocks * (blocks > 4.0 ? 1.3 : 1.0);
    } else {
        time = 3.0 + kt * (!a_k ? 0.1 : b_k ? 0.07 : 0.085) * std::max(1.0, 0.92 * load);
    }
    return slices > 1 ? time + 3.0 + 0.45 * partial_mb + 0.3 * std::min(partial_mb, 8.0) : time;
}

Plan make_plan(const GemmArgs& g) {
    Plan plan;
    const long units = compute_units();
    const bool f32 = g.dtype == CGPTX_F32;
    const long k_step = f32 ? kBK<float> : kBK<bf16_t>;
    const long k_tiles = (static_cast<long>(g.k) + k_step - 1) / k_step;
    auto tiles_of = [&](long edge) {
        return static_cast<long>((g.m + edge - 1) / edge) * static_cast<long>((g.n + edge - 1) / edge);
    };
    const bool may_split = (!g.no_split || g.split_workspace != nullptr) && g.residual == nullptr && g.addend_f32 == nullptr &&
                           g.swiglu_out == nullptr && g.swiglu_saved == nullptr && g.c_segments.count == 0 &&
                           !(g.a_k_contiguous && g.a_segments.count > 0);
    auto set_slices = [&](long slices) {
        plan.k_tiles_per_slice = static_cast<int>((k_tiles + slices - 1) / slices);
        if (slices > 1) plan.k_tiles_per_slice = (plan.k_tiles_per_slice + kSteps - 1) / kSteps * kSteps;  // whole K tiles of the large kernels
        plan.slices = static_cast<int>((k_tiles + plan.k_tiles_per_slice - 1) / plan.k_tiles_per_slice);
    };
    if (g.swiglu_out != nullptr || g.swiglu_saved != nullptr || (!f32 && tiles_of(256) >= 3 * units && g.batch_rows == 0)) {
        set_slices(1);
        return plan;
    }
    if (g.batch_rows != 0) {
        // A stack of products brings any number of tiles: the slice count that needs the least time, counted in
        // rounds of the persistent blocks times the length of a slice (fewer slices on a tie: fewer partial tiles).
        long slices = 1;
        double best = 0.0;
        for (long s = 1; s <= 8 && may_split && k_tiles >= 32 && k_tiles / s >= 16; ++s) {
            const long rounds = (tiles_of(256) * s + units - 1) / units;
            const double time = static_cast<double>(rounds) / static_cast<double>(s) * (s > 1 ? 1.02 : 1.0);
            if (s == 1 || time < best * 0.999) {
                best = time;
                slices = s;
            }
        }
        set_slices(slices);
        return plan;
    }
    const int forced = forced_tile();
    const double slice_bytes = static_cast<double>(g.m) * static_cast<double>(round_up(g.n, 8)) * sizeof(float);
    // Calls that 256 x 256 tiles spread over three quarters of the chip keep the order of additions of the kernels with a
    // SwiGLU epilogue, which take such calls only (one sum over all of K): the fused and the separate operators give the same
    // bits. A split would fill the last quarter, less the partial tiles' way: 16384 x 768 x 32000 688 us, in four slices 650.
    const bool whole_k = !f32 && tiles_of(256) * 4 >= units * 3;
    double best = -1.0;
    long best_slices = 1;
    for (int tile : {32, 64, 128, 256}) {
        if ((whole_k && tile < 128) || (forced != 0 && tile != forced && !(f32 && forced == 256)) || (f32 && tile == 256)) continue;
        const long tiles = tiles_of(tile);
        if (forced == 0 && tile <= 64 && tiles > 16 * units) continue;
        for (long s = 1; s <= 16; ++s) {
            if (s > 1 && (whole_k || !may_split || k_tiles / s < 8 || tiles * s > 4 * units ||
                          (g.no_split && slice_bytes * static_cast<double>(s) > static_cast<double>(g.split_workspace_bytes))))
                break;
            const double time = predicted_us(tile, tiles, s, k_tiles, slice_bytes * static_cast<double>(s) * 1e-6, f32,
                                             g.a_k_contiguous, g.b_k_contiguous, units);
            if (best < 0.0 || time < best) {
                best = time;
                plan.tile = tile;
                best_slices = s;
            }
        }
    }
    set_slices(best_slices);
    plan.deep = tiles_of(plan.tile) * plan.slices <= units;
    return plan;
}

// Arguments of the small kernel (gemm_small_kernel.hpp) from the streamed ones.
SmallArgs small_args(const KernelArgs& p, bool split, int k_tiles_per_slice) {
    SmallArgs a{};
    a.a = p.a;
    a.b = p.b;
    a.c = p.c;
    a.lda = p.lda;
    a.ldb = p.ldb;
    a.ldc = split ? p.ld_partial : p.ldc;
    a.m = p.m;
    a.n = p.n;
    a.k = p.k;
    a.a_extent = p.a_extent;
    a.b_extent = p.b_extent;
    a.b_k = p.b_k;
    a.k_tiles = p.k_tiles;
    a.k_tiles_per_slice = k_tiles_per_slice;
    a.bias = p.bias;
    a.residual = p.residual;
    a.addend = p.addend;
    a.ldr = p.ldr;
    a.ld_addend = p.ld_addend;
    a.accumulate = p.accumulate;
    a.c_f32 = p.c_f32;
    a.ragged = p.ragged;
    auto copy = [](const KernelSegments& in, SmallSegments& out) {
        for (int i = 0; i < 3; ++i) {
            out.ptr[i] = in.ptr[i];
            out.ld[i] = in.ld[i];
            out.cols[i] = in.cols[i];
        }
        out.count = in.count;
    };
    copy(p.a_seg, a.a_seg);
    copy(p.c_seg, a.c_seg);
    return a;
}

template <typename T>
int launch_small_call(const GemmArgs& g, const KernelArgs& p, const Plan& plan, bool split, hipStream_t stream) {
    SmallCall call{};
    call.args = small_args(p, split, plan.k_tiles_per_slice);
    call.a_k_contiguous = g.a_k_contiguous;
    call.b_k_contiguous = g.b_k_contiguous;
    call.tile = plan.tile;
    call.deep = plan.deep;
    call.slices = plan.slices;
    const bool plain = p.bias == nullptr && p.residual == nullptr && p.addend == nullptr && !p.accumulate &&
                       (!p.c_f32 || std::is_same_v<T, float>) && !p.ragged;
    call.epilogue = split ? SmallEpilogue::split : plain ? SmallEpilogue::plain : SmallEpilogue::general;
    if constexpr (std::is_same_v<T, bf16_t>) return gemm_small_bf16(call, stream);
    else if constexpr (std::is_same_v<T, f16_t>) return gemm_small_f16(call, stream);
    else return gemm_small_f32(call, stream);
}

template <typename T>
int run_plan(const GemmArgs& g, const Plan& plan, KernelArgs p, hipStream_t stream) {
    p.tiles_m = (p.m + plan.tile - 1) / plan.tile;
    p.tiles_n = (p.n + plan.tile - 1) / plan.tile;
    p.k_tiles_per_slice = plan.k_tiles_per_slice;
    auto launch = [&]<bool SPLIT>(const KernelArgs& args) -> int {
        if (plan.tile <= 64) return launch_small_call<T>(g, args, plan, SPLIT, stream);
        if constexpr (!std::is_same_v<T, float>) {
            if (plan.tile == 256) return launch_layout<T, 256, 256, SPLIT>(args, g.a_k_contiguous, g.b_k_contiguous, plan.slices, stream);
        }
        return launch_layout<T, 128, 128, SPLIT>(args, g.a_k_contiguous, g.b_k_contiguous, plan.slices, stream);
    };
    if (plan.slices == 1) return launch.template operator()<false>(p);
    KernelArgs split = p;
    split.c = g.split_workspace;
    split.ld_partial = static_cast<long>(round_up(g.n, 8));
    if (int s = launch.template operator()<true>(split)) return s;
    const long quads = static_cast<long>(p.m) * (split.ld_partial / 4);
    const long blocks = std::min<long>((quads + kThreads - 1) / kThreads, static_cast<long>(compute_units()) * 8);
    hipLaunchKernelGGL((splitk_reduce_kernel<T>), dim3(static_cast<unsigned int>(blocks)), dim3(kThreads), 0, stream,
                       g.c, static_cast<const float*>(g.split_workspace), static_cast<const T*>(g.bias), p.m,
                       static_cast<int>(split.ld_partial), p.n, p.ldc, plan.slices, p.accumulate, p.c_f32, p.ragged);
    CGPTX_LAUNCH_CHECK();
    return CGPTX_OK;
}

// Validates column segments (widths multiples of `granule` except the last, summing to `total`,
// 16-byte aligned rows) and copies them into the kernel arguments.
int copy_segments(const GemmSegments& in, std::size_t total, std::size_t granule, KernelSegments& out) {
    out = KernelSegments{};
    if (in.count == 0) return CGPTX_OK;
    if (in.count < 0 || in.count > 3) return fail(CGPTX_INVALID_ARGUMENT, "gemm: one to three segments");
    std::size_t sum = 0;
    for (int s = 0; s < in.count; ++s) {
        const bool last = s + 1 == in.count;
        if (in.ptr[s] == nullptr || in.cols[s] == 0 || in.ld[s] < in.cols[s] || in.ld[s] % 8 != 0 || in.cols[s] % 8 != 0 ||
            !is_aligned16(in.ptr[s]) || (!last && in.cols[s] % granule != 0) ||
            in.cols[s] > static_cast<std::size_t>(std::numeric_limits<int>::max()))
            return fail(CGPTX_INVALID_ARGUMENT, "gemm: malformed operand segment");
        out.ptr[s] = in.ptr[s];
        out.ld[s] = static_cast<long>(in.ld[s]);
        out.cols[s] = static_cast<int>(in.cols[s]);
        sum += in.cols[s];
    }
    if (sum != total) return fail(CGPTX_INVALID_ARGUMENT, "gemm: segments do not cover the operand");
    out.count = in.count;
    return CGPTX_OK;
}

// The streamed loads address an operand relative to the block's tile origin with 32-bit byte
// offsets: a tile's rows (k-contiguous operand) or the whole K extent (n-contiguous operand).
bool offsets_fit_32bit(const GemmArgs& g, std::size_t elem) {
    // Below 2 GiB: bit 31 of a scalar offset is what pushes the loads of K tiles past the end out of range.
    constexpr std::size_t limit = (std::size_t{1} << 31) - (std::size_t{1} << 20);
    const std::size_t a_span = g.a_k_contiguous ? (256 * g.lda + g.k) * elem : (g.k * g.lda + 256) * elem;
    const std::size_t b_span = g.b_k_contiguous ? (256 * g.ldb + g.k) * elem : (g.k * g.ldb + 256) * elem;
    // The epilogues address a wavefront's part of C (of the residual, of a split-K partial tile)
    // through a range-checked descriptor with 32-bit offsets as well: up to 256 rows.
    std::size_t c_ld = std::max(g.ldc, g.n);
    for (int s = 0; s < g.c_segments.count; ++s) c_ld = std::max(c_ld, g.c_segments.ld[s]);
    const std::size_t c_span = 256 * c_ld * 4;
    const std::size_t r_span = g.residual != nullptr ? 256 * g.ldr * elem : 0;
    return a_span < limit && b_span < limit && c_span < limit && r_span < limit;
}

// Which operands the streamed kernels can read as they lie: 16-byte aligned rows whose K range (k-contiguous) or
// whose rows or columns (otherwise) are whole units of what a load instruction or a K tile covers. The K range of a
// k-contiguous operand has to end with a K tile, since what lies behind it in the row is multiplied too; a k-strided
// operand's may end anywhere (rows past it are out of the buffer's range).
bool a_streams(const GemmArgs& g) {
    const std::size_t chunk = 16 / dtype_size(g.dtype);
    return is_aligned16(g.a) && g.lda % chunk == 0 &&
           (g.a_k_contiguous ? g.k % (4 * chunk) == 0 : std::max(g.a_extent, g.m) % chunk == 0);
}
bool b_streams(const GemmArgs& g) {
    const std::size_t chunk = 16 / dtype_size(g.dtype);
    return is_aligned16(g.b) && g.ldb % chunk == 0 &&
           (g.b_k_contiguous ? g.k % (4 * chunk) == 0 : std::max(g.b_extent, g.n) % chunk == 0);
}
// Whether C and what is added to it lie in whole aligned chunks.
bool c_streams(const GemmArgs& g, std::size_t elem) {
    const std::size_t c_elem = g.c_is_f32 ? 4 : elem;
    const std::uintptr_t four = 4 * elem - 1;  // bias and residual are read four elements at a time
    return g.n % 8 == 0 && (g.ldc * c_elem) % 16 == 0 && is_aligned16(g.c) &&
           (g.bias == nullptr || (reinterpret_cast<std::uintptr_t>(g.bias) & four) == 0) &&
           (g.residual == nullptr || ((reinterpret_cast<std::uintptr_t>(g.residual) & four) == 0 && g.ldr % 4 == 0)) &&
           (g.addend_f32 == nullptr || (is_aligned16(g.addend_f32) && g.ld_addend % 4 == 0));
}

// An operand whose rows the streamed kernels cannot read (odd widths, unaligned storage) is copied to padded rows
// first: one pass over the operand (a few microseconds) against a contraction that ran at the fp32 matrix rate, a
// sixteenth of the 16-bit one. Copies and split-K partial tiles share one request to the arena. *taken: whether the arena
// has room for the copies; nothing was launched if not.
template <typename T>
int run_padded(const GemmArgs& g, bool pad_a, bool pad_b, hipStream_t stream, bool* taken);

// Whole aligned calls that leave at least half of the chip idle unless a long K is split (weight gradients). A graph recorded
// without the partial tiles' memory would pay for that at every replay, so these insist on it and report that the arena
// cannot grow; the other calls are faster split but run as they can.
bool insists_on_split(const GemmArgs& g, bool ragged) {
    if (g.dtype == CGPTX_F32 || ragged || g.k % kBK<bf16_t> != 0 || g.m % 8 != 0 || g.k / kBK<bf16_t> < 32) return false;
    const std::size_t units = static_cast<std::size_t>(compute_units());
    const std::size_t large = ((g.m + 255) / 256) * ((g.n + 255) / 256), small = ((g.m + 127) / 128) * ((g.n + 127) / 128);
    return small <= units || (large >= 8 && 2 * large <= units && g.k / kBK<bf16_t> >= 32 * ((units + large - 1) / large));
}

// Whether a call's operands lie within the streamed kernels' 32-bit offsets, and which of them can be read as they lie.
struct Streams {
    bool reach = false, a = false, b = false;
};

// The kernels' arguments of a call.
template <typename T>
int describe(const GemmArgs& g, KernelArgs& p, Streams& streams) {
    p = KernelArgs{};
    p.a = g.a;
    p.b = g.b;
    p.c = g.c;
    p.bias = g.bias;
    p.residual = g.residual;
    p.ldr = static_cast<long>(g.ldr);
    p.addend = g.addend_f32;
    p.ld_addend = static_cast<long>(g.ld_addend);
    p.m = static_cast<int>(g.m);
    p.n = static_cast<int>(g.n);
    p.k = static_cast<int>(g.k);
    p.a_extent = static_cast<int>(std::max(g.a_extent, g.m));
    p.b_extent = static_cast<int>(g.b_extent != 0 ? g.b_extent : g.n);
    p.b_k = static_cast<int>(g.b_k != 0 ? g.b_k : g.k);
    p.k_tiles = static_cast<int>((g.k + kBK<T> - 1) / kBK<T>);
    p.lda = static_cast<long>(g.lda);
    p.ldb = static_cast<long>(g.ldb);
    p.ldc = static_cast<long>(g.ldc);
    p.accumulate = g.accumulate ? 1 : 0;
    p.c_f32 = g.c_is_f32 ? 1 : 0;
    if (g.swiglu_out != nullptr) {
        if (!gemm_fuses_swiglu(g)) return fail(CGPTX_INVALID_ARGUMENT, "gemm: this call cannot carry the SwiGLU epilogue");
        p.act = g.swiglu_out;
        p.ld_act = static_cast<long>(g.ld_swiglu);
        p.inter = static_cast<int>(g.n / 2);
    }
    if (g.swiglu_saved != nullptr) {
        if (!gemm_fuses_swiglu_gradient(g)) return fail(CGPTX_INVALID_ARGUMENT, "gemm: this call cannot carry the SwiGLU gradient epilogue");
        p.saved = g.swiglu_saved;
        p.ld_saved = static_cast<long>(g.ld_swiglu);
        p.inter = static_cast<int>(g.n);
    }
    if (g.batch_rows != 0) {
        if (!gemm_takes_batch(g)) return fail(CGPTX_INVALID_ARGUMENT, "gemm: this call cannot be a stack of products");
        p.batch_rows = static_cast<int>(g.batch_rows);
        p.a_batch_stride = static_cast<long>(g.a_batch_stride);
        p.b_batch_stride = static_cast<long>(g.b_batch_stride);
        for (int s = 0; s < 3; ++s) p.a_seg_batch_stride[s] = static_cast<long>(g.a_segment_batch_stride[s]);
    }
    const bool segmented = g.a_segments.count > 0 || g.c_segments.count > 0;
    if (segmented) {
        if (int s = copy_segments(g.a_segments, g.a_k_contiguous ? g.k : (g.batch_rows != 0 ? g.batch_rows : g.m),
                                  g.a_k_contiguous ? kSteps * kBK<T> : 256, p.a_seg))
            return s;
        if (int s = copy_segments(g.c_segments, g.n, 256, p.c_seg)) return s;
        if (g.c_segments.count > 0 && (g.c_is_f32 || g.residual != nullptr))
            return fail(CGPTX_INVALID_ARGUMENT, "gemm: a segmented output takes neither fp32 storage nor a residual");
        if (std::is_same_v<T, float>) return fail(CGPTX_INVALID_ARGUMENT, "gemm: segmented operands need 16-bit storage");
    }

    GemmArgs whole = g;  // alignment of segmented operands was checked per segment
    if (g.a_segments.count > 0) {
        whole.a = g.a_segments.ptr[0];
        whole.lda = g.a_segments.ld[0];
    }
    if (g.c_segments.count > 0) {
        whole.c = const_cast<void*>(g.c_segments.ptr[0]);
        whole.ldc = g.c_segments.ld[0];
    }
    streams = Streams{};
    if ((g.a_k_contiguous || !g.b_k_contiguous) && offsets_fit_32bit(whole, sizeof(T))) {
        streams.reach = true;
        streams.a = a_streams(whole);
        streams.b = b_streams(whole);
        p.ragged = c_streams(whole, sizeof(T)) ? 0 : 1;
    }
    return CGPTX_OK;
}

template <typename T>
int run_typed(const GemmArgs& g, hipStream_t stream) {
    KernelArgs p;
    Streams streams;
    if (int s = describe<T>(g, p, streams)) return s;
    const bool segmented = g.a_segments.count > 0 || g.c_segments.count > 0;
    const bool fast = streams.a && streams.b;
    if (streams.reach && !fast && !segmented && g.batch_rows == 0 && !g.no_split) {
        bool taken = false;
        const int s = run_padded<T>(g, !streams.a, !streams.b, stream, &taken);
        if (taken || s != CGPTX_OK) return s;
    }
    if (p.ragged && segmented) return fail(CGPTX_INVALID_ARGUMENT, "gemm: segmented operands need the aligned MFMA path");
    if (!fast && segmented) return fail(CGPTX_INVALID_ARGUMENT, "gemm: segmented operands need the aligned MFMA path");
    if (!fast && g.batch_rows != 0) return fail(CGPTX_INVALID_ARGUMENT, "gemm: a stack of products needs the aligned MFMA path");
    if (!fast) {
        const dim3 grid(static_cast<unsigned int>((g.n + kF32Tile - 1) / kF32Tile),
                        static_cast<unsigned int>((g.m + kF32Tile - 1) / kF32Tile));
        if (grid.y > 65535u) return fail(CGPTX_OVERFLOW, "gemm: too many rows for the fp32 kernel's grid");
        hipLaunchKernelGGL((gemm_f32_mfma_kernel<T>), grid, dim3(kThreads), 0, stream, p, g.a_k_contiguous ? 1 : 0,
                           g.b_k_contiguous ? 1 : 0);
        CGPTX_LAUNCH_CHECK();
        return CGPTX_OK;
    }
    Plan plan = make_plan(g);
    if (plan.slices == 1 || g.no_split) return run_plan<T>(g, plan, p, stream);
    GemmArgs split = g;
    const std::size_t wanted = plan.partial_bytes(g);
    if (int s = scratch_up_to(stream, wanted, &split.split_workspace, &split.split_workspace_bytes)) return s;
    if (split.split_workspace_bytes < wanted) {
        split.no_split = true;  // but into the room there is
        const Plan smaller = make_plan(split);
        if (g.batch_rows != 0 || (smaller.slices == 1 && insists_on_split(g, p.ragged != 0))) {
            if (int s = scratch(stream, wanted, &split.split_workspace)) return s;  // says what is in the way
        } else {
            plan = smaller;
        }
    }
    return run_plan<T>(split, plan, p, stream);
}

template <typename T>
int run_padded(const GemmArgs& g, bool pad_a, bool pad_b, hipStream_t stream, bool* taken) {
    GemmArgs padded = g;
    const std::size_t k_whole = round_up(g.k, kBK<T>), chunk = kVec128<T>;
    std::size_t a_bytes = 0, b_bytes = 0;
    if (pad_a) {
        padded.lda = g.a_k_contiguous ? k_whole : round_up(g.m, chunk);
        padded.a_extent = g.a_k_contiguous ? g.m : padded.lda;
        a_bytes = round_up((g.a_k_contiguous ? g.m : g.k) * padded.lda * sizeof(T), 256);
    }
    if (pad_b) {
        padded.ldb = g.b_k_contiguous ? k_whole : round_up(g.n, chunk);
        padded.b_extent = g.b_k_contiguous ? g.n : padded.ldb;
        b_bytes = round_up((g.b_k_contiguous ? g.n : g.k) * padded.ldb * sizeof(T), 256);
    }
    if (g.a_k_contiguous) padded.k = k_whole;  // A's rows then end in zeros, B's K range ends where it did
    if (!g.b_k_contiguous) padded.b_k = g.b_k != 0 ? g.b_k : g.k;
    const std::size_t split_bytes = make_plan(padded).partial_bytes(padded);
    void* mem = nullptr;
    std::size_t held = 0;
    if (int s = scratch_up_to(stream, a_bytes + b_bytes + split_bytes, &mem, &held)) return s;
    *taken = held >= a_bytes + b_bytes;
    if (!*taken) return CGPTX_OK;
    auto* base = static_cast<char*>(mem);
    if (pad_a) {
        padded.a = base;
        const std::size_t rows = g.a_k_contiguous ? g.m : g.k, cols = g.a_k_contiguous ? g.k : g.m;
        if (int s = pad_rows(base, g.a, rows, cols, g.lda, padded.lda, g.dtype, stream)) return s;
    }
    if (pad_b) {
        padded.b = base + a_bytes;
        const std::size_t rows = g.b_k_contiguous ? g.n : g.k, cols = g.b_k_contiguous ? g.k : g.n;
        if (int s = pad_rows(base + a_bytes, g.b, rows, cols, g.ldb, padded.ldb, g.dtype, stream)) return s;
    }
    padded.no_split = true;
    padded.split_workspace = split_bytes != 0 ? base + a_bytes + b_bytes : nullptr;
    padded.split_workspace_bytes = std::min(split_bytes, held - a_bytes - b_bytes);
    return run_typed<T>(padded, stream);
}

// A group's tiles: those whose predicted time in one launch is least. The launch takes as long as its longest workgroup or
// as the busiest CU's share of the work, whatever is more (us per K tile and workgroup as in predicted_us; 3.5 us before and
// after the K loops). Joined if that is less than the calls' own predictions in turn. [M, N] x K measured apart and joined:
// dX and dW of 128 x 768 x 768 10.4 -> 7.7 us, of 2000 x 1024 x 2048 37.4 -> 34.3; 5005 x 1024 x 256, whose dW is better
// split along K, 23.9 -> 28.8: stays apart.
struct GroupPlan {
    int tile[kGroupCalls] = {};
    long blocks = 0;
    bool joined = false;
};

GroupPlan plan_group(const GemmArgs* calls, int count) {
    GroupPlan best_plan;
    const double units = static_cast<double>(compute_units());
    double separate = 0.0;
    for (int i = 0; i < count; ++i) {
        const GemmArgs& g = calls[i];
        const Plan plan = make_plan(g);
        const long tiles = static_cast<long>((g.m + plan.tile - 1) / plan.tile) * static_cast<long>((g.n + plan.tile - 1) / plan.tile);
        const bool f32 = g.dtype == CGPTX_F32;
        const long k_step = f32 ? kBK<float> : kBK<bf16_t>, k_tiles = (static_cast<long>(g.k) + k_step - 1) / k_step;
        separate += predicted_us(plan.tile, tiles, plan.slices, k_tiles, static_cast<double>(plan.partial_bytes(g)) * 1e-6, f32,
                                 g.a_k_contiguous, g.b_k_contiguous, compute_units());
        if (g.a_sums != nullptr) separate += 6.0;  // two launches of their own
    }
    double best = separate;
    for (int choice = 0; choice < 1 << count; ++choice) {
        double longest = 0.0, work = 0.0, blocks = 0.0;
        for (int i = 0; i < count; ++i) {
            const GemmArgs& g = calls[i];
            const bool f32 = g.dtype == CGPTX_F32, small = ((choice >> i) & 1) != 0;
            const long edge = small ? 32 : 64, k_step = f32 ? kBK<float> : kBK<bf16_t>;
            const double kt = static_cast<double>((static_cast<long>(g.k) + k_step - 1) / k_step);
            const double tiles = static_cast<double>((g.m + edge - 1) / edge) * static_cast<double>((g.n + edge - 1) / edge);
            const double lone = f32 ? (small ? 0.088 : 0.265) : small ? (!g.a_k_contiguous ? 0.1 : g.b_k_contiguous ? 0.07 : 0.085) : 0.135;
            const double shared = f32 ? lone : small ? 0.92 * lone : 0.128;
            longest = std::max(longest, f32 || small ? kt * lone : 0.02 * std::min(kt, 16.0) + std::max(0.0, kt - 16.0) * lone);
            work += tiles * kt * shared;
            blocks += tiles;
        }
        const double load = blocks / units;
        if (load > 1.0) longest *= 1.4;  // beside the other workgroup of its CU
        const double time = 3.5 + std::max(longest, load <= 1.0 ? 0.0 : work / units * std::ceil(load) / load * (load > 4.0 ? 1.3 : 1.0));
        if (time < best && blocks <= 16.0 * units) {
            best = time;
            best_plan.joined = true;
            best_plan.blocks = static_cast<long>(blocks);
            for (int i = 0; i < count; ++i) best_plan.tile[i] = ((choice >> i) & 1) != 0 ? 32 : 64;
        }
    }
    return best_plan;
}

// Whether a call can be part of a group: streamed as it lies, one sum over K, nothing but the plain additions behind it.
template <typename T>
bool joinable(const GemmArgs& g, KernelArgs& p) {
    if (g.a == nullptr && g.a_segments.count == 0) return false;
    if (g.b == nullptr || g.c == nullptr || g.m == 0 || g.n == 0 || g.k == 0 || g.batch_rows != 0 || g.swiglu_out != nullptr ||
        g.swiglu_saved != nullptr || g.c_segments.count > 0 || (g.a_sums != nullptr && g.a_k_contiguous) ||
        (g.a_segments.count > 0 && (!g.a_k_contiguous || g.b_k_contiguous || std::is_same_v<T, float>)))
        return false;
    constexpr std::size_t i32max = std::numeric_limits<int>::max();
    if (g.m > i32max || g.n > i32max || g.k > i32max) return false;
    GemmArgs whole = g;
    GemmSegments segments = g.a_segments;
    whole.a_segments = GemmSegments{};
    if (segments.count > 0) {
        whole.a = segments.ptr[0];
        whole.lda = segments.ld[0];
    }
    Streams streams;
    if (describe<T>(whole, p, streams) != CGPTX_OK || !streams.a || !streams.b) {
        clear_error();
        return false;
    }
    if (segments.count > 0) {
        if (copy_segments(segments, g.k, kBK<T>, p.a_seg) != CGPTX_OK || segments.cols[segments.count - 1] % kBK<T> != 0) {
            clear_error();
            return false;
        }
    }
    return true;
}

template <typename T>
int run_joined(const GemmArgs* calls, int count, const GroupPlan& plan, hipStream_t stream) {
    SmallGroup group{};
    long order[kGroupCalls];
    for (int i = 0; i < count; ++i) order[i] = i;
    // The workgroups with the longest K loops start first.
    std::sort(order, order + count, [&](long x, long y) { return calls[x].k * plan.tile[x] > calls[y].k * plan.tile[y]; });
    int blocks = 0;
    for (int j = 0; j < count; ++j) {
        const long i = order[j];
        const GemmArgs& g = calls[i];
        KernelArgs p;
        if (!joinable<T>(g, p)) return fail(CGPTX_RUNTIME, "gemm: this call cannot be part of a group");
        group.call[j] = small_args(p, false, p.k_tiles);
        group.call[j].a_sums = g.a_sums;
        group.call[j].a_sums_accumulate = g.a_sums_accumulate ? 1 : 0;
        group.first_block[j] = blocks;
        group.tile[j] = plan.tile[i];
        group.tiles_m[j] = (p.m + plan.tile[i] - 1) / plan.tile[i];
        group.layout[j] = !g.a_k_contiguous ? SmallLayout::weight_gradient
                          : g.b_k_contiguous ? SmallLayout::forward
                          : p.a_seg.count > 0 ? SmallLayout::segmented_input_gradient : SmallLayout::input_gradient;
        blocks += group.tiles_m[j] * ((p.n + plan.tile[i] - 1) / plan.tile[i]);
    }
    group.count = count;
    const bool deep = blocks <= compute_units();
    if constexpr (std::is_same_v<T, bf16_t>) return gemm_small_bf16(group, blocks, deep, stream);
    else if constexpr (std::is_same_v<T, f16_t>) return gemm_small_f16(group, blocks, deep, stream);
    else return gemm_small_f32(group, blocks, deep, stream);
}

}  // namespace

bool gemm_joins(const GemmArgs* calls, int count) {
    if (count < 2 || count > kGroupCalls || forced_tile() != 0) return false;
    for (int i = 0; i < count; ++i) {
        if (calls[i].dtype != calls[0].dtype || !valid_dtype(calls[i].dtype)) return false;
        KernelArgs p;
        const bool fits = calls[i].dtype == CGPTX_F32 ? joinable<float>(calls[i], p)
                          : calls[i].dtype == CGPTX_F16 ? joinable<f16_t>(calls[i], p) : joinable<bf16_t>(calls[i], p);
        if (!fits) return false;
    }
    return plan_group(calls, count).joined;
}

int gemm_joined(const GemmArgs* calls, int count, hipStream_t stream) {
    if (!gemm_joins(calls, count)) return fail(CGPTX_RUNTIME, "gemm: these calls cannot share a launch");
    const GroupPlan plan = plan_group(calls, count);
    return dispatch_dtype(calls[0].dtype, [&]<typename T>() -> int { return run_joined<T>(calls, count, plan, stream); });
}

bool gemm_fuses_swiglu(const GemmArgs& g) {
    if (g.swiglu_out == nullptr || g.dtype == CGPTX_F32 || !g.a_k_contiguous || !g.b_k_contiguous || g.bias != nullptr ||
        g.residual != nullptr || g.accumulate || g.c_is_f32 || g.a_segments.count > 0 || g.c_segments.count > 0 ||
        g.a == nullptr || g.b == nullptr || g.c == nullptr)
        return false;
    const std::size_t elem = 2, inter = g.n / 2;
    // Whole 128-column units of gate and of up per tile, tiles that fill the chip (the 256x256
    // configuration), 16-byte aligned rows everywhere, and the whole weight within 32-bit offsets.
    if (g.n % 256 != 0 || g.k % kBK<bf16_t> != 0 || g.lda % 8 != 0 || g.ldb % 8 != 0 || g.ldc % 8 != 0 ||
        g.ld_swiglu % 8 != 0 || g.ld_swiglu < inter || !is_aligned16(g.a) || !is_aligned16(g.b) || !is_aligned16(g.c) ||
        !is_aligned16(g.swiglu_out))
        return false;
    const long tiles = static_cast<long>((g.m + 255) / 256) * static_cast<long>(g.n / 256);
    if ((forced_tile() != 0 && forced_tile() != 256) || tiles * 5 < static_cast<long>(compute_units()) * 4) return false;
    constexpr std::size_t limit = (std::size_t{1} << 31) - (std::size_t{1} << 20);
    return offsets_fit_32bit(g, elem) && (g.n * g.ldb + g.k) * elem < limit && 256 * g.ld_swiglu * elem < limit;
}

bool gemm_fuses_swiglu_gradient(const GemmArgs& g) {
    if (g.swiglu_saved == nullptr || g.swiglu_out != nullptr || g.dtype == CGPTX_F32 || !g.a_k_contiguous || g.b_k_contiguous ||
        g.bias != nullptr || g.residual != nullptr || g.accumulate || g.c_is_f32 || g.a_segments.count > 0 ||
        g.c_segments.count > 0 || g.a == nullptr || g.b == nullptr || g.c == nullptr)
        return false;
    const std::size_t elem = 2;
    // 16-byte chunks of whole rows everywhere, tiles that fill the chip (the 256x256 configuration),
    // and a wavefront's 128 rows of the saved and of the written [gate | up] within 32-bit offsets.
    if (g.n % 8 != 0 || g.k % kBK<bf16_t> != 0 || g.lda % 8 != 0 || g.ldb % 8 != 0 || g.ldc % 8 != 0 ||
        g.ld_swiglu % 8 != 0 || g.ldc < 2 * g.n || g.ld_swiglu < 2 * g.n || !is_aligned16(g.a) || !is_aligned16(g.b) ||
        !is_aligned16(g.c) || !is_aligned16(g.swiglu_saved))
        return false;
    const long tiles = static_cast<long>((g.m + 255) / 256) * static_cast<long>((g.n + 255) / 256);
    if ((forced_tile() != 0 && forced_tile() != 256) || tiles * 5 < static_cast<long>(compute_units()) * 4) return false;
    constexpr std::size_t limit = (std::size_t{1} << 31) - (std::size_t{1} << 20);
    return offsets_fit_32bit(g, elem) && 256 * g.ld_swiglu * elem < limit;
}

bool gemm_takes_batch(const GemmArgs& g) {
    if (g.batch_rows == 0) return true;
    if (g.dtype == CGPTX_F32 || g.a_k_contiguous || g.b_k_contiguous || g.bias != nullptr || g.residual != nullptr ||
        g.addend_f32 != nullptr || g.accumulate || g.c_is_f32 || g.c_segments.count > 0 || g.swiglu_out != nullptr ||
        g.swiglu_saved != nullptr || g.no_split || g.c == nullptr || g.b == nullptr)
        return false;
    if (g.batch_rows % 256 != 0 || g.m % g.batch_rows != 0 || g.n % 8 != 0 || g.ldb % 8 != 0 ||
        g.ldc % 8 != 0 || g.b_batch_stride % 8 != 0)
        return false;
    if (g.a_segments.count == 0) return g.a != nullptr && g.lda % 8 == 0 && g.a_batch_stride % 8 == 0;
    for (int s = 0; s < g.a_segments.count && s < 3; ++s)
        if (g.a_segment_batch_stride[s] % 8 != 0) return false;
    return true;
}

int pad_rows(void* dst, const void* src, std::size_t rows, std::size_t cols, std::size_t ld, std::size_t pitch, int dtype,
             hipStream_t stream) {
    const std::size_t chunks = rows * (pitch * dtype_size(dtype) / 16);
    const dim3 grid(static_cast<unsigned int>(std::min<std::size_t>((chunks + kThreads - 1) / kThreads, static_cast<std::size_t>(compute_units()) * 16)));
    auto launch = [&]<typename E>() {
        hipLaunchKernelGGL((pad_rows_kernel<E>), grid, dim3(kThreads), 0, stream, static_cast<E*>(dst), static_cast<const E*>(src),
                           static_cast<long>(rows), static_cast<int>(cols), static_cast<long>(ld), static_cast<int>(pitch));
    };
    if (dtype == CGPTX_F32) launch.template operator()<std::uint32_t>();
    else launch.template operator()<std::uint16_t>();
    CGPTX_LAUNCH_CHECK();
    return CGPTX_OK;
}

std::size_t gemm_split_bytes(const GemmArgs& g) { return make_plan(g).partial_bytes(g); }

int gemm(const GemmArgs& g, hipStream_t stream) {
    if ((g.a == nullptr && g.a_segments.count == 0) || g.b == nullptr || (g.c == nullptr && g.c_segments.count == 0) ||
        g.m == 0 || g.n == 0 || g.k == 0)
        return fail(CGPTX_INVALID_ARGUMENT, "gemm: null or empty operand");
    constexpr std::size_t i32max = std::numeric_limits<int>::max();
    if (g.m > i32max || g.n > i32max || g.k > i32max)
        return fail(CGPTX_OVERFLOW, "gemm: dimension exceeds int range");
    return dispatch_dtype(g.dtype, [&]<typename T>() -> int { return run_typed<T>(g, stream); });
}

}  // namespace cgptx
