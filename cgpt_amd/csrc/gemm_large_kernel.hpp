// Persistent contraction kernels: C[M,N] (+)= op(A)·op(B) on 256 x 256, 256 x 192 and 128 x 128 tiles.
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
#pragma once

#include "gemm_large.hpp"
#include "gemm_tiles.hpp"

#include <algorithm>

namespace cgptx {
namespace {

// An n-contiguous operand's tile.
template <typename T, int COLS>
struct ColumnTile {
    using type = NTile<T, COLS>;
};
template <typename T>
struct ColumnTile<T, 192> {
    using type = NTile192<T>;
};

// Tiles that are not square, but 256 x 192 ones: more heights between 128 and 256 rows, for calls whose square tiles would leave CUs
// idle (oblong_tiles).
template <int BM, int BN>
constexpr bool is_oblong = BM != BN && BN != 192;

// The rings' slots of a tile that has a CU to itself: whatever lets the operand that is requested last be requested earliest (A's K
// tile 2 kASlots - 3 steps before it is read, B's 2 kBSlots - 2), in as little of the LDS as that takes.
struct RingSlots {
    int a, b;
};
constexpr RingSlots ring_slots(int a_bytes, int b_bytes) {
    RingSlots best{0, 0};
    int best_lead = 0, best_bytes = 0;
    for (int a = 3; a <= 8; ++a)
        for (int b = 2; b <= 8; ++b) {
            const int bytes = a * a_bytes + b * b_bytes, lead = 2 * a - 3 < 2 * b - 2 ? 2 * a - 3 : 2 * b - 2;
            if (bytes > kLdsBytes || lead < best_lead || (lead == best_lead && bytes >= best_bytes)) continue;
            best = {a, b};
            best_lead = lead;
            best_bytes = bytes;
        }
    return best;
}

// LDS holds a ring of K tiles of A and one of B (a K tile: two K steps, 128 bytes along K per row or column). Two slots of
// each hold the K tile being multiplied and the next one, the rest what is in flight beyond them. 256 x 256 blocks own a CU
// (3 x 32 + 2 x 32 KiB; 256 x 192: 3 x 32 + 2 x 24), 128 x 128 blocks run two per CU (3 x 16 + 2 x 16 KiB each) or, where there is no second one for a
// CU, DEEP: one with 5 + 4 slots.
template <typename T, int BM, int BN, bool A_K, bool B_K, bool DEEP>
struct TileLayout {
    using ATile = std::conditional_t<A_K, KTile<T, BM>, NTile<T, BM>>;
    using BTile = std::conditional_t<B_K, KTile<T, BN>, typename ColumnTile<T, BN>::type>;
    static constexpr RingSlots kOblong = ring_slots(ATile::kElems * static_cast<int>(sizeof(T)), BTile::kElems * static_cast<int>(sizeof(T)));
    static constexpr int kASlots = is_oblong<BM, BN> ? kOblong.a : DEEP ? 5 : 3, kBSlots = is_oblong<BM, BN> ? kOblong.b : DEEP ? 4 : 2;
    static constexpr int kSmemBytes = (kASlots * ATile::kElems + kBSlots * BTile::kElems) * static_cast<int>(sizeof(T));
    // The order of an item's requests: A's K tile x is requested in the first step of K tile x + 1 - kASlots, B's in the
    // second step of x - kBSlots. Steps are numbered 2 t (first) and 2 t + 1 (second); what is due before step 0 is
    // requested ahead of the loop, in the same order.
    static constexpr int a_due(int x) { return 2 * (x + 1 - kASlots); }
    static constexpr int b_due(int x) { return 2 * (x - kBSlots) + 1; }
    // Requests due after `after` and before `until`, in loads of a wavefront.
    static constexpr int loads_between(int after, int until) {
        int loads = 0;
        for (int due = after + 1; due < until; ++due) loads += due % 2 == 0 ? ATile::kLoads : BTile::kLoads;
        return loads;
    }
    // Loads that may still be outstanding when K tile x's operands are needed, just before step `until`.
    static constexpr int outstanding(int x, int until) { return loads_between(a_due(x) > b_due(x) ? a_due(x) : b_due(x), until); }
    // The first request ahead of the loop, and how many there are.
    static constexpr int kFirstDue = a_due(0) < b_due(0) ? a_due(0) : b_due(0);
    static constexpr bool requested_ahead(int due) { return due % 2 == 0 ? due >= a_due(0) : due >= b_due(0); }
};

// Stores a lane's 16 bytes at voffset + soffset of a buffer. The sum is taken in the vector register: behind a 16-byte store
// with a scalar offset the compiler lets the very next instruction overwrite the data registers, and on this chip the store
// has then not always read them (128 x 128 tiles, two wavefronts a SIMD: the first four bytes of some hundred stores in a
// [32768, 768] result were the next value's). Without one it keeps the distance.
__device__ __forceinline__ void store_chunk(const u32x4& data, __amdgpu_buffer_rsrc_t rsrc, int voffset, int soffset) {
    __builtin_amdgcn_raw_buffer_store_b128(data, rsrc, voffset + soffset, 0, 0);
}

// Nothing is added to the result, and it is stored in the operands' type on rows of whole 16 bytes.
__device__ __host__ __forceinline__ bool stored_as_it_is(const KernelArgs& p) {
    return p.bias == nullptr && p.residual == nullptr && p.addend == nullptr && !p.accumulate && !p.c_f32 && !p.ragged;
}
// Such calls have a kernel of their own. Not on 256 x 256 tiles, which gain nothing by it (0.996 - 1.009 over four workloads).
template <int BM, bool SPLIT, bool RESIDUAL, bool SWIGLU, bool GRAD>
constexpr bool plain_apart = BM == 128 && !SPLIT && !RESIDUAL && !SWIGLU && !GRAD;

// The K slices of a tile, each in the accumulators of a workgroup: everybody leaves its own in memory, takes a ticket, and
// the last one adds them up in slice order (whoever it is) and goes on with the sum. Written through to the memory behind the XCDs'
// L2s and read from there: the workgroups of a tile run on any XCD. In the accumulators' own layout, 16 bytes per lane: whole
// cache lines, and no way through LDS. True for the last one (fold_share says how it knows).
template <typename T, int TM, int TN, bool SUMS>
__device__ __forceinline__ bool fold_slices(const KernelArgs& p, acc_t (&acc)[TM][TN], acc_t (&column_sums)[SUMS ? TM : 1], bool sums,
                                            int slice, int tiles, int tile, int wm, unsigned char* smem_raw) {
    constexpr int kAgent = 16;  // sc1
    constexpr int kTileBytes = fold_tile_bytes(TM * 32, TN * 32);
    const int lane = threadIdx.x & (kWave - 1);
    auto rsrc_of = [&](int s) __attribute__((always_inline)) {
        return __builtin_amdgcn_make_buffer_rsrc(p.fold_partial + (static_cast<long>(s) * tiles + tile) * kTileBytes, 0, kTileBytes, 0x00020000);
    };
    const int voffset = threadIdx.x * 16, sum_voffset = TM * 32 * TN * 32 * 4 + (wm * TM * 16 + lane) * 4;
    {
        const auto rsrc = rsrc_of(slice);
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                acc_t v;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    float x = acc[i][j][e];
                    asm volatile("v_accvgpr_read_b32 %0, %1" : "=v"(x) : "a"(x));
                    v[e] = x;
                }
                __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), rsrc, voffset + (i * TN + j) * kThreads * 16, 0, kAgent);
            }
        if constexpr (SUMS) {
            if (sums && lane < 16) {
#pragma unroll
                for (int i = 0; i < TM; ++i)
                    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned int, static_cast<float>(column_sums[i][0])), rsrc, sum_voffset + i * 64, 0, kAgent);
            }
        }
    }
    __builtin_amdgcn_s_waitcnt(vmcnt_immediate(0));
    __syncthreads();
    auto* const arrived = reinterpret_cast<unsigned int*>(smem_raw);
    if (threadIdx.x == 0) {
        const unsigned int share = fold_share(slice, p.slices);
        *arrived = __hip_atomic_fetch_add(p.fold_tickets + tile, share, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + share;
    }
    __syncthreads();
    const bool last = __builtin_amdgcn_readfirstlane(*arrived) == 0u;
    __syncthreads();
    if (!last) return false;
    for (int s = 0; s < p.slices; ++s) {
        const auto rsrc = rsrc_of(s);
        u32x4 part[TM][TN];
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) part[i][j] = __builtin_amdgcn_raw_buffer_load_b128(rsrc, voffset + (i * TN + j) * kThreads * 16, 0, kAgent);
        float sum[TM];
        if constexpr (SUMS) {
#pragma unroll
            for (int i = 0; i < TM; ++i) sum[i] = sums && lane < 16 ? __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsrc, sum_voffset + i * 64, 0, kAgent)) : 0.0f;
        }
#pragma unroll
        for (int i = 0; i < TM; ++i) {
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                const acc_t v = __builtin_bit_cast(acc_t, part[i][j]);
                if (s == 0) acc[i][j] = v;
                else acc[i][j] += v;
            }
            if constexpr (SUMS) column_sums[i][0] = s == 0 ? sum[i] : column_sums[i][0] + sum[i];
        }
    }
    return true;
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
// PLAIN: the result is stored as it is, in the operands' type, by kernels of their own: with the general epilogue beside it the
// compiler spills 35 - 60 scalar registers (256-wide tiles: 120 - 150) and asks for private memory that nothing touches, without
// it 0 - 29 and none.
// FOLD: one item, whose K slice is added to the tile's others by whichever workgroup ends last (fold_slices), with the sums of A's
// columns beside it: the two gradients of a projection in one launch (gemm_pair_kernel).
template <typename T, int BM, int BN, bool A_K, bool B_K, bool SPLIT, bool SEGMENTED, bool RESIDUAL, bool SWIGLU, bool GRAD, bool DEEP,
          bool PLAIN, bool FOLD>
__device__ __forceinline__ void contract(const KernelArgs& p, int item, const int item_end, const int item_stride, unsigned char* smem_raw) {
    static_assert(!GRAD || (A_K && !B_K && !SPLIT && !SEGMENTED && !RESIDUAL && !SWIGLU && BN == 256),
                  "the SwiGLU gradient epilogue belongs to the plain input-gradient kernel with 256-wide tiles");
    static_assert(!SEGMENTED || (A_K && !B_K && !SPLIT && (PLAIN || BM == 256)),
                  "segments along K are read by unsplit input gradients that nothing is added to");
    static_assert(!RESIDUAL || (!SPLIT && !SEGMENTED), "the residual epilogue belongs to plain unsplit kernels");
    static_assert(!SWIGLU || (A_K && B_K && !SPLIT && !SEGMENTED && !RESIDUAL && BN == 256),
                  "the SwiGLU epilogue belongs to the plain forward kernel with 256-wide tiles");
    static_assert(!FOLD || (!SPLIT && !SEGMENTED && !RESIDUAL && !SWIGLU && !GRAD && !std::is_same_v<T, float>),
                  "slices are folded in the accumulators' layout");
    using frag_t = typename Mfma<T>::frag;
    using Layout = TileLayout<T, BM, BN, A_K, B_K, DEEP>;
    using ATile = typename Layout::ATile;
    using BTile = typename Layout::BTile;
    constexpr int WM = BM / 2, WN = BN / 2;
    constexpr int TM = WM / 16, TN = WN / 16;  // 16 x 16 MFMA blocks of a wavefront's part
    T* smem = reinterpret_cast<T*>(smem_raw);
    // K tile x of A lives in A's slot x % kASlots, of B in B's slot x % kBSlots.
    constexpr int kASlots = Layout::kASlots, kBSlots = Layout::kBSlots;
    constexpr unsigned int kASlotBytes = ATile::kElems * sizeof(T), kBSlotBytes = BTile::kElems * sizeof(T);
    constexpr int kBBase = kASlots * ATile::kElems;  // elements

    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int wm = wave >> 1, wn = wave & 1;
    // 256 x 192 tiles: a wavefront has half of the tile's first 128 columns and half of its last 64, so that each of its blocks
    // of 16 columns lies in one part of the operand's tile and C is stored in half lines at least.
    constexpr bool kNarrow = BN == 192;
    constexpr bool kOblong = is_oblong<BM, BN>;
    static_assert(!kOblong || ((A_K || FOLD) && !SPLIT && !RESIDUAL && !SWIGLU && !GRAD && PLAIN), "oblong tiles take unsplit calls of k-contiguous A that are stored as they are or with a residual");
    static_assert(!kNarrow || (BM == 256 && !SPLIT && !RESIDUAL && !SWIGLU && !GRAD && !FOLD), "256 x 192 tiles have an epilogue of their own");
    auto column_of = [&](int j) { return !kNarrow ? wn * WN + j * 16 : j < 4 ? wn * 64 + j * 16 : 128 + wn * 32 + (j - 4) * 16; };

    const int tiles = p.tiles_m * p.tiles_n;

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
    TileCursor cn;  // 256 x 192 tiles, B as [K, N]: its 64 columns' loads
    auto aim_b = [&](int t, TileCursor& cb) __attribute__((always_inline)) {
        const unsigned int past_end = src_begin + t * kSteps >= src_end ? 0x80000000u : 0u;
        const int k0 = min(src_begin + t * kSteps, src_end - 1) * kBK<T>;
        cb.rsrc = b_src.rsrc;
        cb.voffset = b_src.voffset;
        cb.soffset = b_src.first_offset(k0, wave) | past_end;
        cb.step = kWaves * b_src.group_bytes;
        if constexpr (kNarrow && !B_K) {
            cn.voffset = b_src.narrow_voffset;
            cn.soffset = b_src.narrow_first_offset(k0, wave) | past_end;
            cn.step = 2 * kWaves * b_src.group_bytes;
        }
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
    constexpr int kALoads = ATile::kLoads, kBLoads = BTile::kLoads;  // per wavefront and K tile
    static_assert(kASlots * kALoads + kBSlots * kBLoads < 64, "vmcnt counts the loads in flight");
    auto issue_a = [&](auto index, unsigned int slot_lds, TileCursor& ca) __attribute__((always_inline)) {
        constexpr int l = decltype(index)::value;
        ca.soffset = load_to_lds<l * kWaves * kLoadBytes>(ca.rsrc, slot_lds, ca.voffset, ca.soffset, ca.step);
    };
    auto issue_b = [&](auto index, unsigned int slot_lds, TileCursor& cb) __attribute__((always_inline)) {
        constexpr int l = decltype(index)::value;
        if constexpr (kNarrow && !B_K && l % 3 == 2) {
            cn.soffset = load_to_lds<l * kWaves * kLoadBytes>(cb.rsrc, slot_lds, cn.voffset, cn.soffset, cn.step);
            return;
        }
        const unsigned int step = !SWIGLU || l % 2 == 0 ? cb.step : l % 4 == 1 ? cb.step_up : cb.step_back;
        cb.soffset = load_to_lds<l * kWaves * kLoadBytes>(cb.rsrc, slot_lds, cb.voffset, cb.soffset, step);
    };
    const unsigned int a_lds = lds_address_of(smem) + wave * kLoadBytes, b_lds = a_lds + kBBase * static_cast<int>(sizeof(T));
    TileCursor ca, cb;
    // The opened item's requests due FIRST .. LAST-1 (all before its first step).
    auto request_due = [&]<int FIRST, int LAST>() __attribute__((always_inline)) {
        static_for<FIRST - Layout::kFirstDue, LAST - Layout::kFirstDue>([&](auto index) {
            constexpr int due = decltype(index)::value + Layout::kFirstDue;
            if constexpr (!Layout::requested_ahead(due)) {
            } else if constexpr (due % 2 == 0) {
                constexpr int x = due / 2 - 1 + kASlots;
                aim_a(x, ca);
                static_for<0, kALoads>([&](auto l) { issue_a(l, a_lds + x * kASlotBytes, ca); });
            } else {
                constexpr int x = (due - 1) / 2 + kBSlots;
                aim_b(x, cb);
                static_for<0, kBLoads>([&](auto l) { issue_b(l, b_lds + x * kBSlotBytes, cb); });
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
    for (int j = 0; j < kBOffsets; ++j) {
        if constexpr (kNarrow && !B_K) b_off[j] = j < 4 ? BTile::wide_offset(lane, column_of(j)) : BTile::narrow_offset(lane, column_of(j) - 128);
        else b_off[j] = B_K ? BTile::lane_offset(lane, j) : BTile::lane_offset(lane, column_of(j));
    }

    // FOLD, weight gradients: the sums of A's columns are one more block of columns whose B is ones, in the tiles of the first
    // tile column.
    constexpr bool kSums = FOLD && !A_K;
    bool sums = false;
    acc_t column_sums[kSums ? TM : 1];
    frag_t ones;
    // Fragments of the K step being multiplied and of the next one: step s of a K tile is in af[s], bf[s].
    acc_t acc[TM][TN];
    frag_t af[kSteps][TM], bf[kSteps][TN];
    constexpr int kFrags = TM + TN;
    // The F-th fragment in the order of first use (A's block 0, B's blocks, A's other blocks) of K step STEP.
    auto read_frag = [&]<int STEP, int F>(const T* a_tile, const T* b_tile) __attribute__((always_inline)) {
        if constexpr (F >= 1 && F <= TN) {
            constexpr int j = F - 1;
            if constexpr (B_K) bf[STEP][j] = BTile::frag(b_tile, column_of(j), b_off[STEP]);
            else if constexpr (kNarrow && j < 4) bf[STEP][j] = NTile<T, 128>::frag(b_tile + STEP * BTile::kStepElems, b_off[j]);
            else if constexpr (kNarrow) bf[STEP][j] = NTile<T, 64>::frag(b_tile + STEP * BTile::kStepElems, b_off[j]);
            else bf[STEP][j] = BTile::frag(b_tile + STEP * BTile::kStepElems, b_off[j]);
        } else {
            constexpr int i = F == 0 ? 0 : F - TN;
            if constexpr (A_K) af[STEP][i] = ATile::frag(a_tile, wm * WM + i * 16, a_off[STEP]);
            else af[STEP][i] = ATile::frag(a_tile + STEP * ATile::kStepElems, a_off[i]);
        }
    };

    // Epilogue staging. acc[i][j][e] holds C[m, n] with m = lane%16, n = 4*(lane/16) + e, relative
    // to the 16 x 16 block (i, j) of the wavefront's WM x WN part of the tile. Each wavefront passes
    // its part through a private part of A's last LDS slot (the only one the first K tiles of
    // the next item do not fill), 32 rows at a time (16 of an oblong tile), and stores it row by row:
    // whole contiguous row segments of C per instruction instead of 32 separate 8-byte pieces, and no
    // workgroup barrier. When bias, residual or the old C are added (or the output is fp32 / a split-K
    // partial) the staging is fp32, half the columns per pass, and rounding to the storage dtype
    // still happens once, after the additions; otherwise (and on oblong tiles with a bias, which is
    // added there) the values are rounded in registers and staged in the storage dtype. A staged row is kRowBytes long; its 16-byte chunk c sits at
    // chunk position c ^ sw(row), which spreads both the column-wise writes and the row-wise reads
    // over all banks.
    constexpr bool kIsF32 = std::is_same_v<T, float>;
    static_assert(!kIsF32 || (BM <= 128 && !SEGMENTED && !RESIDUAL && !SWIGLU && !GRAD), "fp32 storage has the plain kernels only");
    constexpr int kStaged = kNarrow ? 4 : TN;  // 16-bit blocks of a staged row
    constexpr int kRowBytes = kStaged * 32;    // fp32 values always pass in two halves
    constexpr int kRowChunks = kRowBytes / 16;
    constexpr int kPassRows = kOblong ? 16 : 32;  // 80 and 112 rows of a wavefront are no multiple of 32, and the slot may be smaller
    static_assert(kPassRows * kRowBytes * kWaves <= static_cast<int>(kASlotBytes), "staging fits a slot of A");
    unsigned char* region = smem_raw + (kASlots - 1) * kASlotBytes + wave * (kPassRows * kRowBytes);
    auto sw = [](int row) { return (row / (256 / kRowBytes)) % kRowChunks; };
    const int m_lane = lane & 15, q_lane = lane >> 4;
    // Writes blocks (r, j0 .. j0+JP-1) of kPassRows rows into the wavefront's staging region as element type S.
    constexpr bool kTakesBias = kOblong && A_K && B_K;
    auto stage = [&]<typename S, int JP>(int r, int j0, const auto&... column_bias) __attribute__((always_inline)) {
        static_assert(JP * 16 * sizeof(S) == kRowBytes, "a pass fills whole staged rows");
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int ii = 0; ii < kPassRows / 16; ++ii) {
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
                    float x = acc[r * (kPassRows / 16) + ii][j0 + jj][e];
                    if constexpr (!kIsF32) asm volatile("v_accvgpr_read_b32 %0, %1" : "=v"(x) : "a"(x));
                    v[e] = x;
                }
                ((v += vec_to_f32<T, 4>(column_bias[j0 + jj])), ...);
                const int byte = (jj * 16 + q_lane * 4) * static_cast<int>(sizeof(S));
                unsigned char* slot = write_row + (((byte / 16) ^ sw(row)) * 16) + byte % 16;
                if constexpr (std::is_same_v<S, float>) *reinterpret_cast<vec_t<float, 4>*>(slot) = v;
                else store_vec<T, 4>(reinterpret_cast<T*>(slot), vec_from_f32<T, 4>(v));
            }
        }
        __builtin_amdgcn_wave_barrier();
    };
    // Stages those blocks and hands each lane 8 consecutive staged elements at a time:
    // consume(round, row, col, pointer to the 8 elements' first chunk, to the second chunk when S is
    // float), row/col relative to the wavefront's part; in round u the lane gets element
    // q = 64 u + lane of the kPassRows x (8-element groups per row) grid, row-major.
    auto pass = [&]<typename S, int JP>(int r, int j0, auto&& consume) __attribute__((always_inline)) {
        stage.template operator()<S, JP>(r, j0);
        constexpr int kLanesPerRow = kRowBytes / (8 * static_cast<int>(sizeof(S)));
        constexpr int kChunksPerLane = 8 * static_cast<int>(sizeof(S)) / 16;
        constexpr int kRounds = kPassRows * kLanesPerRow / kWave;
#pragma unroll
        for (int u = 0; u < kRounds; ++u) {
            const int q = u * kWave + lane;
            const int row = q / kLanesPerRow, part = q % kLanesPerRow;
            const unsigned char* base = region + row * kRowBytes;
            const int first = part * kChunksPerLane;
            consume(u, r * kPassRows + row, j0 * 16 + part * 8, base + ((first ^ sw(row)) * 16),
                    base + (((first + kChunksPerLane - 1) ^ sw(row)) * 16));
        }
    };
    constexpr int kRowBlocks = WM / kPassRows;  // passes over a wavefront's rows
    auto request_share = [&](int r) __attribute__((always_inline)) {
        static_for<0, kRowBlocks>([&](auto index) {
            constexpr int block = decltype(index)::value;
            if (r == block)
                request_due.template operator()<Layout::kFirstDue - Layout::kFirstDue * block / kRowBlocks,
                                                Layout::kFirstDue - Layout::kFirstDue * (block + 1) / kRowBlocks>();
        });
    };
    // Before block r of the tile's rows is staged and stored, its share of the first K tiles of the next item
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
        constexpr int kGroups = kStaged, kRowsF = kWave / kGroups, kRoundsF = kPassRows / kRowsF;
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
        if constexpr (kNarrow) {
            // 32 columns at a time through fp32 staging, 8 consecutive ones of row 16u + l/4 to lane l in round u. What is added is
            // requested one pass ahead.
            const int cols_left = min(BN, p.n - w.n0);
            const int c_elem = p.c_f32 ? 4 : static_cast<int>(sizeof(T)), c_row_bytes = static_cast<int>(p.ldc) * c_elem;
            char* const c_origin = static_cast<char*>(p.c) + (static_cast<long>(row0) * p.ldc + w.n0) * c_elem;
            const __amdgpu_buffer_rsrc_t out_rsrc = part_rsrc(c_origin, p.ldc, c_elem, rows_left, cols_left);
            // fp32: the addend, or the old C of an fp32 result; 16 bits: the residual, or the old C of a 16-bit result.
            const bool old_f32 = p.c_f32 && p.accumulate, old_16 = !p.c_f32 && p.accumulate;
            const bool adds_f32 = p.addend != nullptr || old_f32, adds_16 = p.residual != nullptr || old_16;
            const long f32_ld = p.addend != nullptr ? p.ld_addend : p.ldc, ld_16 = p.residual != nullptr ? p.ldr : p.ldc;
            const float* f32_origin = (p.addend != nullptr ? p.addend : static_cast<const float*>(p.c)) + static_cast<long>(row0) * f32_ld + w.n0;
            const T* origin_16 = static_cast<const T*>(p.residual != nullptr ? p.residual : p.c) + static_cast<long>(row0) * ld_16 + w.n0;
            const __amdgpu_buffer_rsrc_t f32_rsrc = part_rsrc(f32_origin, f32_ld, 4, rows_left, cols_left);
            const __amdgpu_buffer_rsrc_t rsrc_16 = part_rsrc(origin_16, ld_16, sizeof(T), rows_left, cols_left);
            const int n_row = lane / 4, n_col = (lane % 4) * 8;
            constexpr int kPasses = kRowBlocks * 3;
            u32x4 ahead_f32[2][2][2], ahead_16[2][2];
            auto column = [&](int q) { return (q % 3 < 2 ? wn * 64 + q % 3 * 32 : 128 + wn * 32) + n_col; };
            auto voffset_of = [&](int q, long ld, int elem) {
                return column(q) < cols_left ? n_row * static_cast<int>(ld) * elem + column(q) * elem : std::numeric_limits<int>::min();
            };
            auto request_added = [&](int q) __attribute__((always_inline)) {
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    const int row = q / 3 * 32 + u * 16;
                    if (adds_f32) {
                        const int voffset = voffset_of(q, f32_ld, 4), soffset = row * static_cast<int>(f32_ld) * 4;
                        ahead_f32[q & 1][u][0] = __builtin_amdgcn_raw_buffer_load_b128(f32_rsrc, voffset, soffset, 0);
                        ahead_f32[q & 1][u][1] = __builtin_amdgcn_raw_buffer_load_b128(f32_rsrc, voffset + 16, soffset, 0);
                    }
                    if (adds_16)
                        ahead_16[q & 1][u] = __builtin_amdgcn_raw_buffer_load_b128(rsrc_16, voffset_of(q, ld_16, sizeof(T)),
                                                                                  row * static_cast<int>(ld_16) * static_cast<int>(sizeof(T)), 0);
                }
            };
            request_added(0);
#pragma unroll
            for (int q = 0; q < kPasses; ++q) {
                __builtin_amdgcn_sched_barrier(0);
                if (q % 3 == 0 && request) request_share(q / 3);
                if (q + 1 < kPasses) request_added(q + 1);
                stage.template operator()<float, 2>(q / 3, q % 3 * 2);
                const int voffset = voffset_of(q, p.ldc, c_elem);
                vec_t<float, 4> v[2][2];
#pragma unroll
                for (int u = 0; u < 2; ++u)
#pragma unroll
                    for (int c = 0; c < 2; ++c) {
                        const int row = u * 16 + n_row;
                        v[u][c] = *reinterpret_cast<const vec_t<float, 4>*>(region + row * kRowBytes + (((n_col / 4 + c) ^ sw(row)) * 16));
                    }
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    if (adds_f32) {
                        v[u][0] += __builtin_bit_cast(acc_t, ahead_f32[q & 1][u][0]);
                        v[u][1] += __builtin_bit_cast(acc_t, ahead_f32[q & 1][u][1]);
                    }
                    vec_t<float, 8> sum;
#pragma unroll
                    for (int e = 0; e < 8; ++e) sum[e] = v[u][e / 4][e % 4];
                    if (adds_16) sum += vec_to_f32<T, 8>(__builtin_bit_cast(vec_t<T, 8>, ahead_16[q & 1][u]));
                    const int soffset = (q / 3 * 32 + u * 16) * c_row_bytes;
                    if (p.c_f32) {
                        store_chunk(__builtin_bit_cast(u32x4, v[u][0]), out_rsrc, voffset, soffset);
                        store_chunk(__builtin_bit_cast(u32x4, v[u][1]), out_rsrc, voffset + 16, soffset);
                    } else {
                        store_chunk(__builtin_bit_cast(u32x4, vec_from_f32<T, 8>(sum)), out_rsrc, voffset, soffset);
                    }
                }
            }
            return;
        }
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
                stage.template operator()<T, kStaged>(r, 0);
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
                stage.template operator()<T, kStaged>(r, 0);
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
        // Of a pair's calls, and on oblong tiles, either the result is stored as it is or a residual is all that is added (C its own).
        if constexpr (RESIDUAL || (FOLD && PLAIN) || kOblong) if (RESIDUAL || p.residual != nullptr) {
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
                        into[half][u] = __builtin_amdgcn_raw_buffer_load_b128(res_rsrc, voffset, (r * kPassRows + u * kRowsF) * res_row_bytes, 0);
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
                    stage.template operator()<float, kStaged / 2>(r, half * (kStaged / 2));
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
                                                               (r * kPassRows + u * kRowsF) * out_row_bytes);
                    }
                }
            }
            return;
        }
        bool plain = PLAIN;
        if constexpr (!PLAIN && !SPLIT && !plain_apart<BM, SPLIT, RESIDUAL, SWIGLU, GRAD>) plain = stored_as_it_is(p);
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
            constexpr int kLanesPerRow = kRowBytes / 16, kRowsPerRound = kWave / kLanesPerRow, kRounds = kPassRows / kRowsPerRound;
            const int lane_row = lane / kLanesPerRow, lane_chunk = lane % kLanesPerRow;
            const int row_bytes = static_cast<int>(c_ld * static_cast<long>(sizeof(T)));
            const int voffset = lane_chunk * 8 < cols_left ? lane_row * row_bytes + lane_chunk * 16 : std::numeric_limits<int>::min();
            if constexpr (kTakesBias) if (p.bias != nullptr) {
                // A lane's accumulators are the same columns in every block of rows: it holds their bias, added before the rounding.
                // Square tiles leave a bias to the general epilogue, which takes no longer (2000 x 1024 x 2048 13.3 us either way).
                // Columns past the matrix are past the buffer's range and get zeros.
                const __amdgpu_buffer_rsrc_t bias_rsrc = part_rsrc(p.bias, 0, sizeof(T), 1, p.n);
                vec_t<T, 4> column_bias[TN];
#pragma unroll
                for (int j = 0; j < TN; ++j)
                    column_bias[j] = __builtin_bit_cast(vec_t<T, 4>, __builtin_amdgcn_raw_buffer_load_b64(
                        bias_rsrc, (w.n0 + col0 + j * 16 + q_lane * 4) * static_cast<int>(sizeof(T)), 0, 0));
#pragma unroll
                for (int r = 0; r < kRowBlocks; ++r) {
                    __builtin_amdgcn_sched_barrier(0);
                    if (request) request_share(r);
                    stage.template operator()<T, kStaged>(r, 0, column_bias);
                    u32x4 data[kRounds];
#pragma unroll
                    for (int u = 0; u < kRounds; ++u) {
                        const int row = u * kRowsPerRound + lane_row;
                        data[u] = *reinterpret_cast<const u32x4*>(region + row * kRowBytes + ((lane_chunk ^ sw(row)) * 16));
                    }
#pragma unroll
                    for (int u = 0; u < kRounds; ++u)
                        store_chunk(data[u], rsrc, voffset, (r * kPassRows + u * kRowsPerRound) * row_bytes);
                }
                return;
            }
#pragma unroll
            for (int r = 0; r < kRowBlocks; ++r) {
                // Accumulators leave their registers block by block: read ahead of their block they
                // would not fit the vector registers.
                __builtin_amdgcn_sched_barrier(0);
                if (request) request_share(r);
                stage.template operator()<T, kStaged>(r, 0);
                u32x4 data[kRounds];
#pragma unroll
                for (int u = 0; u < kRounds; ++u) {
                    const int row = u * kRowsPerRound + lane_row;
                    data[u] = *reinterpret_cast<const u32x4*>(region + row * kRowBytes + ((lane_chunk ^ sw(row)) * 16));
                }
#pragma unroll
                for (int u = 0; u < kRounds; ++u)
                    store_chunk(data[u], rsrc, voffset, (r * kPassRows + u * kRowsPerRound) * row_bytes);
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
                    stage.template operator()<float, kStaged / 2>(r, half * (kStaged / 2));
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
            constexpr int kCols = kStaged * 8, kRowsE = kWave / kCols;
            const int e_row = lane / kCols, e_col = lane % kCols;
#pragma unroll
            for (int r = 0; r < kRowBlocks; ++r) {
                __builtin_amdgcn_sched_barrier(0);
                if (request) request_share(r);
#pragma unroll
                for (int half = 0; half < 2; ++half) {
                    stage.template operator()<float, kStaged / 2>(r, half * (kStaged / 2));
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
                pass.template operator()<float, kStaged / 2>(r, half * (kStaged / 2), [&](int, int row, int col, const unsigned char* lo,
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
    //   first step   MFMAs ‖ LDS reads of this tile's second-step fragments ‖ the loads of A's K tile t-1+kASlots (into the
    //                slot of A's K tile t-1)
    //   wait         this wavefront's loads of K tile t+1 have landed and its reads of K tile t are through; barrier:
    //                everybody's have, so K tile t's slots are free
    //   second step  MFMAs ‖ LDS reads of K tile t+1's first-step fragments ‖ the loads of B's K tile t+kBSlots (into the
    //                slot of B's K tile t)
    // so LDS latency and one to one and a half K tiles of global latency sit in the shadow of MFMAs, and the workgroup
    // meets once per K tile. With one wavefront per SIMD nothing else hides an instruction that is not next to an MFMA, so
    // every MFMA is followed by its share of the loads and fragment reads and a scheduling fence keeps them there. A
    // wavefront's load instruction keeps it from issuing for about as long as an MFMA runs.
    constexpr int kMfmas = TM * TN;
    constexpr int kReadEvery = kMfmas / kFrags >= 3 ? 3 : 1;  // MFMAs between fragment reads
    static_assert(kReadEvery * kFrags <= kMfmas && kALoads <= kMfmas && kBLoads <= kMfmas, "a step has room for its reads and loads");
    // STEP 0: a_tile, b_tile are K tile t's; STEP 1: K tile t+1's. slot_lds: where the step's loads go.
    auto multiply_step = [&]<int STEP, bool FIRST>(int t, const T* a_tile, const T* b_tile, unsigned int slot_lds) __attribute__((always_inline)) {
        static_for<0, kMfmas>([&](auto index) {
            constexpr int m = decltype(index)::value;
            // Rows one after the other, their columns left to right and right to left alternately:
            // consecutive MFMAs always share an operand (measurably less power on a power-limited chip).
            constexpr int i = m / TN, jj = m % TN, j = (i & 1) ? TN - 1 - jj : jj;
            if constexpr (FIRST && STEP == 0) Mfma<T>::start(acc[i][j], bf[STEP][j], af[STEP][i]);
            else Mfma<T>::run(acc[i][j], bf[STEP][j], af[STEP][i]);
            if constexpr (m % kReadEvery == 0 && m / kReadEvery < kFrags)
                read_frag.template operator()<1 - STEP, m / kReadEvery>(a_tile, b_tile);
            constexpr int kLoads = STEP == 0 ? kALoads : kBLoads;
            static_for<(m * kLoads) / kMfmas, ((m + 1) * kLoads) / kMfmas>([&](auto l) {
                if constexpr (STEP == 0) issue_a(l, slot_lds, ca);
                else issue_b(l, slot_lds, cb);
            });
            // The next step's cursor, where its scalar arithmetic has MFMAs around it.
            if constexpr (m == kMfmas / 2) {
                if constexpr (STEP == 0) aim_b(t + kBSlots, cb);
                else aim_a(t + kASlots, ca);
            }
            __builtin_amdgcn_sched_barrier(0);
        });
        if constexpr (kSums) {
            if (sums) {
#pragma unroll
                for (int i = 0; i < TM; ++i) Mfma<T>::add(column_sums[i], ones, af[STEP][i]);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    };
    auto next_slot = []<int SLOTS>(int slot) __attribute__((always_inline)) { return slot + 1 == SLOTS ? 0 : slot + 1; };

    // Per round: multiply an item, request the first K tiles of the next one, store the finished
    // tile (its stores drain under the MFMAs that follow). The sources are opened every round, also
    // when no item is left (then for the last one again, unused): values that are set on every path
    // stay in scalar registers.
    Item current = locate(item);
    open(current);
    if constexpr (kSums) {
        sums = p.a_sums != nullptr && current.n0 == 0 && wn == 0;
#pragma unroll
        for (int i = 0; i < TM; ++i) column_sums[i] = acc_t(0.0f);
#pragma unroll
        for (int e = 0; e < static_cast<int>(sizeof(frag_t) / sizeof(T)); ++e) ones[e] = static_cast<T>(1.0f);
    }
    request_due.template operator()<Layout::kFirstDue, 0>();
    while (true) {
        const int steps = current.kt_end - current.kt_begin;
        // Loads and stores retire in the order they were issued: at most the requests after those of K tile 0
        // (and no older store of the previous epilogue) may still be outstanding.
        __builtin_amdgcn_s_waitcnt(vmcnt_immediate(Layout::outstanding(0, 0)));
        barrier_only();
        static_for<0, kFrags>([&](auto f) { read_frag.template operator()<0, decltype(f)::value>(smem, smem + kBBase); });
        aim_a(kASlots - 1, ca);
        int a_slot = 0, b_slot = 0;  // of K tile t
        auto first_step = [&]<bool FIRST>(int t) __attribute__((always_inline)) {
            const int freed = a_slot == 0 ? kASlots - 1 : a_slot - 1;
            multiply_step.template operator()<0, FIRST>(t, smem + a_slot * ATile::kElems, smem + kBBase + b_slot * BTile::kElems,
                                                        a_lds + freed * kASlotBytes);
        };
        auto second_step = [&](int t) __attribute__((always_inline)) {
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            __builtin_amdgcn_s_waitcnt(vmcnt_immediate(Layout::outstanding(1, 1)));
            barrier_only();
            const int a_next = next_slot.template operator()<kASlots>(a_slot), b_next = next_slot.template operator()<kBSlots>(b_slot);
            multiply_step.template operator()<1, false>(t, smem + a_next * ATile::kElems, smem + kBBase + b_next * BTile::kElems,
                                                        b_lds + b_slot * kBSlotBytes);
            a_slot = a_next;
            b_slot = b_next;
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
        if constexpr (FOLD) {
            const int first_row = current.m0 + wm * WM + lane;  // of A's columns whose sums this lane stores, 16 apart
            const bool last = p.slices == 1 || fold_slices<T, TM, TN, kSums>(p, acc, column_sums, sums, current.slice, tiles,
                                                                             current.m0 / BM * p.tiles_n + current.n0 / BN, wm, smem_raw);
            if (!last) return;
            if constexpr (kSums) {
                if (sums && lane < 16) {
#pragma unroll
                    for (int i = 0; i < TM; ++i) {
                        if (first_row + i * 16 >= p.m) continue;
                        T* out = static_cast<T*>(p.a_sums) + first_row + i * 16;
                        *out = from_f32<T>(p.a_sums_accumulate ? column_sums[i][0] + to_f32(*out) : column_sums[i][0]);
                    }
                }
            }
            store_tile(current, false);
            return;
        }
        item += item_stride;
        const bool more = item < item_end;
        const Item next = locate(more ? item : item_end - 1);
        open(next);
        store_tile(current, more);
        if (!more) break;
        current = next;
    }
}

template <typename T, int BM, int BN, bool A_K, bool B_K, bool SPLIT, bool SEGMENTED, bool RESIDUAL = false,
          bool SWIGLU = false, bool GRAD = false, bool DEEP = false, bool PLAIN = false>
__global__ __launch_bounds__(kThreads) void gemm_mfma_kernel(KernelArgs p) {
    extern __shared__ __align__(1024) unsigned char smem_raw[];
    // Work items are numbered slice-major (all tiles of K slice 0, then of slice 1, ...), tiles in
    // groups of 1 << group_rows_log2 tile-rows, down the rows first. Blocks are dealt round-robin to the 8
    // XCDs, so XCD x takes the x-th eighth of the items and its blocks walk it side by side: the
    // items in flight on one XCD are neighbours and share A and B panels in that XCD's L2.
    const int items = p.tiles_m * p.tiles_n * p.slices;
    const int per_xcd = (items + kXcds - 1) / kXcds;
    const int item_end = min(items, static_cast<int>(blockIdx.x % kXcds + 1) * per_xcd);
    const int item = static_cast<int>(blockIdx.x % kXcds) * per_xcd + static_cast<int>(blockIdx.x / kXcds);
    if (item >= item_end) return;
    contract<T, BM, BN, A_K, B_K, SPLIT, SEGMENTED, RESIDUAL, SWIGLU, GRAD, DEEP, PLAIN, false>(p, item, item_end, gridDim.x / kXcds, smem_raw);
}

// Both gradients of a projection on 128 x 128 tiles in one launch, a workgroup per tile and K slice, the longer ones first. Either
// gradient by itself leaves CUs idle (a weight gradient of 1024 x 1024 has 64 tiles, an input gradient of 5005 x 1024 320 for 256
// CUs) and pays a launch, a pipeline fill and an epilogue of its own; a weight gradient split along K paid one more launch for its
// partial tiles. Not persistent: the dispatcher deals the workgroups out to the two slots of a CU as they become free, and one's
// epilogue runs beside the other's K loop. What bounds it is the path from the L2s (0.22 - 0.24 us per K step and CU), and with few
// rounds the last one. Inputs from memory, bf16, us before and now: 2000 x 1024 x 2048 with bias, added to old gradients 32 -> 24
// (on 64 x 64 tiles before); a block of 5 x 1001 tokens, 1024 wide, forward and backward 752 -> 699.
template <typename T, bool DEEP, bool PLAIN>
__global__ __launch_bounds__(kThreads, DEEP ? 1 : 2) void gemm_pair_kernel(PairArgs pair) {
    extern __shared__ __align__(1024) unsigned char smem_raw[];
    const int block = blockIdx.x;
    const bool weight = (block < pair.first_blocks) == (pair.weight_first != 0);
    const int local = block < pair.first_blocks ? block : block - pair.first_blocks;
    auto item_of = [&](const KernelArgs& p) __attribute__((always_inline)) {
        const int items = p.tiles_m * p.tiles_n * p.slices, per_xcd = (items + kXcds - 1) / kXcds;
        const int within = local / kXcds, item = local % kXcds * per_xcd + within;
        return within < per_xcd && item < items ? item : -1;
    };
    if (weight) {
        const int item = item_of(pair.weight);
        if (item < 0) return;
        contract<T, 128, 128, false, false, false, false, false, false, false, DEEP, PLAIN, true>(pair.weight, item, item + 1, 1, smem_raw);
    } else {
        const int item = item_of(pair.input);
        if (item < 0) return;
        contract<T, 128, 128, true, false, false, false, false, false, false, DEEP, PLAIN, true>(pair.input, item, item + 1, 1, smem_raw);
    }
}

// The same with tiles of 256 x 128 of the weight gradient and oblong ones of the input gradient, one workgroup per CU and one round of
// them: 40 per cent less operand traffic per product than 128 x 128 tiles, which the path from the L2s binds. 5005 x 1024 x 2048 is 92 tiles of 224 x 256
// and 64 of 256 x 128 in two slices, 220 workgroups: 50.5 -> 46.2 us.
template <typename T, int BM, int BN>
__global__ __launch_bounds__(kThreads, 1) void gemm_oblong_pair_kernel(PairArgs pair) {
    extern __shared__ __align__(1024) unsigned char smem_raw[];
    const int block = blockIdx.x;
    const bool weight = (block < pair.first_blocks) == (pair.weight_first != 0);
    const int local = block < pair.first_blocks ? block : block - pair.first_blocks;
    auto item_of = [&](const KernelArgs& p) __attribute__((always_inline)) {
        const int items = p.tiles_m * p.tiles_n * p.slices, per_xcd = (items + kXcds - 1) / kXcds;
        const int within = local / kXcds, item = local % kXcds * per_xcd + within;
        return within < per_xcd && item < items ? item : -1;
    };
    if (weight) {
        const int item = item_of(pair.weight);
        if (item < 0) return;
        contract<T, kPairWeightRows, kPairWeightColumns, false, false, false, false, false, false, false, false, true, true>(pair.weight, item, item + 1, 1, smem_raw);
    } else {
        const int item = item_of(pair.input);
        if (item < 0) return;
        contract<T, BM, BN, true, false, false, false, false, false, false, false, true, true>(pair.input, item, item + 1, 1, smem_raw);
    }
}

// ------------------------------------------------------------------- host side
constexpr int blocks_per_unit(std::size_t smem) { return smem * 2 <= kLdsBytes ? 2 : 1; }  // resident blocks per CU: what the LDS slots allow

// Groups of 1 << rows_log2 tile-rows, and what divides by their size.
inline void set_groups(KernelArgs& p, int rows_log2) {
    p.group_rows_log2 = rows_log2;
    // x * ceil(2^32 / d) >> 32 == x / d for every x with x * d < 2^32.
    const unsigned long divisor = (1ul << rows_log2) * static_cast<unsigned long>(p.tiles_n);
    const unsigned long tiles = static_cast<unsigned long>(p.tiles_m) * static_cast<unsigned long>(p.tiles_n);
    const bool exact = divisor > 1 && tiles * divisor < (1ul << 32);
    p.group_reciprocal = exact ? static_cast<unsigned int>(((1ul << 32) + divisor - 1) / divisor) : 0u;
}

template <typename T, int BM, int BN, bool A_K, bool B_K, bool SPLIT, bool SEGMENTED, bool RESIDUAL, bool SWIGLU, bool GRAD,
          bool DEEP, bool PLAIN>
int launch_kernel(const KernelArgs& p, int slices, hipStream_t stream) {
    const long items = static_cast<long>(p.tiles_m) * p.tiles_n * slices;
    constexpr std::size_t smem = TileLayout<T, BM, BN, A_K, B_K, DEEP>::kSmemBytes;
    auto kernel = gemm_mfma_kernel<T, BM, BN, A_K, B_K, SPLIT, SEGMENTED, RESIDUAL, SWIGLU, GRAD, DEEP, PLAIN>;
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
    // Tile-rows per L2 locality group. 8 (x 4 tile-columns = the 32 tiles in flight on an XCD) shares operand
    // panels best. The SwiGLU-gradient epilogue moves four times the bytes of a plain one, two loads and two
    // stores of whole [gate | up] rows: there the tiles in flight on an XCD are better spread along the rows
    // (2 tile-rows x all 8 tile-columns of the training shape: 250 -> 212 us per launch; 1, 2 and 4 tile-rows
    // measure the same, every other kernel is at its best with 8).
    set_groups(args, GRAD ? 1 : 3);
    const long slots = static_cast<long>(compute_units()) * blocks_per_unit(smem) / kXcds * kXcds;
    const long blocks = std::min<long>((items + kXcds - 1) / kXcds * kXcds, std::max<long>(slots, kXcds));
    hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned int>(blocks)), dim3(kThreads), smem, stream, args);
    CGPTX_LAUNCH_CHECK();
    return CGPTX_OK;
}

template <typename T, int BM, int BN, bool A_K, bool B_K, bool SPLIT, bool SEGMENTED, bool RESIDUAL = false,
          bool SWIGLU = false, bool GRAD = false>
int launch_mfma(const KernelArgs& p, int slices, hipStream_t stream) {
    auto with_depth = [&]<bool DEEP>() -> int {
        if constexpr (plain_apart<BM, SPLIT, RESIDUAL, SWIGLU, GRAD>) {
            if (stored_as_it_is(p))
                return launch_kernel<T, BM, BN, A_K, B_K, SPLIT, SEGMENTED, RESIDUAL, SWIGLU, GRAD, DEEP, true>(p, slices, stream);
            if constexpr (SEGMENTED) return fail(CGPTX_RUNTIME, "gemm: an operand in segments along K takes nothing added to its product");
        }
        if constexpr (!(SEGMENTED && BM == 128))
            return launch_kernel<T, BM, BN, A_K, B_K, SPLIT, SEGMENTED, RESIDUAL, SWIGLU, GRAD, DEEP, false>(p, slices, stream);
    };
    if constexpr (BM == 128) {
        if (static_cast<long>(p.tiles_m) * p.tiles_n * slices <= compute_units()) return with_depth.template operator()<true>();
    }
    return with_depth.template operator()<false>();
}

template <typename T, int BM, int BN, bool SPLIT>
int launch_layout(const KernelArgs& p, bool a_k, bool b_k, int slices, hipStream_t stream) {
    // A given in segments along K has kernels of its own (the source of a K tile is then picked
    // per tile), and only unsplit ones of input gradients.
    const bool segmented = a_k && p.a_seg.count > 0;
    if constexpr (!SPLIT && !std::is_same_v<T, float>) {
        if (segmented && !b_k) return launch_mfma<T, BM, BN, true, false, false, true>(p, slices, stream);
    }
    if (segmented) return fail(CGPTX_RUNTIME, "gemm: an operand in segments along K is that of an unsplit input gradient");
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

// 256 x 192 tiles (call.tile 192): for results whose columns are not near a multiple of 256, or whose 256 x 256 tiles leave part of the
// last round of CUs idle. 768 columns are three tiles of 256, 192 of them for 16384 rows, and four of 192, 256 of them. Same sums in
// the same order. The K loop is 0.77 of a 256 x 256 tile's (48 MFMAs a step for 64, 56 KiB of operands a K tile for 64); that a
// filled chip runs at a lower clock than one of which a quarter idles takes most of the rest. us, 256 and 192 columns: 16384 x 768 x
// 32000 626 -> 587, 32000 x 768 x 16384 (weight gradient) 661 -> 630, 32768 x 768 x 4096 172 -> 159, 32768 x 768 x 2048 91 -> 85;
// 32768 x 768 x 768 46 -> 44 (128 x 128: 41.5), 32768 x 960 x 960 56 -> 70. The step of 8 x 4096 tokens, 768 wide, 10294 -> 10002.
template <typename T>
int launch_narrow(const LargeCall& call, hipStream_t stream) {
    const KernelArgs& p = call.args;
    const bool a_k = call.a_k_contiguous, b_k = call.b_k_contiguous;
    if (call.split || p.bias != nullptr || p.ragged || p.act != nullptr || p.saved != nullptr || p.c_seg.count > 0 || p.batch_rows > 0)
        return fail(CGPTX_RUNTIME, "gemm: 256 x 192 tiles take plain products");
    if (a_k && p.a_seg.count > 0) {
        if (b_k) return fail(CGPTX_RUNTIME, "gemm: an operand in segments along K is that of an input gradient");
        return launch_kernel<T, 256, 192, true, false, false, true, false, false, false, false, false>(p, 1, stream);
    }
    if (a_k && b_k) return launch_kernel<T, 256, 192, true, true, false, false, false, false, false, false, false>(p, 1, stream);
    if (a_k) return launch_kernel<T, 256, 192, true, false, false, false, false, false, false, false, false>(p, 1, stream);
    if (!b_k) return launch_kernel<T, 256, 192, false, false, false, false, false, false, false, false, false>(p, 1, stream);
    return fail(CGPTX_RUNTIME, "gemm: unsupported operand layout");
}

// Oblong tiles, one block per CU: 160, 192 or 256 rows of 128 columns, 160, 192 or 224 of 256. A few thousand rows are 1.2 or 2.3
// rounds of square tiles: 5005 x 1024 is 320 tiles of 128 x 128, of which 64 CUs get two, or 80 of 256 x 256. A tile of 160 x 128 is
// one round. A call of one round costs 6 to 9 us that are no K loop (launch, first loads, store) and then what the L2s deliver
// (128 columns: 0.25 us a K step, 1.34 PFLOP/s over a full chip) or the matrix cores at the power limit (160 x 256: 0.44 us, 1.5 PFLOP/s). Same
// sums in the same order as square tiles. Block of 5 x 1001 tokens, 1024 wide, forward and backward 695 -> 671 us; with a bias 5005 x 2048 x 1024
// 30.6 -> 23.1, 10000 x 1024 x 1024 30.8 -> 22.7, 16384 x 768 x 768 31.2 -> 22.3.
template <typename T, int BM, int BN>
int launch_oblong_tile(const LargeCall& call, hipStream_t stream) {
    KernelArgs p = call.args;
    const bool a_k = call.a_k_contiguous, b_k = call.b_k_contiguous;
    if (p.accumulate && p.residual == nullptr) {  // C as its own residual, see launch_layout
        p.residual = p.c;
        p.ldr = p.ldc;
        p.accumulate = 0;
    }
    if (call.split || !a_k || (p.bias != nullptr && (!b_k || p.residual != nullptr)) || p.addend != nullptr || p.accumulate || p.c_f32 ||
        p.ragged || p.act != nullptr || p.saved != nullptr || p.batch_rows > 0 || (p.residual != nullptr && p.c_seg.count > 0) || (p.a_seg.count > 0 && b_k))
        return fail(CGPTX_RUNTIME, "gemm: oblong tiles take products that are stored as they are, with a bias or with a residual");
    if (p.a_seg.count > 0) return launch_kernel<T, BM, BN, true, false, false, true, false, false, false, false, true>(p, 1, stream);
    if (b_k) return launch_kernel<T, BM, BN, true, true, false, false, false, false, false, false, true>(p, 1, stream);
    return launch_kernel<T, BM, BN, true, false, false, false, false, false, false, false, true>(p, 1, stream);
}

template <typename T, bool DEEP, bool PLAIN>
int launch_pair_kernel(const PairArgs& pair, int blocks, hipStream_t stream) {
    constexpr int smem = std::max(TileLayout<T, 128, 128, true, false, DEEP>::kSmemBytes, TileLayout<T, 128, 128, false, false, DEEP>::kSmemBytes);
    auto kernel = gemm_pair_kernel<T, DEEP, PLAIN>;
    static const hipError_t status =
        hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, smem);
    CGPTX_HIP(status);
    hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned int>(blocks)), dim3(kThreads), smem, stream, pair);
    CGPTX_LAUNCH_CHECK();
    return CGPTX_OK;
}

// Tile groups, workgroups and which call goes first; C += A·B in the storage dtype becomes C as its own residual, see launch_layout.
inline int prepare_pair(PairArgs& pair, int* total) {
    long items[2];
    int blocks[2], i = 0;
    for (KernelArgs* p : {&pair.input, &pair.weight}) {
        set_groups(*p, 3);
        items[i] = static_cast<long>(p->tiles_m) * p->tiles_n * p->slices;
        if (items[i] > std::numeric_limits<int>::max() / 4) return fail(CGPTX_OVERFLOW, "gemm: too many tiles");
        blocks[i] = static_cast<int>((items[i] + kXcds - 1) / kXcds * kXcds);
        ++i;
    }
    if (!pair.input.ragged && !pair.weight.ragged) {
        for (KernelArgs* p : {&pair.input, &pair.weight}) {
            if (!p->accumulate) continue;
            p->residual = p->c;
            p->ldr = p->ldc;
            p->accumulate = 0;
        }
    }
    pair.weight_first = pair.weight.k_tiles_per_slice >= pair.input.k_tiles_per_slice ? 1 : 0;
    pair.first_blocks = blocks[pair.weight_first];
    *total = blocks[0] + blocks[1];
    return CGPTX_OK;
}

template <typename T>
int launch_pair(const PairArgs& pair_in, hipStream_t stream) {
    PairArgs pair = pair_in;
    int total = 0;
    if (int s = prepare_pair(pair, &total)) return s;
    const bool plain = !pair.input.ragged && !pair.weight.ragged;
    const long items = static_cast<long>(pair.input.tiles_m) * pair.input.tiles_n * pair.input.slices +
                       static_cast<long>(pair.weight.tiles_m) * pair.weight.tiles_n * pair.weight.slices;
    const bool deep = items <= compute_units();
    if (deep) return plain ? launch_pair_kernel<T, true, true>(pair, total, stream) : launch_pair_kernel<T, true, false>(pair, total, stream);
    return plain ? launch_pair_kernel<T, false, true>(pair, total, stream) : launch_pair_kernel<T, false, false>(pair, total, stream);
}

template <typename T, int BM, int BN>
int launch_oblong_pair_tile(const PairArgs& pair, int blocks, hipStream_t stream) {
    constexpr int smem = std::max(TileLayout<T, BM, BN, true, false, false>::kSmemBytes,
                                  TileLayout<T, kPairWeightRows, kPairWeightColumns, false, false, false>::kSmemBytes);
    auto kernel = gemm_oblong_pair_kernel<T, BM, BN>;
    static const hipError_t status =
        hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, smem);
    CGPTX_HIP(status);
    hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned int>(blocks)), dim3(kThreads), smem, stream, pair);
    CGPTX_LAUNCH_CHECK();
    return CGPTX_OK;
}

// pair_in.input_tile names the input gradient's tile. Nothing ragged.
template <typename T>
int launch_oblong_pair(const PairArgs& pair_in, hipStream_t stream) {
    PairArgs pair = pair_in;
    int blocks = 0;
    if (int s = prepare_pair(pair, &blocks)) return s;
    if (pair.input.ragged || pair.weight.ragged) return fail(CGPTX_RUNTIME, "gemm: oblong tiles store whole chunks");
    switch (pair.input_tile) {
        case oblong_tile(160, 128): return launch_oblong_pair_tile<T, 160, 128>(pair, blocks, stream);
        case oblong_tile(192, 128): return launch_oblong_pair_tile<T, 192, 128>(pair, blocks, stream);
        case oblong_tile(256, 128): return launch_oblong_pair_tile<T, 256, 128>(pair, blocks, stream);
        case oblong_tile(160, 256): return launch_oblong_pair_tile<T, 160, 256>(pair, blocks, stream);
        case oblong_tile(192, 256): return launch_oblong_pair_tile<T, 192, 256>(pair, blocks, stream);
        case oblong_tile(224, 256): return launch_oblong_pair_tile<T, 224, 256>(pair, blocks, stream);
    }
    return fail(CGPTX_RUNTIME, "gemm: no pair of tiles of this size");
}

template <typename T>
int launch_large(const LargeCall& call, hipStream_t stream) {
    auto with_tile = [&]<int TILE>() -> int {
        return call.split ? launch_layout<T, TILE, TILE, true>(call.args, call.a_k_contiguous, call.b_k_contiguous, call.slices, stream)
                          : launch_layout<T, TILE, TILE, false>(call.args, call.a_k_contiguous, call.b_k_contiguous, call.slices, stream);
    };
    if constexpr (!std::is_same_v<T, float>) {
        if (call.tile == 256) return with_tile.template operator()<256>();
        if (call.tile == 192) return launch_narrow<T>(call, stream);
    }
    if (call.tile != 128) return fail(CGPTX_RUNTIME, "gemm: no large tiles of this size for the storage type");
    return with_tile.template operator()<128>();
}

template <typename T>
int launch_oblong(const LargeCall& call, hipStream_t stream) {
    if (call.tile == oblong_tile(160, 128)) return launch_oblong_tile<T, 160, 128>(call, stream);
    if (call.tile == oblong_tile(192, 128)) return launch_oblong_tile<T, 192, 128>(call, stream);
    if (call.tile == oblong_tile(256, 128)) return launch_oblong_tile<T, 256, 128>(call, stream);
    if (call.tile == oblong_tile(160, 256)) return launch_oblong_tile<T, 160, 256>(call, stream);
    if (call.tile == oblong_tile(192, 256)) return launch_oblong_tile<T, 192, 256>(call, stream);
    if (call.tile == oblong_tile(224, 256)) return launch_oblong_tile<T, 224, 256>(call, stream);
    return fail(CGPTX_RUNTIME, "gemm: no oblong tiles of this size");
}

}  // namespace
}  // namespace cgptx
