// Small contractions: K split between the wavefronts of a workgroup.
//
// C of at most a few hundred tiles (short sequences, narrow layers, the weight gradients of a small batch) leaves the
// persistent kernels with little to do per K tile and a workgroup barrier around each: what such a call costs
// is the latency of its start and of its serial K loop. Here a workgroup owns one 64 x 64 or 32 x 32 tile and its four
// wavefronts take every fourth K tile each, the whole C tile of it: the loop is four times shorter and has no barrier,
// since a wavefront loads its K tiles into LDS stages of its own (global -> LDS) and waits for nobody. A K tile is two MFMA
// steps long, whole cache lines of a k-contiguous operand (see KTile); the fragments of the step to come are read, and the
// loads of the K tile to come are issued, between the MFMAs of the present step. At the end
// the four partial tiles meet in LDS and are added in wavefront order. Same swizzled operand tiles and same edges (buffer
// range checks) as the persistent kernels.
//
// What bounds it: with few workgroups the latency of the loads, i.e. the K bytes of a workgroup over the bytes it keeps
// in flight (64 or 128 KiB), which is why short rows of tiles take 32 x 32 ones; with a full chip the path from the L2s
// (8 KiB per 64 x 64 tile and step: 0.128 us in half cache lines, 0.09 in whole ones), where larger tiles win.
#pragma once

#include "gemm_small.hpp"
#include "gemm_tiles.hpp"

namespace cgptx {
namespace {

template <int COUNT>
__device__ __forceinline__ void wait_loads() {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(COUNT) : "memory");
}

// One of three values, all of them read first: a choice between places would keep the arguments in memory.
template <typename V>
__device__ __forceinline__ V one_of(bool in1, bool in2, V v0, V v1, V v2) { return in2 ? v2 : in1 ? v1 : v0; }

__device__ __forceinline__ SegmentPick pick_small_segment(const SmallSegments& seg, int col) {
    const int cols0 = seg.cols[0], cols1 = seg.cols[1], cols2 = seg.cols[2], end0 = cols0, end1 = end0 + cols1;
    const bool in1 = seg.count > 1 && col >= end0, in2 = seg.count > 2 && col >= end1;
    SegmentPick pick;
    pick.ptr = one_of(in1, in2, seg.ptr[0], seg.ptr[1], seg.ptr[2]);
    pick.ld = one_of(in1, in2, seg.ld[0], seg.ld[1], seg.ld[2]);
    pick.first = one_of(in1, in2, 0, end0, end1);
    pick.cols = one_of(in1, in2, cols0, cols1, cols2);
    pick.index = one_of(in1, in2, 0, 1, 2);
    return pick;
}

template <int TILE, bool DEEP>
constexpr int small_smem_bytes() { return DEEP ? 128 * 1024 : 64 * 1024; }

// The tile at (m0, n0) of one call. SUMS: sums of A's columns beside it, by the workgroups of the first tile column.
template <typename T, int TILE, bool DEEP, bool A_K, bool B_K, SmallEpilogue EPILOGUE, bool SEGMENTED, bool SUMS>
__device__ __forceinline__ void small_tile(const SmallArgs& p, int m0, int n0, int slice, unsigned char* smem_raw) {
    using frag_t = typename Mfma<T>::frag;
    using ATile = std::conditional_t<A_K, KTile<T, TILE>, NTile<T, TILE>>;
    using BTile = std::conditional_t<B_K, KTile<T, TILE>, NTile<T, TILE>>;
    constexpr int kBlocks = TILE / 16;                  // 16 x 16 MFMA blocks along an edge
    constexpr int kOperandBytes = TILE * 64 * kSteps;   // 128 bytes along K per row, or the same bytes k-strided
    constexpr int kStageBytes = 2 * kOperandBytes;      // [A | B]
    constexpr int kLoadBytes = 1024, kOperandLoads = kOperandBytes / kLoadBytes, kLoads = 2 * kOperandLoads;
    constexpr int STAGES = small_smem_bytes<TILE, DEEP>() / (kWaves * kStageBytes);
    static_assert(STAGES >= 1 && STAGES * kLoads < 64, "the loads in flight are counted by vmcnt");
    static_assert(!SUMS || !A_K, "columns of A are summed where its rows are K positions");
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);

    const int kt_begin = slice * p.k_tiles_per_slice, kt_end = min(p.k_tiles, kt_begin + p.k_tiles_per_slice);
    // This wavefront's K tiles: steps kt_begin + kSteps (wave + kWaves i) and the one after it, which the last may lack.
    const int tiles = max(0, ((kt_end - kt_begin + kSteps - 1) / kSteps - wave + kWaves - 1) / kWaves);
    const bool whole_last = kt_begin + kSteps * (wave + kWaves * (tiles - 1)) + 1 < kt_end;

    // Sources. A in column segments: along K (k-contiguous) the segment is picked per K tile, along M once.
    ATile a_src;
    BTile b_src;
    // In segments along K all three are set up (absent ones repeat the first and are never picked), and a K tile's is
    // picked field by field: selecting an object would keep all of them in memory.
    ATile a_src1, a_src2;
    int a_end0 = std::numeric_limits<int>::max(), a_end1 = std::numeric_limits<int>::max();
    if constexpr (A_K && SEGMENTED) {
        const int count = p.a_seg.count;
        const void* base0 = one_of(count == 0, false, p.a_seg.ptr[0], p.a, p.a);
        const long ld0 = one_of(count == 0, false, p.a_seg.ld[0], p.lda, p.lda);
        const int cols0 = one_of(count == 0, false, p.a_seg.cols[0], p.k, p.k), rows = p.m - m0;
        auto segment = [&](ATile& source, const void* base, long ld, int cols) __attribute__((always_inline)) {
            source.init(static_cast<const T*>(base) + static_cast<long>(m0) * ld, ld, rows, cols, 0);
        };
        segment(a_src, base0, ld0, cols0);
        segment(a_src1, one_of(count > 1, false, base0, p.a_seg.ptr[1], base0), one_of(count > 1, false, ld0, p.a_seg.ld[1], ld0),
                one_of(count > 1, false, cols0, p.a_seg.cols[1], cols0));
        segment(a_src2, one_of(count > 2, false, base0, p.a_seg.ptr[2], base0), one_of(count > 2, false, ld0, p.a_seg.ld[2], ld0),
                one_of(count > 2, false, cols0, p.a_seg.cols[2], cols0));
        if (count > 1) a_end0 = cols0;
        if (count > 2) a_end1 = cols0 + p.a_seg.cols[1];
    } else if constexpr (A_K) {
        a_src.init(static_cast<const T*>(p.a) + static_cast<long>(m0) * p.lda, p.lda, p.a_extent - m0, p.k, 0);
    } else {
        const T* base = static_cast<const T*>(p.a) + m0;
        long ld = p.lda;
        int width = p.a_extent - m0;
        if constexpr (SEGMENTED) {
            if (p.a_seg.count > 0) {
                const SegmentPick pick = pick_small_segment(p.a_seg, m0);
                base = static_cast<const T*>(pick.ptr) + (m0 - pick.first);
                ld = pick.ld;
                width = pick.cols - (m0 - pick.first);
            }
        }
        a_src.init(base, ld, width, p.k, 0);
    }
    if constexpr (B_K) b_src.init(static_cast<const T*>(p.b) + static_cast<long>(n0) * p.ldb, p.ldb, p.b_extent - n0, p.b_k, 0);
    else b_src.init(static_cast<const T*>(p.b) + n0, p.ldb, p.b_extent - n0, p.b_k, 0);

    const unsigned int lds_wave = lds_address_of(smem_raw) + wave * (STAGES * kStageBytes);
    const T* const wave_stages = reinterpret_cast<const T*>(smem_raw + wave * (STAGES * kStageBytes));
    constexpr int kStageElems = kStageBytes / static_cast<int>(sizeof(T)), kOperandElems = kStageElems / 2;
    unsigned int a_soffset = 0, b_soffset = 0;
    u32x4 a_rsrc = a_src.rsrc;
    int a_voffset = a_src.voffset, a_voffset_odd = a_src.load_voffset(1);
    unsigned int a_step = a_src.group_bytes;
    auto aim = [&](int i) __attribute__((always_inline)) {
        const int k0 = (kt_begin + kSteps * (wave + kWaves * i)) * kBK<T>;
        if constexpr (A_K && SEGMENTED) {
            const bool in1 = k0 >= a_end0, in2 = k0 >= a_end1;
            const u32x4 rsrc0 = a_src.rsrc, rsrc1 = a_src1.rsrc, rsrc2 = a_src2.rsrc;
            const int voffset0 = a_src.voffset, voffset1 = a_src1.voffset, voffset2 = a_src2.voffset;
            const int odd0 = a_src.load_voffset(1), odd1 = a_src1.load_voffset(1), odd2 = a_src2.load_voffset(1);
            const unsigned int bytes0 = a_src.group_bytes, bytes1 = a_src1.group_bytes, bytes2 = a_src2.group_bytes;
            const int end0 = a_end0, end1 = a_end1;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const unsigned int w0 = rsrc0[e], w1 = rsrc1[e], w2 = rsrc2[e];
                a_rsrc[e] = in2 ? w2 : in1 ? w1 : w0;
            }
            a_voffset = in2 ? voffset2 : in1 ? voffset1 : voffset0;
            a_voffset_odd = in2 ? odd2 : in1 ? odd1 : odd0;
            a_step = in2 ? bytes2 : in1 ? bytes1 : bytes0;
            a_soffset = (k0 - (in2 ? end1 : in1 ? end0 : 0)) * static_cast<unsigned int>(sizeof(T));
        } else {
            a_soffset = a_src.first_offset(k0, 0);
        }
        b_soffset = b_src.first_offset(k0, 0);
    };
    auto issue = [&](auto index, unsigned int stage_lds) __attribute__((always_inline)) {
        constexpr int l = decltype(index)::value;
        if constexpr (l < kOperandLoads && A_K && SEGMENTED)
            a_soffset = load_to_lds<l * kLoadBytes>(a_rsrc, stage_lds, l % 2 == 0 ? a_voffset : a_voffset_odd, a_soffset, a_step);
        else if constexpr (l < kOperandLoads)
            a_soffset = load_to_lds<l * kLoadBytes>(a_src.rsrc, stage_lds, a_src.load_voffset(l), a_soffset, a_src.group_bytes);
        else
            b_soffset = load_to_lds<l * kLoadBytes>(b_src.rsrc, stage_lds, b_src.load_voffset(l - kOperandLoads), b_soffset, b_src.group_bytes);
    };

    static_for<0, STAGES>([&](auto s) {
        if (decltype(s)::value < tiles) {
            aim(decltype(s)::value);
            static_for<0, kLoads>([&](auto l) { issue(l, lds_wave + decltype(s)::value * kStageBytes); });
        }
    });

    constexpr int kAOffsets = A_K ? kSteps : kBlocks, kBOffsets = B_K ? kSteps : kBlocks;
    int a_off[kAOffsets], b_off[kBOffsets];
#pragma unroll
    for (int i = 0; i < kAOffsets; ++i) a_off[i] = A_K ? ATile::lane_offset(lane, i) : ATile::lane_offset(lane, i * 16);
#pragma unroll
    for (int j = 0; j < kBOffsets; ++j) b_off[j] = B_K ? BTile::lane_offset(lane, j) : BTile::lane_offset(lane, j * 16);
    // Fragments of the step being multiplied and of the next one: step s of a K tile is in af[s], bf[s].
    constexpr int kFrags = 2 * kBlocks;
    frag_t af[kSteps][kBlocks], bf[kSteps][kBlocks];
    auto read_frag = [&]<int STEP, int F>(const T* stage) __attribute__((always_inline)) {
        if constexpr (F < kBlocks) {
            if constexpr (A_K) af[STEP][F] = ATile::frag(stage, F * 16, a_off[STEP]);
            else af[STEP][F] = ATile::frag(stage + STEP * ATile::kStepElems, a_off[F]);
        } else {
            constexpr int j = F - kBlocks;
            if constexpr (B_K) bf[STEP][j] = BTile::frag(stage + kOperandElems, j * 16, b_off[STEP]);
            else bf[STEP][j] = BTile::frag(stage + kOperandElems + STEP * BTile::kStepElems, b_off[j]);
        }
    };

    acc_t acc[kBlocks][kBlocks];
#pragma unroll
    for (int i = 0; i < kBlocks; ++i)
#pragma unroll
        for (int j = 0; j < kBlocks; ++j) acc[i][j] = acc_t(0.0f);
    // fp32, segments along K: a sum per segment, and those added up, as calls of their own that accumulate would. One chain over
    // all of them rounds more often: 512 + 512 + 512 columns, 300 rows, 1.38e-5 off the sums in 64 bits, this 8.24e-6, calls of their
    // own 8.23e-6. Both forms of 64 x 64 tiles keep their workgroups per CU, 251 registers of 256; a step of 256 tokens as long as before.
    constexpr bool kSegmentSums = A_K && SEGMENTED && std::is_same_v<T, float>;
    acc_t segment_sums[kSegmentSums ? kBlocks : 1][kSegmentSums ? kBlocks : 1];
    int border0 = 0, border1 = 0;  // this wavefront's first K tiles past the segments' ends
    if constexpr (kSegmentSums) {
        const int first_tile = kt_begin / kSteps + wave;
        border0 = (a_end0 / (kSteps * kBK<T>) - first_tile + kWaves - 1) / kWaves;
        border1 = (a_end1 / (kSteps * kBK<T>) - first_tile + kWaves - 1) / kWaves;
#pragma unroll
        for (int i = 0; i < kBlocks; ++i)
#pragma unroll
            for (int j = 0; j < kBlocks; ++j) segment_sums[i][j] = acc_t(0.0f);
    }
    auto close_segment = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < kBlocks; ++i)
#pragma unroll
            for (int j = 0; j < kBlocks; ++j) {
                segment_sums[i][j] += acc[i][j];
                acc[i][j] = acc_t(0.0f);
            }
    };
    // The column sums are one more block of columns whose B is ones. Not in fp32 storage, where such a chain of additions
    // shows (5399 rows: 7.0e-7 off the sums in 64 bits, the separate operator 1.2e-7) and takes the matrix cores' time: there a
    // lane adds the four values it holds and collects them in 64 bits (both gradients and the bias's, us: 512 x 512 x 512 8.7 -> 8.3,
    // 2000 x 1024 x 1024 75.5 -> 70.4; 6e-8 off).
    constexpr bool kWideSums = std::is_same_v<T, float>;
    const bool sums = SUMS && p.a_sums != nullptr && n0 == 0;
    std::conditional_t<kWideSums, double, acc_t> column_sums[SUMS ? kBlocks : 1];
    frag_t ones;
    if constexpr (SUMS) {
#pragma unroll
        for (int i = 0; i < kBlocks; ++i) {
            if constexpr (kWideSums) column_sums[i] = 0.0;
            else column_sums[i] = acc_t(0.0f);
        }
#pragma unroll
        for (int e = 0; e < static_cast<int>(sizeof(frag_t) / sizeof(T)); ++e) ones[e] = static_cast<T>(1.0f);
    }
    // One step's MFMAs. NEXT: the fragments of the step after it are read from `next_stage`, one per MFMA; LOADS: a K tile
    // is requested into the stage at refill_lds, its loads dealt out over the step.
    constexpr int kMfmas = kBlocks * kBlocks;
    auto multiply = [&]<int STEP, bool NEXT, bool LOADS>(const T* next_stage, unsigned int refill_lds) __attribute__((always_inline)) {
        static_for<0, kMfmas>([&](auto index) {
            constexpr int m = decltype(index)::value, row = m / kBlocks, column = (row & 1) ? kBlocks - 1 - m % kBlocks : m % kBlocks;
            Mfma<T>::add(acc[row][column], bf[STEP][column], af[STEP][row]);
            if constexpr (NEXT && m < kFrags) read_frag.template operator()<1 - STEP, m>(next_stage);
            if constexpr (LOADS) static_for<m * kLoads / kMfmas, (m + 1) * kLoads / kMfmas>([&](auto l) { issue(l, refill_lds); });
            __builtin_amdgcn_sched_barrier(0);
        });
        if constexpr (SUMS) {
            if (sums) {
#pragma unroll
                for (int i = 0; i < kBlocks; ++i) {
                    const frag_t& a = af[STEP][i];
                    if constexpr (kWideSums) column_sums[i] += static_cast<double>((a[0] + a[1]) + (a[2] + a[3]));
                    else Mfma<T>::add(column_sums[i], ones, a);
                }
            }
        }
    };
    static_assert(kFrags <= kMfmas, "a fragment read per MFMA");
    // With one stage the next K tile's first fragments wait for its loads, which the other wavefront of the SIMD covers; with
    // more, they are read a step ahead.
    constexpr bool kAhead = STAGES > 1;
    auto first_fragments = [&](const T* stage) __attribute__((always_inline)) {
        static_for<0, kFrags>([&](auto f) { read_frag.template operator()<0, decltype(f)::value>(stage); });
    };
    if (kAhead && tiles > 0) {
        if (tiles >= STAGES) wait_loads<(STAGES - 1) * kLoads>();
        else wait_loads<0>();
        first_fragments(wave_stages);
    }
    int stage = 0, t = 0;
    // First step of K tile t, and the wait after which its stage is free.
    auto first_step = [&]() __attribute__((always_inline)) {
        if constexpr (kSegmentSums)
            if (t == border0 || t == border1) close_segment();
        if constexpr (!kAhead) {
            wait_loads<0>();
            first_fragments(wave_stages);
        }
        multiply.template operator()<0, true, false>(wave_stages + stage * kStageElems, 0u);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    };
    for (; t + STAGES < tiles; ++t) {
        first_step();
        aim(t + STAGES);
        const int next_stage = stage + 1 == STAGES ? 0 : stage + 1;
        if constexpr (kAhead) wait_loads<(STAGES - (kAhead ? 2 : 1)) * kLoads>();
        multiply.template operator()<1, kAhead, true>(wave_stages + next_stage * kStageElems, lds_wave + stage * kStageBytes);
        stage = next_stage;
    }
    for (; t < tiles; ++t) {
        first_step();
        const int next_stage = stage + 1 == STAGES ? 0 : stage + 1;
        if (kAhead && t + 1 < tiles) {
            wait_loads<0>();
            multiply.template operator()<1, true, false>(wave_stages + next_stage * kStageElems, 0u);
        } else if (t + 1 < tiles || whole_last) {
            multiply.template operator()<1, false, false>(wave_stages, 0u);
        }
        stage = next_stage;
    }

    if constexpr (kSegmentSums) {
        close_segment();
#pragma unroll
        for (int i = 0; i < kBlocks; ++i)
#pragma unroll
            for (int j = 0; j < kBlocks; ++j) acc[i][j] = segment_sums[i][j];
    }
    // The partial tiles, [wavefront][row][column] in fp32. Everybody's fragments have to be read before the stages are reused.
    constexpr int kPitch = TILE + 4;
    static_assert(kWaves * TILE * kPitch * 4 <= kWaves * STAGES * kStageBytes + 8192, "partial tiles fit where the stages were");
    float* const partial = reinterpret_cast<float*>(smem_raw);
    wait_loads<0>();
    __syncthreads();
    {
        float* mine = partial + wave * TILE * kPitch + (lane & 15) * kPitch + (lane >> 4) * 4;
#pragma unroll
        for (int i = 0; i < kBlocks; ++i)
#pragma unroll
            for (int j = 0; j < kBlocks; ++j) *reinterpret_cast<acc_t*>(mine + i * 16 * kPitch + j * 16) = acc[i][j];
        if constexpr (SUMS) {
            // Row r's sum into the padding behind the row: every lane of row lane%16 holds it, or its share.
            if (sums) {
#pragma unroll
                for (int i = 0; i < kBlocks; ++i) {
                    float total;
                    if constexpr (kWideSums) {
                        double shares = column_sums[i];
                        shares += __shfl_xor(shares, 16, kWave);
                        shares += __shfl_xor(shares, 32, kWave);
                        total = static_cast<float>(shares);
                    } else {
                        total = column_sums[i][0];
                    }
                    if (lane < 16) partial[wave * TILE * kPitch + (i * 16 + lane) * kPitch + TILE] = total;
                }
            }
        }
    }
    __syncthreads();
    if constexpr (SUMS) {
        if (sums && threadIdx.x < TILE && m0 + static_cast<int>(threadIdx.x) < p.m) {
            const float* from = partial + threadIdx.x * kPitch + TILE;
            float v = from[0];
#pragma unroll
            for (int w = 1; w < kWaves; ++w) v += from[w * TILE * kPitch];
            T* out = static_cast<T*>(p.a_sums) + m0 + threadIdx.x;
            *out = from_f32<T>(p.a_sums_accumulate ? v + to_f32(*out) : v);
        }
    }
    void* c_base = p.c;
    long c_ld = p.ldc;
    int c_col0 = n0, c_cols = p.n;
    if constexpr (SEGMENTED && EPILOGUE != SmallEpilogue::split) {
        if (p.c_seg.count > 0) {
            const SegmentPick pick = pick_small_segment(p.c_seg, n0);
            c_base = const_cast<void*>(pick.ptr);
            c_ld = pick.ld;
            c_col0 = n0 - pick.first;
            c_cols = pick.cols;
        }
    }
    if constexpr (EPILOGUE == SmallEpilogue::split) {
        c_base = static_cast<float*>(p.c) + static_cast<long>(slice) * p.m * p.ldc;
        c_cols = static_cast<int>(p.ldc);
    }
    // Thread t owns TILE / 8 consecutive columns of row t/8 (and of row 32 + t/8).
    constexpr int kColumns = TILE / 8, kQuads = kColumns / 4;
#pragma unroll
    for (int pass = 0; pass < TILE / 32; ++pass) {
        const int row = pass * 32 + threadIdx.x / 8, col = (threadIdx.x % 8) * kColumns;
        const float* from = partial + row * kPitch + col;
        acc_t v[kQuads];
#pragma unroll
        for (int q = 0; q < kQuads; ++q) v[q] = *reinterpret_cast<const acc_t*>(from + 4 * q);
#pragma unroll
        for (int w = 1; w < kWaves; ++w)
#pragma unroll
            for (int q = 0; q < kQuads; ++q) v[q] += *reinterpret_cast<const acc_t*>(from + w * TILE * kPitch + 4 * q);
        const int m = m0 + row, c_col = c_col0 + col;
        if (m >= p.m || c_col >= c_cols) continue;
        const long at = static_cast<long>(m) * c_ld + c_col;
        if constexpr (EPILOGUE == SmallEpilogue::split) {
#pragma unroll
            for (int q = 0; q < kQuads; ++q) *reinterpret_cast<acc_t*>(static_cast<float*>(c_base) + at + 4 * q) = v[q];
        } else if constexpr (EPILOGUE == SmallEpilogue::plain) {
            T* out = static_cast<T*>(c_base) + at;
            if constexpr (kQuads == 2 && sizeof(T) == 2) {
                vec_t<float, 8> whole;
#pragma unroll
                for (int e = 0; e < 8; ++e) whole[e] = v[e / 4][e % 4];
                store_vec<T, 8>(out, vec_from_f32<T, 8>(whole));
            } else {
#pragma unroll
                for (int q = 0; q < kQuads; ++q) store_vec<T, 4>(out + 4 * q, vec_from_f32<T, 4>(v[q]));
            }
        } else {
            const int n = n0 + col;
            // Four columns at a time where C and what is added lie in whole aligned chunks, else one by one.
#pragma unroll
            for (int q = 0; q < kQuads; ++q) {
                const int nq = n + 4 * q;
                const long atq = at + 4 * q;
                if (!p.ragged) {
                    acc_t x = v[q];
                    if (p.addend != nullptr) x += *reinterpret_cast<const acc_t*>(p.addend + static_cast<long>(m) * p.ld_addend + nq);
                    if (p.bias != nullptr) x += vec_to_f32<T, 4>(load_vec<T, 4>(static_cast<const T*>(p.bias) + nq));
                    if (p.residual != nullptr)
                        x += vec_to_f32<T, 4>(load_vec<T, 4>(static_cast<const T*>(p.residual) + static_cast<long>(m) * p.ldr + nq));
                    if (p.c_f32) {
                        auto* out = reinterpret_cast<acc_t*>(static_cast<float*>(c_base) + atq);
                        *out = p.accumulate ? x + *out : x;
                    } else {
                        T* out = static_cast<T*>(c_base) + atq;
                        if (p.accumulate) x += vec_to_f32<T, 4>(load_vec<T, 4>(out));
                        store_vec<T, 4>(out, vec_from_f32<T, 4>(x));
                    }
                    continue;
                }
                for (int e = 0; e < 4; ++e) {
                    if (c_col + 4 * q + e >= c_cols) break;
                    float x = e == 0 ? v[q][0] : e == 1 ? v[q][1] : e == 2 ? v[q][2] : v[q][3];
                    if (p.addend != nullptr) x += p.addend[static_cast<long>(m) * p.ld_addend + nq + e];
                    if (p.bias != nullptr) x += to_f32(static_cast<const T*>(p.bias)[nq + e]);
                    if (p.residual != nullptr) x += to_f32(static_cast<const T*>(p.residual)[static_cast<long>(m) * p.ldr + nq + e]);
                    if (p.c_f32) {
                        float* out = static_cast<float*>(c_base) + atq + e;
                        *out = p.accumulate ? x + *out : x;
                    } else {
                        T* out = static_cast<T*>(c_base) + atq + e;
                        *out = from_f32<T>(p.accumulate ? x + to_f32(*out) : x);
                    }
                }
            }
        }
    }
}

template <typename T, int TILE, bool DEEP, bool A_K, bool B_K, SmallEpilogue EPILOGUE, bool SEGMENTED>
__global__ __launch_bounds__(kThreads) void gemm_small_kernel(SmallArgs p) {
    extern __shared__ __align__(1024) unsigned char smem_raw[];
    // Workgroups go to the XCDs round-robin, tile rows first: an XCD reads its share of A's panels and all of B.
    small_tile<T, TILE, DEEP, A_K, B_K, EPILOGUE, SEGMENTED, false>(p, blockIdx.x * TILE, blockIdx.y * TILE, blockIdx.z, smem_raw);
}

// Several calls in one launch. A launch of its own costs a small call more than its work does (2 us of start and end
// around 1 - 2 us), and two calls of a few dozen tiles each find room on the chip side by side. Both gradients of a
// projection, us in two launches and in one: 128 x 768 x 768 bf16 10.4, 7.7; 512 x 512 x 512 11.0, 7.4; 128 x 768 x 2048 fp32
// 23.0, 15.7; 2000 x 1024 x 2048 bf16 with bias 46, 34 (the bias's gradient took two launches more).
// CALLS: six, or two in translation units of their own, for the gradients of one projection. The host writes a launch's arguments across
// the bus, 1784 bytes for six: linear_backward of 128 x 768 x 768 takes 4.6 us of host time a call with them, 4.0 with two, and the block of
// 128 tokens, seven such calls of 46 and bound by the host, 200 and 187 us (one stream, calls in a row).
template <typename T, bool DEEP, int CALLS>
__global__ __launch_bounds__(kThreads) void gemm_small_group_kernel(SmallGroup<CALLS> group) {
    extern __shared__ __align__(1024) unsigned char smem_raw[];
    const int block = blockIdx.x;
    int which = 0;
#pragma unroll
    for (int i = 1; i < CALLS; ++i)
        if (i < group.count && block >= group.first_block[i]) which = i;
    int first = 0, tiles_m = 0, tile = 0;
    SmallLayout layout = SmallLayout::forward;
#pragma unroll
    for (int i = 0; i < CALLS; ++i) {
        const int first_i = group.first_block[i], tiles_i = group.tiles_m[i], tile_i = group.tile[i];
        const SmallLayout layout_i = group.layout[i];
        first = which == i ? first_i : first;
        tiles_m = which == i ? tiles_i : tiles_m;
        tile = which == i ? tile_i : tile;
        layout = which == i ? layout_i : layout;
    }
    // The call's arguments, read where they lie (the group is the kernel's only argument): indexing the parameter by a
    // run-time value would copy it to private memory.
    constexpr int kWords = sizeof(SmallArgs) / 4;
    struct Words {
        unsigned int w[kWords];
    } words;
    const auto* source = (const __attribute__((address_space(4))) unsigned int*)__builtin_amdgcn_kernarg_segment_ptr() +
                         offsetof(SmallGroup<CALLS>, call) / 4 + which * kWords;
#pragma unroll
    for (int i = 0; i < kWords; ++i) words.w[i] = source[i];
    const SmallArgs p = __builtin_bit_cast(SmallArgs, words);
    const int index = block - first;
    const int column = index / tiles_m, row = index - column * tiles_m;
    auto with_tile = [&]<int TILE>() __attribute__((always_inline)) {
        const int m0 = row * TILE, n0 = column * TILE;
        if (layout == SmallLayout::weight_gradient)
            small_tile<T, TILE, DEEP, false, false, SmallEpilogue::general, false, true>(p, m0, n0, 0, smem_raw);
        else if (layout == SmallLayout::input_gradient)
            small_tile<T, TILE, DEEP, true, false, SmallEpilogue::general, false, false>(p, m0, n0, 0, smem_raw);
        else if (layout == SmallLayout::forward)
            small_tile<T, TILE, DEEP, true, true, SmallEpilogue::general, false, false>(p, m0, n0, 0, smem_raw);
        else
            small_tile<T, TILE, DEEP, true, false, SmallEpilogue::general, true, false>(p, m0, n0, 0, smem_raw);
    };
    if (tile == 32) with_tile.template operator()<32>();
    else with_tile.template operator()<64>();
}

template <typename T, bool DEEP, int CALLS>
int launch_small_group_kernel(const SmallGroup<CALLS>& group, int blocks, hipStream_t stream) {
    constexpr int smem = small_smem_bytes<64, DEEP>() + (DEEP ? 0 : 8192);  // 64 x 64 partial tiles need 68 KiB
    auto kernel = gemm_small_group_kernel<T, DEEP, CALLS>;
    static const hipError_t status =
        hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, smem);
    CGPTX_HIP(status);
    hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned int>(blocks)), dim3(kThreads), smem, stream, group);
    CGPTX_LAUNCH_CHECK();
    return CGPTX_OK;
}

template <typename T, int CALLS>
int launch_small_group(const SmallGroup<CALLS>& group, int blocks, bool deep, hipStream_t stream) {
    return deep ? launch_small_group_kernel<T, true, CALLS>(group, blocks, stream) : launch_small_group_kernel<T, false, CALLS>(group, blocks, stream);
}

template <typename T, int TILE, bool DEEP, bool A_K, bool B_K, SmallEpilogue EPILOGUE, bool SEGMENTED>
int launch_small_kernel(const SmallCall& call, hipStream_t stream) {
    constexpr int smem = small_smem_bytes<TILE, DEEP>() + (TILE == 64 && !DEEP ? 8192 : 0);  // 64 x 64 partial tiles need 68 KiB
    auto kernel = gemm_small_kernel<T, TILE, DEEP, A_K, B_K, EPILOGUE, SEGMENTED>;
    static const hipError_t status =
        hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, smem);
    CGPTX_HIP(status);
    const auto& a = call.args;
    const dim3 grid(static_cast<unsigned int>((a.m + TILE - 1) / TILE), static_cast<unsigned int>((a.n + TILE - 1) / TILE),
                    static_cast<unsigned int>(call.slices));
    if (grid.y > 65535u || grid.z > 65535u) return fail(CGPTX_OVERFLOW, "gemm: too many tiles");
    hipLaunchKernelGGL(kernel, grid, dim3(kThreads), smem, stream, a);
    CGPTX_LAUNCH_CHECK();
    return CGPTX_OK;
}

template <typename T, int TILE, bool DEEP, bool A_K, bool B_K>
int launch_small_epilogue(const SmallCall& call, hipStream_t stream) {
    if constexpr (sizeof(T) == 2) {
        if (call.args.a_seg.count > 0 || call.args.c_seg.count > 0) {
            if (call.epilogue == SmallEpilogue::plain)
                return launch_small_kernel<T, TILE, DEEP, A_K, B_K, SmallEpilogue::plain, true>(call, stream);
            if (call.epilogue == SmallEpilogue::split)
                return launch_small_kernel<T, TILE, DEEP, A_K, B_K, SmallEpilogue::split, true>(call, stream);
            return fail(CGPTX_RUNTIME, "gemm: segmented operands take nothing added to their product");
        }
    }
    switch (call.epilogue) {
        case SmallEpilogue::plain: return launch_small_kernel<T, TILE, DEEP, A_K, B_K, SmallEpilogue::plain, false>(call, stream);
        case SmallEpilogue::split: return launch_small_kernel<T, TILE, DEEP, A_K, B_K, SmallEpilogue::split, false>(call, stream);
        default: return launch_small_kernel<T, TILE, DEEP, A_K, B_K, SmallEpilogue::general, false>(call, stream);
    }
}

template <typename T>
int launch_small(const SmallCall& call, hipStream_t stream) {
    auto with_layout = [&]<bool A_K, bool B_K>() -> int {
        if (call.tile == 32)
            return call.deep ? launch_small_epilogue<T, 32, true, A_K, B_K>(call, stream)
                             : launch_small_epilogue<T, 32, false, A_K, B_K>(call, stream);
        return call.deep ? launch_small_epilogue<T, 64, true, A_K, B_K>(call, stream)
                         : launch_small_epilogue<T, 64, false, A_K, B_K>(call, stream);
    };
    if (call.a_k_contiguous && call.b_k_contiguous) return with_layout.template operator()<true, true>();
    if (call.a_k_contiguous) return with_layout.template operator()<true, false>();
    if (!call.b_k_contiguous) return with_layout.template operator()<false, false>();
    return fail(CGPTX_RUNTIME, "gemm: unsupported operand layout");
}

}  // namespace
}  // namespace cgptx
