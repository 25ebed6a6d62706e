// Operand tiles and matrix instructions shared by the contraction kernels (gemm.hip, gemm_small.hpp).
#pragma once

#include "gemm_large.hpp"

#include <limits>
#include <type_traits>
#include <utility>

namespace cgptx {
namespace {

constexpr int kThreads = 256;
constexpr int kWaves = kThreads / kWave;
// K step per LDS stage: 64 bytes of a k-contiguous operand's row.
template <typename T>
constexpr int kBK = 64 / static_cast<int>(sizeof(T));
// K steps of one MFMA each per 16 x 16 block in a K tile of the persistent kernels: 128 bytes of a row.
constexpr int kSteps = 2;
constexpr int kXcds = 8;


using acc_t = vec_t<float, 4>;

// fp32 storage: four v_mfma_f32_16x16x4_f32 take the K tile of 16 (lane l holds row or column l%16 at k = 4*(l/16) + e
// for step e; the accumulator's layout is that of the 16-bit form). 64 accumulator registers at most, left to the
// compiler.
template <typename T>
struct Mfma;
template <>
struct Mfma<float> {
    using frag = vec_t<float, 4>;
    __device__ static __forceinline__ void run(acc_t& c, const frag& a, const frag& b) {
#pragma unroll
        for (int e = 0; e < 4; ++e) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[e], b[e], c, 0, 0, 0);
    }
    __device__ static __forceinline__ void add(acc_t& c, const frag& a, const frag& b) { run(c, a, b); }
    __device__ static __forceinline__ void start(acc_t& c, const frag& a, const frag& b) {
        c = acc_t(0.0f);
        run(c, a, b);
    }
};

// 16-bit storage: c += a x b with v_mfma_f32_16x16x32 (a: 16 rows x 32 k, b: 32 k x 16 columns; lane l holds row or
// column l%16, k = 8*(l/16) .. +7; c: lane l holds rows 4*(l/16) .. +3 of column l%16). Written as
// assembly so that the accumulator is updated in place: the four-register form of the instruction
// does not tie its result to its addend, and with all 256 accumulator registers in use the register
// allocator would otherwise shuffle accumulators around every MFMA. The kernel keeps the distances
// the hardware asks for by construction: an accumulator is touched once per K step (64, 48 or 16 MFMAs
// apart), zeroed long before its first MFMA and read by the epilogue only after a barrier.
template <>
struct Mfma<bf16_t> {
    using frag = vec_t<bf16_t, 8>;
    __device__ static __forceinline__ void run(acc_t& c, const frag& a, const frag& b) {
        asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
    }
    // The same through the compiler, which then knows the instruction's wait states: for kernels with registers to spare.
    __device__ static __forceinline__ void add(acc_t& c, const frag& a, const frag& b) {
        c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
    }
    // c = a x b: the first K tile of an item starts the sums, so the accumulators are never cleared.
    __device__ static __forceinline__ void start(acc_t& c, const frag& a, const frag& b) {
        asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, 0" : "=a"(c) : "v"(a), "v"(b));
    }
};
template <>
struct Mfma<f16_t> {
    using frag = vec_t<f16_t, 8>;
    __device__ static __forceinline__ void run(acc_t& c, const frag& a, const frag& b) {
        asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
    }
    __device__ static __forceinline__ void add(acc_t& c, const frag& a, const frag& b) {
        c = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
    }
    __device__ static __forceinline__ void start(acc_t& c, const frag& a, const frag& b) {
        asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, 0" : "=a"(c) : "v"(a), "v"(b));
    }
};

using u32x4 = vec_t<unsigned int, 4>;

// The column segment (of up to three) that holds column `col`, picked with selects: indexing the
// kernel-argument arrays by a run-time value would move them to private memory.
struct SegmentPick {
    const void* ptr;
    long ld;
    int first;  // first column of the segment
    int cols;
    int index;  // which segment
};
__device__ __forceinline__ SegmentPick pick_segment(const KernelSegments& seg, int col) {
    const int end0 = seg.cols[0], end1 = end0 + seg.cols[1];
    const bool in1 = seg.count > 1 && col >= end0;
    const bool in2 = seg.count > 2 && col >= end1;
    SegmentPick pick;
    pick.ptr = in2 ? seg.ptr[2] : in1 ? seg.ptr[1] : seg.ptr[0];
    pick.ld = in2 ? seg.ld[2] : in1 ? seg.ld[1] : seg.ld[0];
    pick.first = in2 ? end1 : in1 ? end0 : 0;
    pick.cols = in2 ? seg.cols[2] : in1 ? seg.cols[1] : seg.cols[0];
    pick.index = in2 ? 2 : in1 ? 1 : 0;
    return pick;
}

// s_waitcnt immediate that waits until at most `count` vector-memory operations are outstanding
// (and for nothing else).
constexpr int vmcnt_immediate(int count) { return (count & 15) | ((count >> 4) << 14) | 0x0F70; }

// Buffer descriptor (raw buffer, range-checked) over `bytes` bytes starting at base (both the same
// for all lanes). The words are pinned to scalar registers: 64-bit comparisons have no scalar form,
// and one of them on the way would drag the descriptor, and every address derived with it, into
// vector registers.
__device__ __forceinline__ u32x4 make_rsrc(const void* base, long bytes) {
    const unsigned long address = reinterpret_cast<unsigned long>(base);
    const unsigned int size_low = static_cast<unsigned int>(bytes);
    const unsigned int size_high = static_cast<unsigned int>(static_cast<unsigned long>(bytes) >> 32);
    u32x4 words;
    words[0] = __builtin_amdgcn_readfirstlane(static_cast<unsigned int>(address));
    words[1] = __builtin_amdgcn_readfirstlane(static_cast<unsigned int>(address >> 32) & 0xFFFFu);  // stride 0
    words[2] = __builtin_amdgcn_readfirstlane(size_high != 0 ? 0xFFFFFFFFu : size_low);
    words[3] = 0x00020000u;
    return words;
}

// One wavefront-wide 16-byte-per-lane load from a buffer straight into LDS: lane l's bytes land at
// lds_base + LDS_OFFSET + 16 l. Returns soffset + step, the scalar offset of the operand's next load
// (that addition sits between the write of M0 and the load, which need one instruction between them
// anyway). Written as assembly on purpose: the compiler would order every later LDS read after *all*
// outstanding loads of this kind (vmcnt(0)), which defeats keeping several K tiles in flight; the
// kernel counts its loads itself (vmcnt_immediate). M0 is used by nothing else here.
template <int LDS_OFFSET>
__device__ __forceinline__ unsigned int load_to_lds(const u32x4& rsrc, unsigned int lds_base, int voffset,
                                                    unsigned int soffset, unsigned int step) {
    unsigned int next;
    asm volatile("s_add_u32 m0, %1, %2\n\ts_add_u32 %0, %3, %4\n\tbuffer_load_dwordx4 %5, %6, %3 offen lds"
                 : "=&s"(next)
                 : "s"(lds_base), "n"(LDS_OFFSET), "s"(soffset), "s"(step), "v"(voffset), "s"(rsrc)
                 : "scc");
    return next;
}

// Workgroup barrier without the fence __syncthreads() carries: LDS reads still in flight may
// cross it (their registers are waited for where they are used).
__device__ __forceinline__ void barrier_only() { asm volatile("s_barrier" ::: "memory"); }

// Where a wavefront's loads of one operand's K tile come from: load i reads at scalar offset
// soffset + i * step.
struct TileCursor {
    u32x4 rsrc;
    int voffset;
    unsigned int soffset;
    unsigned int step;
    // Advance after the operand's odd-numbered loads, towards an up unit and back (differ from step only for SWIGLU's B).
    unsigned int step_up, step_back;
};

template <int BEGIN, int... I, typename F>
__device__ __forceinline__ void static_for_impl(std::integer_sequence<int, I...>, F&& f) {
    (f(std::integral_constant<int, BEGIN + I>{}), ...);
}
// f(integral_constant<int, i>) for i = BEGIN .. END-1, unrolled at compile time.
template <int BEGIN, int END, typename F>
__device__ __forceinline__ void static_for(F&& f) {
    static_for_impl<BEGIN>(std::make_integer_sequence<int, (END > BEGIN ? END - BEGIN : 0)>{}, f);
}

template <typename T>
__device__ __forceinline__ unsigned int lds_address_of(const T* p) {
    return static_cast<unsigned int>(reinterpret_cast<unsigned long>((__attribute__((address_space(3))) const T*)(p)));
}

// Operand tiles travel global -> LDS with buffer_load ... lds: a wavefront-wide load drops
// 64 x 16 B contiguously into LDS, no staging registers and no LDS stores, and the only per-lane
// address is a loop-invariant byte offset (the K position is a scalar offset). LDS rows therefore
// cannot be padded; bank conflicts are avoided by storing 16-byte chunk c of a row at chunk
// position c ^ swizzle(row) — the lane that owns an LDS slot fetches the matching global chunk.

// ---- operand stored [ROWS, K] (k-contiguous): ROWS x (kSteps * kBK) slab, unpadded LDS rows -----
// A row of the slab is two K steps, a whole cache line: a load instruction then touches 8
// lines instead of 16 halves of lines, which is what the path from the L2s to a CU's LDS is bound by (16 KiB of operand
// tiles per CU, every CU loading: 0.25 us in pieces of 64 bytes, 0.17 us in pieces of 128, no more in longer ones).
// One load instruction covers 1024 B = kRowsPerLoad rows; wavefront w issues the loads of row
// groups w, w+4, ... The chunk swizzle is (row / rows per 256 B) mod chunks per row: the 16 rows a
// quarter-wavefront reads with ds_read_b128 then hit the 16 different 16-byte positions of a
// 256-byte bank period.
template <typename T, int ROWS>
struct KTile {
    using frag_t = typename Mfma<T>::frag;
    static constexpr int kRowElems = kSteps * kBK<T>;
    static constexpr int kChunksPerRow = kRowElems / kVec128<T>;
    static constexpr int kRowsPerLoad = 64 / kChunksPerRow;
    static constexpr int kElems = ROWS * kRowElems;
    static constexpr int kLoads = ROWS / kRowsPerLoad / kWaves;  // load instructions per wavefront and tile

    u32x4 rsrc = {0u, 0u, 0u, 0u};
    int voffset = 0, voffset1 = 0;
    unsigned int group_bytes = 0;  // kRowsPerLoad rows further in global memory

    __device__ __forceinline__ static int swizzle(int row) { return (row / 2) % kChunksPerRow; }

    // base: element (row0, 0) of the operand; rows past rows_left only feed C rows that are never
    // stored (they read zeros or whatever follows, never out of the allocation's last row). A tile may start behind the
    // last row (C wider than the operand's rows): rows_left <= 0, and everything reads as zeros.
    __device__ __forceinline__ void init(const T* base, long ld, int rows_left, int k_total, int wave) {
        const int lane = threadIdx.x & (kWave - 1);
        rsrc = make_rsrc(base, (static_cast<long>(rows_left - 1) * ld + k_total) * static_cast<long>(sizeof(T)));
        rsrc[2] = rows_left > 0 ? rsrc[2] : 0u;
        const int row = lane / kChunksPerRow;
        // The tile row of this lane's slot is (i*4 + wave) * kRowsPerLoad + row; its swizzle does not depend on i.
        voffset = static_cast<int>(row * ld * sizeof(T)) +
                  (((lane % kChunksPerRow) ^ swizzle(wave * kRowsPerLoad + row)) * 16);
        voffset1 = static_cast<int>(row * ld * sizeof(T)) +
                   (((lane % kChunksPerRow) ^ swizzle((wave + 1) * kRowsPerLoad + row)) * 16);
        group_bytes = __builtin_amdgcn_readfirstlane(static_cast<unsigned int>(kRowsPerLoad * ld * sizeof(T)));
    }
    // The lane's offset for load i of a wavefront that loads the whole tile (init with wave 0): with eight rows per load
    // the swizzle of every other load differs.
    __device__ __forceinline__ int load_voffset(int i) const { return (i & 1) != 0 ? voffset1 : voffset; }
    // Scalar offset of wavefront `wave`'s first load of the tile that starts at column k0.
    __device__ __forceinline__ unsigned int first_offset(int k0, int wave) const {
        return wave * group_bytes + k0 * static_cast<unsigned int>(sizeof(T));
    }
    // Element offset of the lane's fragment of K step `step` within a 16-row block: row lane%16, the lane/16-th
    // 16 bytes of the step's part of it. The swizzle of a row does not depend on the block.
    __device__ __forceinline__ static int lane_offset(int lane, int step = 0) {
        return (lane & 15) * kRowElems + ((((lane >> 4) + 4 * step) ^ swizzle(lane & 15)) * kVec128<T>);
    }
    __device__ __forceinline__ static frag_t frag(const T* tile, int block0, int offset) {
        return *reinterpret_cast<const frag_t*>(tile + block0 * kRowElems + offset);
    }
};

// ---- operand stored [K, COLS] (n-contiguous): (kSteps * kBK) x COLS slab kept in that order in LDS
// The transpose happens on the way out of LDS: ds_read_b64_tr_b16 hands lane n of a 16-lane group
// the four k-values of column n from a 4(k) x 16(n) block, so two of them build the 8-k fragment of
// one column. swizzle(k row) = 4*(row%4) on the chunk index (rows of 128 bytes: 4*(row/2%2), the row's parity
// picks the half already): the four k rows that 32 lanes read sit in four different 64-byte windows of the
// 256-byte bank period. K rows past the operand's end are out of the buffer's range and read as zeros.
template <typename T, int COLS>
struct NTile {
    using frag_t = typename Mfma<T>::frag;
    static constexpr int kChunksPerRow = COLS / kVec128<T>;
    static constexpr int kRowsPerLoad = 64 / kChunksPerRow;  // k rows one load instruction covers
    static constexpr int kStepElems = kBK<T> * COLS;         // K step s starts at s * kStepElems
    static constexpr int kElems = kSteps * kStepElems;
    static constexpr int kLoads = kSteps * kBK<T> / kRowsPerLoad / kWaves;

    // fp32: the four k rows a read touches lie four apart (k = 4*(lane/16) + e).
    __device__ __forceinline__ static int swizzle(int k_row) {
        if constexpr (std::is_same_v<T, float>) return COLS == 64 ? k_row & 12 : k_row & 4;
        else return COLS >= 128 ? (k_row & 3) << 2 : COLS == 64 ? (k_row & 2) << 1 : (k_row & 8) >> 2;
    }

    u32x4 rsrc = {0u, 0u, 0u, 0u};
    int voffset = 0, voffset1 = 0, voffset2 = 0, voffset3 = 0;
    unsigned int group_bytes = 0;  // kRowsPerLoad k rows further in global memory

    // base: element (0, col0) of the operand. Column chunks past cols_left are clamped to the last
    // valid chunk: they only feed C columns that are never stored.
    __device__ __forceinline__ void init(const T* base, long ld, int cols_left, int k_total, int wave) {
        const int lane = threadIdx.x & (kWave - 1);
        rsrc = make_rsrc(base, (static_cast<long>(k_total - 1) * ld + cols_left) * static_cast<long>(sizeof(T)));
        const int row = lane / kChunksPerRow;                  // within the instruction's rows
        const int k_row = wave * kRowsPerLoad + row;           // tile row of the first load; its swizzle is that of all
        const int chunk = min((lane % kChunksPerRow) ^ swizzle(k_row), cols_left / kVec128<T> - 1);
        voffset = static_cast<int>(row * ld * sizeof(T)) + chunk * 16;
        if constexpr (std::is_same_v<T, float> && COLS == 64) {
            auto at = [&](int i) { return static_cast<int>(row * ld * sizeof(T)) + min((lane % kChunksPerRow) ^ (4 * i), cols_left / kVec128<T> - 1) * 16; };
            voffset1 = at(1);
            voffset2 = at(2);
            voffset3 = at(3);
        }
        group_bytes = __builtin_amdgcn_readfirstlane(static_cast<unsigned int>(kRowsPerLoad * ld * sizeof(T)));
    }
    // The lane's offset for load i of a wavefront that loads the whole tile (init with wave 0): fp32 tiles of 64 columns
    // cover four k rows per load, so that load i's swizzle is 4 (i % 4).
    __device__ __forceinline__ int load_voffset(int i) const {
        if constexpr (std::is_same_v<T, float> && COLS == 64) return i % 4 == 0 ? voffset : i % 4 == 1 ? voffset1 : i % 4 == 2 ? voffset2 : voffset3;
        else return voffset;
    }
    // Scalar offset of wavefront `wave`'s first load of the tile that starts at row k0.
    __device__ __forceinline__ unsigned int first_offset(int k0, int wave) const {
        return (wave + k0 / kRowsPerLoad) * group_bytes;
    }
    // Lane i of a 16-lane group addresses k row i/4, columns 4*(i%4) .. +3 of the group's 4 x 16
    // block; group g (lanes 16g .. 16g+15) takes the k values 8g .. 8g+7 of the fragment's 16
    // columns in two reads (k rows +0..3, +4..7). The offset is for the first read; block0 is a
    // multiple of 16.
    __device__ __forceinline__ static int lane_offset(int lane, int block0) {
        if constexpr (std::is_same_v<T, float>) {  // k rows 4*(lane/16) + e, column block0 + lane%16
            const int row = (lane >> 4) * 4, column_chunk = (block0 + (lane & 15)) / 4;
            return row * COLS + (column_chunk ^ swizzle(row)) * 4 + (lane & 3);
        }
        const int k_row = (lane >> 4) * 8 + ((lane & 15) >> 2);
        const int chunk = ((block0 / 8) ^ swizzle(k_row)) + ((lane & 3) >> 1);
        return k_row * COLS + chunk * 8 + (lane & 1) * 4;
    }
    __device__ __forceinline__ static frag_t frag(const T* tile, int offset) {
        if constexpr (std::is_same_v<T, float>) {
            const T* q = tile + offset;
            return frag_t{q[0], q[COLS], q[2 * COLS], q[3 * COLS]};
        } else {
        using s16x4 = vec_t<short, 4>;
        using lds_ptr = __attribute__((address_space(3))) s16x4*;
        const T* q = tile + offset;
        const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(q));
        const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(q + 4 * COLS));
        vec_t<short, 8> both;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            both[e] = lo[e];
            both[4 + e] = hi[e];
        }
        return __builtin_bit_cast(frag_t, both);
        }
    }
};

// ---- operand stored [K, 192] (n-contiguous), 16-bit: 128 columns and 64 columns side by side -----
// 384 bytes are no power of two of chunks for a load instruction's lanes, so each K step's slab is that of NTile<128>, then
// that of NTile<64>. Of a wavefront's six loads per K tile the third and the sixth are the 64 columns', at scalar offsets of
// their own.
template <typename T>
struct NTile192 {
    using frag_t = typename Mfma<T>::frag;
    using Wide = NTile<T, 128>;
    using Narrow = NTile<T, 64>;
    static constexpr int kStepElems = kBK<T> * 192;
    static constexpr int kNarrowElems = kBK<T> * 128;  // where a step's 64 columns start
    static constexpr int kElems = kSteps * kStepElems;
    static constexpr int kLoads = Wide::kLoads + Narrow::kLoads;
    static_assert(kSteps == 2 && Wide::kLoads == 4 && Narrow::kLoads == 2, "two loads of the 128 columns, one of the 64 per K step");

    u32x4 rsrc = {0u, 0u, 0u, 0u};
    int voffset = 0, narrow_voffset = 0;
    unsigned int group_bytes = 0;  // of the 128 columns; the 64 columns' loads cover twice the k rows

    __device__ __forceinline__ void init(const T* base, long ld, int cols_left, int k_total, int wave) {
        const int lane = threadIdx.x & (kWave - 1);
        rsrc = make_rsrc(base, (static_cast<long>(k_total - 1) * ld + cols_left) * static_cast<long>(sizeof(T)));
        const int last = cols_left / kVec128<T> - 1;
        auto at = [&](int per_row, int first, int swizzle) {
            const int row = lane / per_row;
            return static_cast<int>(row * ld * sizeof(T)) + min(first + ((lane % per_row) ^ swizzle), last) * 16;
        };
        voffset = at(Wide::kChunksPerRow, 0, Wide::swizzle(wave * Wide::kRowsPerLoad + lane / Wide::kChunksPerRow));
        narrow_voffset = at(Narrow::kChunksPerRow, Wide::kChunksPerRow,
                            Narrow::swizzle(wave * Narrow::kRowsPerLoad + lane / Narrow::kChunksPerRow));
        group_bytes = __builtin_amdgcn_readfirstlane(static_cast<unsigned int>(Wide::kRowsPerLoad * ld * sizeof(T)));
    }
    __device__ __forceinline__ unsigned int first_offset(int k0, int wave) const { return (wave + k0 / Wide::kRowsPerLoad) * group_bytes; }
    __device__ __forceinline__ unsigned int narrow_first_offset(int k0, int wave) const { return (2 * wave + k0 / Wide::kRowsPerLoad) * group_bytes; }
    // A block of 16 columns lies in one of the two parts.
    __device__ __forceinline__ static int wide_offset(int lane, int block0) { return Wide::lane_offset(lane, block0); }
    __device__ __forceinline__ static int narrow_offset(int lane, int block0) { return kNarrowElems + Narrow::lane_offset(lane, block0); }
};

}  // namespace
}  // namespace cgptx
