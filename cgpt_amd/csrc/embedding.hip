// Embedding gather (forward) and embedding-gradient scatter (backward) for gfx950.
//
// Backward semantics: include/ops/backward/embedding_backward.h:35-42. The
// reference scatters with storage-dtype atomics (src/ops/backward/embedding_backward.cu:68-92),
// so its rounding depends on arrival order. Here the tokens are grouped by id with a counting
// sort over the vocabulary (integer work: histogram, scan, fill — one launch), then each
// vocabulary row's tokens are added in ascending token order with one rounding to the
// storage dtype per add — the arithmetic of the reference's CPU operator
// (src/ops/cpu/backward/embedding_backward_cpu.cpp:99-112) — by one wavefront for most ids, by a
// workgroup per 64 columns for frequent ones. The result is deterministic and no float atomics are
// used. Token rows are read once with coalesced 128-bit accesses; rows that no token names are zero-filled by the same launch
// when the gradient is not accumulated.
#include "common.hpp"

#include <cstring>
#include <algorithm>
#include <limits>

namespace cgptx {
namespace {

constexpr int kThreads = 256;
constexpr int kWavesPerBlock = kThreads / kWave;

// ---- grouping: counting sort of the token positions by id -------------------------------------------
// Workgroup b owns the ids [b R, (b+1) R) and reads the whole id list: it counts its ids in an LDS histogram and, on the
// side, the tokens with smaller ids (which is where its part of the output begins: no workgroup waits for another); after an
// exclusive scan of the histogram it hands every token of its range the next free slot of its id's segment. The tokens of
// the range are listed in LDS on the way, by each wavefront in a part of its own, and handed out from there; a wavefront that
// found more than its part holds walks the id list again instead. Slots are handed out with LDS integer atomics, so the order
// inside a segment is whatever order the lanes arrived in: the row kernel puts each segment into ascending order itself.
// A segment of more than kShort tokens contains positions that are multiples of kShort; order's entries there are marked,
// which is how the row kernel finds the long segments, and the offset of a workgroup's first id is marked if there is one
// among its ids, which is how it finds out that it need not look.
// offsets[id] .. offsets[id + 1] is id's segment of `order`; ids >= vocab belong to nobody and are skipped.
// Bound by the walk over the id list: 32768 ids take 8000 clocks (their way through the CU's L1 and 32 comparisons a thread),
// and 4000 more where most of them match (text: half of the tokens are among the first 128 of 32000 ids); the scan 3000, the
// list 5000. With a second walk in place of the list 17000: the kernel took 18.4 us and takes 12.8. Ranges are as small as one
// workgroup per CU allows: fewer lanes match at a time (32000 ids in ranges of 128: 20900 clocks, of 1024: 22500).
constexpr int kGroupThreads = 1024;
constexpr unsigned int kGroupMinIds = 128, kGroupMaxIds = 32768;  // LDS histogram entries of one workgroup (up to 128 KiB)
constexpr int kGroupBatch = 8;                // 128-bit id loads a thread keeps in flight
constexpr unsigned int kShort = 64;           // tokens of a segment that one wavefront orders in registers: one lane each
constexpr unsigned int kLong = 1u << 31;      // the mark of longer segments; positions and tokens stay below it
constexpr std::size_t kGroupLds = 160 * 1024 - 512;  // for the histogram and the lists

// The id list is walked in batches of kGroupBatch x 4 ids per thread, all of a batch's loads requested before the
// first id is looked at (one dependent load per id would cost a memory round trip each). visit(id, t) sees every
// token once, in all lanes of a wavefront at a time: lanes without a token see an id that is in no range. A second walk
// shows a wavefront the same tokens; their order does not matter to any caller.
template <typename Visit>
__device__ __forceinline__ void for_each_id(const std::uint32_t* __restrict__ ids, unsigned int count, bool aligned, Visit&& visit) {
    using u32x4 = vec_t<unsigned int, 4>;
    constexpr unsigned int kNone = ~0u;
    const unsigned int quads = aligned ? count / 4 : 0;
    const unsigned int wave_first = __builtin_amdgcn_readfirstlane(threadIdx.x);
    const auto* wide = reinterpret_cast<const u32x4*>(ids);
    for (unsigned int base = 0; base < quads; base += kGroupBatch * kGroupThreads) {
        u32x4 held[kGroupBatch];
#pragma unroll
        for (int k = 0; k < kGroupBatch; ++k) held[k] = wide[min(base + k * kGroupThreads + threadIdx.x, quads - 1)];
#pragma unroll
        for (int k = 0; k < kGroupBatch; ++k) {
            if (base + k * kGroupThreads + wave_first >= quads) continue;
            const unsigned int q = base + k * kGroupThreads + threadIdx.x;
#pragma unroll
            for (int e = 0; e < 4; ++e) visit(q < quads ? held[k][e] : kNone, 4 * q + e);
        }
    }
    for (unsigned int t0 = 4 * quads; t0 + wave_first < count; t0 += kGroupThreads) {
        const unsigned int t = t0 + threadIdx.x;
        visit(t < count ? ids[t] : kNone, t);
    }
}

struct GroupArgs {
    unsigned int* offsets;
    unsigned int* order;
    const std::uint32_t* ids;
    unsigned int count, vocab, ids_per_group, token_bits, list_entries;
    bool aligned;
};

// bins: [ids_per_group], then the wavefronts' lists [list_entries].
__device__ __forceinline__ void group_ids(const GroupArgs& g, unsigned int* bins) {
    unsigned int* __restrict__ const offsets = g.offsets;
    unsigned int* __restrict__ const order = g.order;
    const std::uint32_t* __restrict__ const ids = g.ids;
    const unsigned int count = g.count, vocab = g.vocab, ids_per_group = g.ids_per_group, token_bits = g.token_bits, list_entries = g.list_entries;
    const bool aligned = g.aligned;
    __shared__ unsigned int wave_totals[kGroupThreads / kWave];
    __shared__ unsigned int smaller_total;
    const unsigned int lo = blockIdx.x * ids_per_group;
    const unsigned int width = min(ids_per_group, vocab - lo);
    const unsigned int tid = threadIdx.x, lane = tid & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    for (unsigned int i = tid; i < width; i += kGroupThreads) bins[i] = 0;
    if (tid == 0) smaller_total = 0;
    __syncthreads();
    // An entry of a list: the token in the lower token_bits, the id's place in the range above them.
    unsigned int* list = bins + ids_per_group + wave * list_entries;
    unsigned int smaller = 0, listed = 0;
    for_each_id(ids, count, aligned, [&](unsigned int id, unsigned int t) {
        const bool match = id - lo < width;
        smaller += id < lo ? 1u : 0u;
        const unsigned long long mask = __ballot(match);
        if (match) {
            atomicAdd(&bins[id - lo], 1u);
            const unsigned int entry = __builtin_amdgcn_mbcnt_hi(static_cast<unsigned int>(mask >> 32),
                                                                 __builtin_amdgcn_mbcnt_lo(static_cast<unsigned int>(mask), listed));
            if (entry < list_entries) list[entry] = t | (id - lo) << token_bits;
        }
        listed += __popcll(mask);
    });
#pragma unroll
    for (int offset = kWave / 2; offset > 0; offset >>= 1) smaller += __shfl_xor(smaller, offset, kWave);
    if (lane == 0 && smaller != 0) atomicAdd(&smaller_total, smaller);
    __syncthreads();
    // Exclusive scan of bins[0, width) in place, starting at the number of tokens with smaller ids: thread i
    // owns the contiguous piece [i per, (i + 1) per).
    const unsigned int per = (width + kGroupThreads - 1) / kGroupThreads;
    const unsigned int first = min(tid * per, width), last = min(first + per, width);
    unsigned int mine = 0;
    bool any_long = false;
    for (unsigned int i = first; i < last; ++i) {
        mine += bins[i];
        any_long = any_long || bins[i] > kShort;
    }
    unsigned int inclusive = mine;
#pragma unroll
    for (int offset = 1; offset < kWave; offset <<= 1) {
        const unsigned int other = __shfl_up(inclusive, offset, kWave);
        if (lane >= static_cast<unsigned int>(offset)) inclusive += other;
    }
    if (lane == kWave - 1) wave_totals[wave] = inclusive;
    any_long = __syncthreads_or(any_long);
    unsigned int before = smaller_total;
    for (unsigned int w = 0; w < wave; ++w) before += wave_totals[w];
    unsigned int running = before + inclusive - mine;
    for (unsigned int i = first; i < last; ++i) {
        const unsigned int n = bins[i];
        bins[i] = n > kShort ? running | kLong : running;
        offsets[lo + i] = i == 0 && any_long ? running | kLong : running;
        running += n;
    }
    if (lo + width == vocab && tid == kGroupThreads - 1) offsets[vocab] = running;  // the piece that ends the last range
    __syncthreads();
    auto place = [&](unsigned int slot, unsigned int t) { order[slot & ~kLong] = slot % kShort == 0 ? t | (slot & kLong) : t; };
    if (listed > list_entries) {
        for_each_id(ids, count, aligned, [&](unsigned int id, unsigned int t) {
            if (id - lo < width) place(atomicAdd(&bins[id - lo], 1u), t);
        });
        return;
    }
    const unsigned int token_mask = (1u << token_bits) - 1;
    constexpr unsigned int kAhead = 4;
    unsigned int i = lane;
    for (; i + (kAhead - 1) * kWave < listed; i += kAhead * kWave) {
        unsigned int entry[kAhead], slot[kAhead];
#pragma unroll
        for (unsigned int u = 0; u < kAhead; ++u) entry[u] = list[i + u * kWave];
#pragma unroll
        for (unsigned int u = 0; u < kAhead; ++u) slot[u] = atomicAdd(&bins[entry[u] >> token_bits], 1u);
#pragma unroll
        for (unsigned int u = 0; u < kAhead; ++u) place(slot[u], entry[u] & token_mask);
    }
    for (; i < listed; i += kWave) place(atomicAdd(&bins[list[i] >> token_bits], 1u), list[i] & token_mask);
}

__global__ __launch_bounds__(kGroupThreads) void embedding_group_kernel(GroupArgs g) {
    extern __shared__ unsigned int bins[];
    group_ids(g, bins);
}

// ---- rows ------------------------------------------------------------------------------------------
// Adds, into row `id` of the table, the rows of grad_output of the tokens with that id, in ascending token
// order with one rounding to the storage dtype per add. Rows without tokens are zero-filled unless the gradient
// is accumulated. Bound by HBM (three rows per token) as long as the serial chain of additions of the most
// frequent id is short; text makes it long: the first ids of a vocabulary take several per cent of a batch each.
//   * Segments of up to kShort tokens: one wavefront per id, tokens ordered in registers (lane i holds the token
//     of rank i), lanes across the columns, kAhead token rows in flight. With few tokens an id it is the chain of
//     loads that counts (offsets, token, row) and the wavefronts that are in flight against it: a wavefront takes two
//     ids, half a vocabulary apart, and looks both up before it adds either.
//   * Longer ones: one workgroup per id and kSlice columns, so that a frequent id occupies hidden / kSlice
//     workgroups instead of one wavefront. The segment is put into ascending order through a bitmap of token
//     positions in LDS, kSpan positions at a time, from which the list of the next kList tokens is drawn as often as it
//     takes; all threads fetch the slices of the next kBatch token rows while the first wavefront adds the
//     previous ones, one column per lane, from LDS, where it reads kReadAhead tokens ahead of the chain. A batch of 128
//     bf16 rows takes 3600 clocks, 2700 of them in the chain (add, round, and the reads beside them).
// Both live in one launch, the long segments' workgroups first: the chains of the frequent ids run beside the short
// segments (in a launch of their own they add their 50 us). So the short segments pay for the long ones' registers and LDS
// with wavefronts in flight, which is why both are bounded (LongRow::kWavesPerSimd) and why nothing is listed where the
// grouping found no long segment. 32768 tokens x 1024 columns in bf16 over 32000 ids, all launches: uniform ids 30 us, ids Zipf
// distributed 47 - 58, of which the most frequent id, 9.3 per cent of the tokens, sets the end (every id by one wavefront 35 and
// 2300; neither bounded nor told that there is nothing to list 48 and 75). A segment is read once per kSpan tokens of the batch,
// so its work grows with its tokens up to batches of millions: 131072 of 262144 tokens in one id, 128 columns, 2.1 ms
// (read once per 4096 tokens: 7.0).
constexpr unsigned int kSlice = 64;      // columns of a long segment's workgroup: one lane each, one or two cache lines
constexpr unsigned int kSpan = 65536;    // token positions covered by the bitmap at a time
constexpr unsigned int kList = 4096;     // tokens ordered at a time

template <typename T, bool Vector>
__device__ __forceinline__ void embedding_short_row(T* __restrict__ row, const T* __restrict__ grad_output,
                                                    unsigned int mine, unsigned int tokens, unsigned int hidden,
                                                    bool accumulate) {
    constexpr int VEC = Vector ? kVec128<T> : 1;
    constexpr unsigned int kAhead = 8;
    using vec_f = vec_t<float, VEC>;
    const unsigned int lane = threadIdx.x & (kWave - 1);
    if (tokens == 0) {
        if (!accumulate)
            for (unsigned int col = lane * VEC; col < hidden; col += kWave * VEC) store_vec<T, VEC>(row + col, vec_t<T, VEC>(0));
        return;
    }
    // rank = number of tokens of the segment below mine; sorted = the token of rank `lane`.
    unsigned int rank = 0;
    for (unsigned int j = 0; j < tokens; ++j)
        rank += static_cast<unsigned int>(__builtin_amdgcn_readlane(static_cast<int>(mine), static_cast<int>(j))) < mine ? 1u : 0u;
    const unsigned int sorted = static_cast<unsigned int>(
        __builtin_amdgcn_ds_permute(static_cast<int>(rank << 2), static_cast<int>(mine)));  // lane `rank` receives mine
    for (unsigned int col = lane * VEC; col < hidden; col += kWave * VEC) {
        vec_f acc = accumulate ? vec_to_f32<T, VEC>(load_vec<T, VEC>(row + col)) : vec_f(0.0f);
        // kAhead token rows are requested at a time; the additions keep their order.
        for (unsigned int j0 = 0; j0 < tokens; j0 += kAhead) {
            vec_t<T, VEC> dy[kAhead];
#pragma unroll
            for (unsigned int u = 0; u < kAhead; ++u)
                if (j0 + u < tokens) {
                    const auto token = static_cast<unsigned int>(
                        __builtin_amdgcn_readlane(static_cast<int>(sorted), static_cast<int>(j0 + u)));
                    dy[u] = load_vec<T, VEC>(grad_output + static_cast<std::size_t>(token) * hidden + col);
                }
#pragma unroll
            for (unsigned int u = 0; u < kAhead; ++u)
                if (j0 + u < tokens)  // one rounding to the storage dtype per add
                    acc = vec_to_f32<T, VEC>(vec_from_f32<T, VEC>(acc + vec_to_f32<T, VEC>(dy[u])));
        }
        store_vec<T, VEC>(row + col, vec_from_f32<T, VEC>(acc));
    }
}

// An element as it comes from LDS, in a register of its own.
template <typename T>
using raw_t = std::conditional_t<sizeof(T) == 2, unsigned int, float>;
template <typename T>
__device__ __forceinline__ raw_t<T> to_raw(T x) {
    if constexpr (sizeof(T) == 2) return __builtin_bit_cast(unsigned short, x);
    else return x;
}
template <typename T>
__device__ __forceinline__ T from_raw(raw_t<T> x) {
    if constexpr (sizeof(T) == 2) return __builtin_bit_cast(T, static_cast<unsigned short>(x));
    else return x;
}

// acc + x rounded to T and widened again. bf16: rounding into the upper half of a register whose lower half is zero is the
// widened value already, one instruction less in the chain.
template <typename T>
__device__ __forceinline__ float add_rounded(float acc, T x) {
    if constexpr (std::is_same_v<T, bf16_t>)
        return __builtin_bit_cast(float, __builtin_convertvector(vec_t<float, 2>{0.0f, acc + to_f32(x)}, vec_t<bf16_t, 2>));
    else return round_to<T>(acc + to_f32(x));
}

template <typename T, bool Vector>
struct LongRow {
    static constexpr unsigned int kBatch = Vector ? (sizeof(T) == 2 ? 128 : 96) : 64;  // token rows per step
    static constexpr unsigned int kReadAhead = Vector ? 16 : 8;  // of them that the first wavefront reads from LDS ahead of its chain
    static constexpr unsigned int kVec = Vector ? kVec128<T> : 1;  // elements of a load
    static constexpr unsigned int kChunks = kSlice / kVec;
    static constexpr unsigned int kRows = kThreads / kChunks;                   // token rows of a load by all threads
    static constexpr unsigned int kPerThread = kBatch / kRows;
    static constexpr int kWavesPerSimd = Vector ? (sizeof(T) == 2 ? 5 : 4) : 6;  // that the launch keeps in flight
    struct Shared {
        union {
            alignas(16) T rows[kBatch][kSlice];
            alignas(16) unsigned int words[kSpan / 32];  // until the list is there
        };
        unsigned short list[kList];  // token positions, ascending, relative to the window's start
        unsigned int wave_counts[kWavesPerBlock];
        unsigned int long_ids[kThreads], wave_longs[kWavesPerBlock];
    };
    static_assert(kThreads == 4 * kWave && sizeof(Shared) <= 160 * 1024 / kWavesPerSimd, "a workgroup is one wavefront per SIMD");
};

template <typename T, bool Vector>
__device__ __forceinline__ void embedding_long_row(typename LongRow<T, Vector>::Shared& lds, T* __restrict__ row,
                                                   const T* __restrict__ grad_output, const unsigned int* __restrict__ segment,
                                                   unsigned int tokens, unsigned int count, unsigned int col0,
                                                   unsigned int hidden, bool accumulate) {
    using L = LongRow<T, Vector>;
    using chunk_t = vec_t<T, static_cast<int>(L::kVec)>;
    using u32x4 = vec_t<unsigned int, 4>;
    constexpr unsigned int kWords = kSpan / 32 / kThreads;  // bitmap words of a thread
    static_assert(kWords % 4 == 0 && kThreads / kWave == kWavesPerBlock, "a thread owns whole 16-byte pieces of the bitmap");
    unsigned int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));  // what follows from it is computed per item, not held in registers over all of them
    const unsigned int lane = tid & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const unsigned int col = col0 + lane;
    // Of a load's rows and chunks this thread takes row `mine` and the chunk at `column`.
    const unsigned int mine = tid / L::kChunks, column = col0 + tid % L::kChunks * L::kVec;
    float acc = 0.0f;
    if (wave == 0 && accumulate && col < hidden) acc = to_f32(row[col]);
    for (unsigned int base = 0; base < count; base += kSpan) {
        // The window's tokens of this segment: a bit per position.
#pragma unroll
        for (unsigned int i = 0; i < kWords; i += 4) *reinterpret_cast<u32x4*>(&lds.words[tid * kWords + i]) = u32x4(0u);
        __syncthreads();
        for (unsigned int i0 = 0; i0 < tokens; i0 += 4 * kThreads) {
            unsigned int position[4];  // four loads in flight, none behind a branch
#pragma unroll
            for (unsigned int u = 0; u < 4; ++u)
                position[u] = (segment[min(i0 + u * kThreads + tid, tokens - 1)] & ~kLong) - base;  // wraps below the window
#pragma unroll
            for (unsigned int u = 0; u < 4; ++u)
                if (i0 + u * kThreads + tid < tokens && position[u] < kSpan) atomicOr(&lds.words[position[u] / 32], 1u << (position[u] % 32));
        }
        __syncthreads();
        unsigned int word[kWords], found = 0;
#pragma unroll
        for (unsigned int i = 0; i < kWords; i += 4) {
            const u32x4 four = *reinterpret_cast<const u32x4*>(&lds.words[tid * kWords + i]);
#pragma unroll
            for (unsigned int e = 0; e < 4; ++e) found += __popc(word[i + e] = four[e]);
        }
        unsigned int inclusive = found;
#pragma unroll
        for (int offset = 1; offset < kWave; offset <<= 1) {
            const unsigned int other = __shfl_up(inclusive, offset, kWave);
            if (lane >= static_cast<unsigned int>(offset)) inclusive += other;
        }
        if (lane == kWave - 1) lds.wave_counts[wave] = inclusive;
        __syncthreads();
        unsigned int slot = inclusive - found, window = 0;
        for (unsigned int w = 0; w < kWavesPerBlock; ++w) {
            if (w < wave) slot += lds.wave_counts[w];
            window += lds.wave_counts[w];
        }
        window = __builtin_amdgcn_readfirstlane(window);  // the same in all lanes: what follows branches without masks
        for (unsigned int listed = 0; listed < window; listed += kList) {
            // The next kList of them in ascending order.
            const unsigned int entries = min(kList, window - listed);
#pragma unroll
            for (unsigned int i = 0; i < kWords; ++i) {
                while (word[i] != 0 && slot < listed + kList) {
                    lds.list[slot++ - listed] = static_cast<unsigned short>((tid * kWords + i) * 32 + __builtin_ctz(word[i]));
                    word[i] &= word[i] - 1;
                }
            }
            __syncthreads();
            // The batch that starts at list entry `first`, into registers. The loads carry no condition (past the end they
            // read the last entry's row and the last columns): a branch around each would make it wait for the one before.
            chunk_t held[L::kPerThread];
            auto fetch = [&](unsigned int first) __attribute__((always_inline)) {
                unsigned int token[L::kPerThread];
#pragma unroll
                for (unsigned int u = 0; u < L::kPerThread; ++u)
                    token[u] = base + lds.list[min(first + u * L::kRows + mine, entries - 1)];
#pragma unroll
                for (unsigned int u = 0; u < L::kPerThread; ++u) {
                    const T* at = grad_output + static_cast<std::size_t>(token[u]) * hidden;
                    held[u] = load_vec<T, static_cast<int>(L::kVec)>(at + min(column, hidden - L::kVec));
                }
            };
            fetch(0);
            for (unsigned int first = 0; first < entries; first += L::kBatch) {
#pragma unroll
                for (unsigned int u = 0; u < L::kPerThread; ++u)
                    store_vec<T, static_cast<int>(L::kVec)>(&lds.rows[u * L::kRows + mine][column - col0], held[u]);
                __syncthreads();
                fetch(first + L::kBatch);
                if (wave == 0) {
                    const unsigned int n = min(L::kBatch, entries - first);
                    raw_t<T> even[L::kReadAhead], odd[L::kReadAhead];
                    auto read = [&](raw_t<T>(&dy)[L::kReadAhead], unsigned int j) __attribute__((always_inline)) {
                        const unsigned int from = min(j, L::kBatch - L::kReadAhead);
#pragma unroll
                        for (unsigned int u = 0; u < L::kReadAhead; ++u) dy[u] = to_raw<T>(lds.rows[from + u][lane]);
                        __builtin_amdgcn_sched_barrier(0);  // the reads stay ahead of the additions that do not need them
                    };
                    auto add = [&](const raw_t<T>(&dy)[L::kReadAhead]) __attribute__((always_inline)) {
#pragma unroll
                        for (unsigned int u = 0; u < L::kReadAhead; ++u) acc = add_rounded<T>(acc, from_raw<T>(dy[u]));
                        __builtin_amdgcn_sched_barrier(0);
                    };
                    unsigned int j = 0;
                    read(even, 0);
                    for (; j + 2 * L::kReadAhead <= n; j += 2 * L::kReadAhead) {
                        read(odd, j + L::kReadAhead);
                        add(even);
                        read(even, j + 2 * L::kReadAhead);
                        add(odd);
                    }
                    if (j < n) {  // the last batch's last rows
                        if (j + L::kReadAhead <= n) {
                            read(odd, j + L::kReadAhead);
                            add(even);
#pragma unroll
                            for (unsigned int u = 0; u < L::kReadAhead; ++u) even[u] = odd[u];
                            j += L::kReadAhead;
                        }
#pragma unroll
                        for (unsigned int u = 0; u < L::kReadAhead; ++u)
                            if (j + u < n) acc = add_rounded<T>(acc, from_raw<T>(even[u]));
                    }
                }
                __syncthreads();
            }
        }
    }
    if (wave == 0 && col < hidden) row[col] = from_f32<T>(acc);
}

// Tokens of an id's segment; *begin: where it starts in `order`.
__device__ __forceinline__ unsigned int segment_of(const unsigned int* __restrict__ offsets, unsigned int id, unsigned int* begin) {
    *begin = offsets[id] & ~kLong;
    return (offsets[id + 1] & ~kLong) - *begin;
}

// Workgroups [0, long_groups): long segments. Each lists the long ids itself, one mark per thread at a time, and takes every
// long_groups-th (id, slice) of the list: a workgroup for every mark and slice would mostly find that there is nothing to do.
// The remaining ones are wavefronts [0, row_waves) for the ids below row_waves and the ids row_waves further on; they leave
// the long ones out.
template <typename T, bool Vector>
__global__ __launch_bounds__(kThreads, (LongRow<T, Vector>::kWavesPerSimd)) void embedding_rows_kernel(
                                                                    T* __restrict__ grad_weight,
                                                                    const T* __restrict__ grad_output,
                                                                    const std::uint32_t* __restrict__ ids,
                                                                    const unsigned int* __restrict__ offsets,
                                                                    const unsigned int* __restrict__ order,
                                                                    unsigned int count, unsigned int vocab,
                                                                    unsigned int hidden, unsigned int slices,
                                                                    unsigned int long_groups, unsigned int ids_per_group, unsigned int row_waves,
                                                                    bool accumulate) {
    if (blockIdx.x < long_groups) {
        __shared__ typename LongRow<T, Vector>::Shared lds;
        const unsigned int tid = threadIdx.x, wave = tid / kWave;
        if (count > kThreads * kShort) {  // fewer tokens: one look at the marks says as much
            bool any_long = false;
            for (unsigned int group = tid; group < (vocab + ids_per_group - 1) / ids_per_group; group += kThreads)
                any_long = any_long || (offsets[group * ids_per_group] & kLong) != 0;
            if (!__syncthreads_or(any_long)) return;
        }
        const unsigned int placed = offsets[vocab];  // ids past the vocabulary have no place in `order`
        unsigned int next_item = blockIdx.x;  // among the items of the marks from `first` on
        for (unsigned int first = 0; first * kShort < count; first += kThreads) {
            const unsigned int position = (first + tid) * kShort;
            const unsigned int token = position < count ? order[position] : 0;  // read beside `placed`, not after it
            unsigned int id = 0;
            bool is_long = position < placed && (token & kLong) != 0;
            if (is_long) {  // the segment's first mark names it
                id = ids[token & ~kLong];
                is_long = position - (offsets[id] & ~kLong) < kShort;
            }
            const unsigned long long mask = __ballot(is_long);
            if ((tid & (kWave - 1)) == 0) lds.wave_longs[wave] = __popcll(mask);
            __syncthreads();
            unsigned int slot = __popcll(mask & ((1ull << (tid & (kWave - 1))) - 1)), found = 0;
            for (unsigned int w = 0; w < kWavesPerBlock; ++w) {
                if (w < wave) slot += lds.wave_longs[w];
                found += lds.wave_longs[w];
            }
            found = __builtin_amdgcn_readfirstlane(found);
            if (is_long) lds.long_ids[slot] = id;
            __syncthreads();
            const unsigned int items = found * slices;
            for (; next_item < items; next_item += long_groups) {
                const unsigned int entry = next_item / slices, row = __builtin_amdgcn_readfirstlane(lds.long_ids[entry]);
                unsigned int begin;
                const unsigned int tokens = segment_of(offsets, row, &begin);
                embedding_long_row<T, Vector>(lds, grad_weight + static_cast<std::size_t>(row) * hidden, grad_output, order + begin,
                                              tokens, count, (next_item - entry * slices) * kSlice, hidden, accumulate);
            }
            next_item -= items;
            __syncthreads();  // the list is written again
        }
        return;
    }
    // The same for the whole wavefront, and known to be: the loads of a segment's rows then sit behind scalar branches, which
    // wait for nothing.
    const unsigned int first = (blockIdx.x - long_groups) * kWavesPerBlock + __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    if (first >= row_waves) return;
    const unsigned int lane = threadIdx.x & (kWave - 1), second = first + row_waves;
    unsigned int begin0, begin1 = 0;
    const unsigned int tokens0 = segment_of(offsets, first, &begin0);
    const unsigned int tokens1 = second < vocab ? segment_of(offsets, second, &begin1) : kShort + 1;
    const unsigned int mine0 = tokens0 <= kShort && lane < tokens0 ? order[begin0 + lane] : 0xFFFFFFFFu;
    const unsigned int mine1 = tokens1 <= kShort && lane < tokens1 ? order[begin1 + lane] : 0xFFFFFFFFu;
    if (tokens0 <= kShort)
        embedding_short_row<T, Vector>(grad_weight + static_cast<std::size_t>(first) * hidden, grad_output, mine0, tokens0, hidden, accumulate);
    if (tokens1 <= kShort)
        embedding_short_row<T, Vector>(grad_weight + static_cast<std::size_t>(second) * hidden, grad_output, mine1, tokens1, hidden, accumulate);
}

// The row of one token by a wavefront.
template <typename T, bool Vector>
__device__ __forceinline__ void gather_row(T* __restrict__ out, const std::uint32_t* __restrict__ ids, const T* __restrict__ weight,
                                           unsigned int token, unsigned int vocab, unsigned int hidden) {
    constexpr int VEC = Vector ? kVec128<T> : 1;
    const unsigned int lane = threadIdx.x & (kWave - 1);
    const std::uint32_t id = ids[token];
    T* dst = out + static_cast<std::size_t>(token) * hidden;
    if (id < vocab) {
        const T* src = weight + static_cast<std::size_t>(id) * hidden;
        for (unsigned int col = lane * VEC; col < hidden; col += kWave * VEC)
            store_vec<T, VEC>(dst + col, load_vec<T, VEC>(src + col));
    } else {
        for (unsigned int col = lane * VEC; col < hidden; col += kWave * VEC)
            store_vec<T, VEC>(dst + col, vec_t<T, VEC>(0));
    }
}

template <typename T, bool Vector>
__global__ __launch_bounds__(kThreads) void embedding_gather_kernel(T* __restrict__ out,
                                                                   const std::uint32_t* __restrict__ ids,
                                                                   const T* __restrict__ weight, unsigned int count,
                                                                   unsigned int vocab, unsigned int hidden) {
    const unsigned int token = blockIdx.x * kWavesPerBlock + threadIdx.x / kWave;
    if (token < count) gather_row<T, Vector>(out, ids, weight, token, vocab, hidden);
}

// The first `groups` workgroups group the ids, the others look their rows up, 16 tokens each.
template <typename T, bool Vector>
__global__ __launch_bounds__(kGroupThreads) void embedding_gather_and_group_kernel(GroupArgs g, unsigned int groups, T* __restrict__ out,
                                                                                  const T* __restrict__ weight, unsigned int hidden) {
    extern __shared__ unsigned int bins[];
    if (blockIdx.x < groups) {
        group_ids(g, bins);
        return;
    }
    const unsigned int token = (blockIdx.x - groups) * (kGroupThreads / kWave) + threadIdx.x / kWave;
    if (token < g.count) gather_row<T, Vector>(out, g.ids, weight, token, g.vocab, hidden);
}

// Scratch: offsets[vocab + 1] | order[token_count].
std::size_t offsets_bytes(std::size_t vocab) { return ((vocab + 1) * sizeof(unsigned int) + 255) & ~std::size_t{255}; }

// How a list of tokens is grouped: arguments, workgroups and their LDS.
struct Grouping {
    GroupArgs args;
    unsigned int groups;
    std::size_t lds;
};
Grouping plan_grouping(void* mem, const std::uint32_t* token_ids, std::size_t token_count, std::size_t vocab) {
    const auto v = static_cast<unsigned int>(vocab);
    // Ranges of a power of two of ids, at most one workgroup per compute unit, each histogram within the LDS.
    unsigned int ids_per_group = kGroupMinIds, token_bits = 25;
    const unsigned int units = static_cast<unsigned int>(compute_units());
    while (ids_per_group < kGroupMaxIds && (v + ids_per_group - 1) / ids_per_group > units) ids_per_group *= 2, --token_bits;
    static_assert(kGroupMinIds == 1u << (32 - 25), "an entry of a list is an id's place in its range above a token");
    // A wavefront's list: room for all the tokens that it may see, as far as the LDS goes.
    constexpr std::size_t kWaves = kGroupThreads / kWave;
    const std::size_t bins_bytes = ids_per_group * sizeof(unsigned int);
    const std::size_t seen = (token_count + 4 * kGroupThreads - 1) / (4 * kGroupThreads) * (4 * kWave);
    const std::size_t list_entries = token_count > std::size_t{1} << token_bits
                                         ? 0
                                         : std::min(seen, (kGroupLds - bins_bytes) / (kWaves * sizeof(unsigned int)));
    Grouping g{};
    g.args = {static_cast<unsigned int*>(mem), reinterpret_cast<unsigned int*>(static_cast<char*>(mem) + offsets_bytes(vocab)), token_ids,
              static_cast<unsigned int>(token_count), v, ids_per_group, token_bits, static_cast<unsigned int>(list_entries), is_aligned16(token_ids)};
    g.groups = (v + ids_per_group - 1) / ids_per_group;
    g.lds = bins_bytes + kWaves * list_entries * sizeof(unsigned int);
    return g;
}

std::size_t groups_bytes(std::size_t token_count, std::size_t vocab) { return offsets_bytes(vocab) + token_count * sizeof(unsigned int); }

}  // namespace

std::size_t embedding_groups_ahead_bytes(std::size_t token_count, std::size_t vocab) {
    // Up to the tokens whose lists leave a CU room for a second workgroup. With the mean loss taken beside the norms' reductions and the
    // logits' gradient written in the rows that its contractions read, four launches less: 3 x 100 tokens, 5003 ids 233.3 -> 225.2 us.
    constexpr std::size_t kMostTokens = 8192, kMostLds = 48 * 1024;
    if (token_count == 0 || token_count > kMostTokens || vocab == 0 || vocab > static_cast<std::size_t>(std::numeric_limits<int>::max())) return 0;
    return plan_grouping(nullptr, nullptr, token_count, vocab).lds <= kMostLds ? groups_bytes(token_count, vocab) : 0;
}

int embedding_forward_and_group(void* output, const std::uint32_t* token_ids, std::size_t token_count, const void* weight, std::size_t vocab,
                                std::size_t hidden, void* groups, int dtype, hipStream_t stream, bool* grouped) {
    *grouped = false;
    if (groups != nullptr && valid_dtype(dtype) && output != nullptr && weight != nullptr && token_ids != nullptr && hidden != 0 &&
        embedding_groups_ahead_bytes(token_count, vocab) != 0) {
        const Grouping g = plan_grouping(groups, token_ids, token_count, vocab);
        const unsigned int blocks = g.groups + (g.args.count + kGroupThreads / kWave - 1) / (kGroupThreads / kWave);
        *grouped = true;
        return dispatch_dtype(dtype, [&]<typename T>() -> int {
            auto* out = static_cast<T*>(output);
            auto* w = static_cast<const T*>(weight);
            const bool vector_ok = hidden % kVec128<T> == 0 && is_aligned16(out) && is_aligned16(w);
            auto kernel = vector_ok ? embedding_gather_and_group_kernel<T, true> : embedding_gather_and_group_kernel<T, false>;
            hipLaunchKernelGGL(kernel, dim3(blocks), dim3(kGroupThreads), g.lds, stream, g.args, g.groups, out, w,
                               static_cast<unsigned int>(hidden));
            CGPTX_LAUNCH_CHECK();
            return CGPTX_OK;
        });
    }
    return cgptx_embedding_forward(output, token_ids, token_count, weight, vocab, hidden, dtype, stream);
}

int embedding_backward_grouped(void* grad_weight, const void* grad_output, const std::uint32_t* token_ids, std::size_t token_count,
                               std::size_t vocab, std::size_t hidden, int accumulate_weight, void* groups, int dtype, hipStream_t stream) {
    const char* name = "embedding_backward";
    if (!valid_dtype(dtype)) return fail(CGPTX_INVALID_ARGUMENT, std::string(name) + ": unsupported dtype");
    if (grad_weight == nullptr || grad_output == nullptr || token_ids == nullptr || token_count == 0 || vocab == 0 ||
        hidden == 0)
        return fail(CGPTX_INVALID_ARGUMENT, std::string(name) + ": incompatible tensors or token count");
    constexpr std::size_t u32max = std::numeric_limits<std::uint32_t>::max();
    if (token_count >= u32max / 2 || vocab >= u32max || hidden > u32max)
        return fail(CGPTX_OVERFLOW, std::string(name) + ": dimension exceeds uint32_t range");
    const auto count = static_cast<unsigned int>(token_count);
    const auto v = static_cast<unsigned int>(vocab);
    void* mem = groups;
    if (groups == nullptr)
        if (int s = scratch(stream, groups_bytes(token_count, vocab), &mem)) return s;
    const Grouping g = plan_grouping(mem, token_ids, token_count, vocab);
    unsigned int *const offsets = g.args.offsets, *const order = g.args.order;
    const unsigned int ids_per_group = g.args.ids_per_group;
    if (groups == nullptr) {
        static bool configured = false;
        if (!configured) {
            CGPTX_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(embedding_group_kernel),
                                          hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(kGroupLds)));
            configured = true;
        }
        hipLaunchKernelGGL(embedding_group_kernel, dim3(g.groups), dim3(kGroupThreads), g.lds, stream, g.args);
        CGPTX_LAUNCH_CHECK();
    }
    return dispatch_dtype(dtype, [&]<typename T>() -> int {
        auto* dw = static_cast<T*>(grad_weight);
        auto* dy = static_cast<const T*>(grad_output);
        const bool vector_ok = hidden % kVec128<T> == 0 && is_aligned16(dw) && is_aligned16(dy);
        const auto h = static_cast<unsigned int>(hidden);
        // Long segments: at most one per kShort + 1 tokens, each with a workgroup per slice of the columns, up to what the
        // chip holds at a time.
        const std::size_t slices = (hidden + kSlice - 1) / kSlice;
        const std::size_t long_groups =
            std::min<std::size_t>(token_count / (kShort + 1) * slices, static_cast<std::size_t>(compute_units()) * 4);
        // Two ids a wavefront unless one each find a place on the chip together (300 tokens over 1000 ids: 7.9 us, with two 8.6;
        // 2048 over 32000: 16.8, with one 17.6).
        const std::size_t row_waves = vocab <= static_cast<std::size_t>(compute_units()) * 16 ? vocab : (vocab + 1) / 2;
        const std::size_t short_groups = (row_waves + kWavesPerBlock - 1) / kWavesPerBlock;
        if (long_groups + short_groups > static_cast<std::size_t>(std::numeric_limits<int>::max()))
            return fail(CGPTX_OVERFLOW, std::string(name) + ": too many workgroups");
        const dim3 grid(static_cast<unsigned int>(long_groups + short_groups));
        auto kernel = vector_ok ? embedding_rows_kernel<T, true> : embedding_rows_kernel<T, false>;
        hipLaunchKernelGGL(kernel, grid, dim3(kThreads), 0, stream, dw, dy, token_ids, offsets, order, count, v, h,
                           static_cast<unsigned int>(slices), static_cast<unsigned int>(long_groups), ids_per_group,
                           static_cast<unsigned int>(row_waves), accumulate_weight != 0);
        CGPTX_LAUNCH_CHECK();
        return CGPTX_OK;
    });
}

}  // namespace cgptx

extern "C" int cgptx_embedding_backward(void* grad_weight, const void* grad_output, const uint32_t* token_ids,
                                        size_t token_count, size_t vocab, size_t hidden, int bounds_check,
                                        int accumulate_weight, int dtype, cgptx_stream stream) {
    (void)bounds_check;  // out-of-range ids are skipped either way
    return cgptx::embedding_backward_grouped(grad_weight, grad_output, token_ids, token_count, vocab, hidden, accumulate_weight, nullptr,
                                             dtype, static_cast<hipStream_t>(stream));
}

extern "C" int cgptx_embedding_forward(void* output, const uint32_t* token_ids, size_t token_count,
                                       const void* weight, size_t vocab, size_t hidden, int dtype,
                                       cgptx_stream stream_) {
    using namespace cgptx;
    const char* name = "embedding_forward";
    if (!valid_dtype(dtype)) return fail(CGPTX_INVALID_ARGUMENT, std::string(name) + ": unsupported dtype");
    if (output == nullptr || weight == nullptr || token_ids == nullptr || token_count == 0 || vocab == 0 || hidden == 0)
        return fail(CGPTX_INVALID_ARGUMENT, std::string(name) + ": incompatible tensors or token count");
    constexpr std::size_t u32max = std::numeric_limits<std::uint32_t>::max();
    if (token_count >= u32max || vocab >= u32max || hidden > u32max)
        return fail(CGPTX_OVERFLOW, std::string(name) + ": dimension exceeds uint32_t range");
    auto stream = static_cast<hipStream_t>(stream_);
    const auto count = static_cast<unsigned int>(token_count);
    return dispatch_dtype(dtype, [&]<typename T>() -> int {
        auto* out = static_cast<T*>(output);
        auto* w = static_cast<const T*>(weight);
        const bool vector_ok = hidden % kVec128<T> == 0 && is_aligned16(out) && is_aligned16(w);
        const dim3 grid((count + kWavesPerBlock - 1) / kWavesPerBlock);
        if (vector_ok) {
            hipLaunchKernelGGL((embedding_gather_kernel<T, true>), grid, dim3(kThreads), 0, stream, out, token_ids, w,
                               count, static_cast<unsigned int>(vocab), static_cast<unsigned int>(hidden));
        } else {
            hipLaunchKernelGGL((embedding_gather_kernel<T, false>), grid, dim3(kThreads), 0, stream, out, token_ids,
                               w, count, static_cast<unsigned int>(vocab), static_cast<unsigned int>(hidden));
        }
        CGPTX_LAUNCH_CHECK();
        return CGPTX_OK;
    });
}
