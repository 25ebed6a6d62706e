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
// Workgroup b owns the ids [b R, (b+1) R) and reads the whole id list twice: first it counts its ids in an
// LDS histogram and, on the side, the tokens with smaller ids (which is where its part of the output begins:
// no workgroup waits for another); after an exclusive scan of the histogram it hands every token of its range
// the next free slot of its id's segment. Slots are handed out with LDS integer atomics, so the order inside a
// segment is whatever order the lanes arrived in: the row kernel puts each segment into ascending order itself.
// offsets[id] .. offsets[id + 1] is id's segment of `order`; ids >= vocab belong to nobody and are skipped.
constexpr int kGroupThreads = 1024;
constexpr unsigned int kGroupMaxIds = 32768;  // LDS histogram entries of one workgroup (128 KiB)
constexpr int kGroupBatch = 8;                // 128-bit id loads a thread keeps in flight

// The id list is walked in batches of kGroupBatch x 4 ids per thread, all of a batch's loads requested before the
// first id is looked at (one dependent load per id would cost a memory round trip each). visit(id, t) sees every
// token once; the order within a workgroup does not matter to any caller.
template <typename Visit>
__device__ __forceinline__ void for_each_id(const std::uint32_t* __restrict__ ids, unsigned int count, bool aligned, Visit&& visit) {
    using u32x4 = vec_t<unsigned int, 4>;
    const unsigned int quads = aligned ? count / 4 : 0;
    const auto* wide = reinterpret_cast<const u32x4*>(ids);
    for (unsigned int base = 0; base < quads; base += kGroupBatch * kGroupThreads) {
        u32x4 held[kGroupBatch];
#pragma unroll
        for (int k = 0; k < kGroupBatch; ++k) {
            const unsigned int q = base + k * kGroupThreads + threadIdx.x;
            if (q < quads) held[k] = wide[q];
        }
#pragma unroll
        for (int k = 0; k < kGroupBatch; ++k) {
            const unsigned int q = base + k * kGroupThreads + threadIdx.x;
            if (q < quads) {
#pragma unroll
                for (int e = 0; e < 4; ++e) visit(held[k][e], 4 * q + e);
            }
        }
    }
    for (unsigned int t = 4 * quads + threadIdx.x; t < count; t += kGroupThreads) visit(ids[t], t);
}

__global__ __launch_bounds__(kGroupThreads) void embedding_group_kernel(unsigned int* __restrict__ offsets,
                                                                       unsigned int* __restrict__ order,
                                                                       const std::uint32_t* __restrict__ ids,
                                                                       unsigned int count, unsigned int vocab,
                                                                       unsigned int ids_per_group, bool aligned) {
    extern __shared__ unsigned int bins[];  // [ids_per_group]
    __shared__ unsigned int wave_totals[kGroupThreads / kWave];
    __shared__ unsigned int smaller_total;
    const unsigned int lo = blockIdx.x * ids_per_group;
    const unsigned int width = min(ids_per_group, vocab - lo);
    const unsigned int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave;
    for (unsigned int i = tid; i < width; i += kGroupThreads) bins[i] = 0;
    if (tid == 0) smaller_total = 0;
    __syncthreads();
    unsigned int smaller = 0;
    for_each_id(ids, count, aligned, [&](unsigned int id, unsigned int) {
        if (id < lo) ++smaller;
        else if (id - lo < width) atomicAdd(&bins[id - lo], 1u);
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
    for (unsigned int i = first; i < last; ++i) mine += bins[i];
    unsigned int inclusive = mine;
#pragma unroll
    for (int offset = 1; offset < kWave; offset <<= 1) {
        const unsigned int other = __shfl_up(inclusive, offset, kWave);
        if (lane >= static_cast<unsigned int>(offset)) inclusive += other;
    }
    if (lane == kWave - 1) wave_totals[wave] = inclusive;
    __syncthreads();
    unsigned int before = smaller_total;
    for (unsigned int w = 0; w < wave; ++w) before += wave_totals[w];
    unsigned int running = before + inclusive - mine;
    for (unsigned int i = first; i < last; ++i) {
        const unsigned int n = bins[i];
        bins[i] = running;
        offsets[lo + i] = running;
        running += n;
    }
    if (lo + width == vocab && tid == kGroupThreads - 1) offsets[vocab] = running;  // the piece that ends the last range
    __syncthreads();
    for_each_id(ids, count, aligned, [&](unsigned int id, unsigned int t) {
        if (id >= lo && id - lo < width) order[atomicAdd(&bins[id - lo], 1u)] = t;
    });
}

// ---- rows ------------------------------------------------------------------------------------------
// Adds, into row `id` of the table, the rows of grad_output of the tokens with that id, in ascending token
// order with one rounding to the storage dtype per add. Rows without tokens are zero-filled unless the gradient
// is accumulated. Bound by HBM (three rows per token) as long as the serial chain of additions of the most
// frequent id is short; text makes it long: the first ids of a vocabulary take several per cent of a batch each.
//   * Segments of up to kShort tokens: one wavefront per id, tokens ordered in registers (lane i holds the token
//     of rank i), lanes across the columns, kAhead token rows in flight.
//   * Longer ones: one workgroup per id and kSlice columns, so that a frequent id occupies hidden / kSlice
//     workgroups instead of one wavefront. The segment is put into ascending order through a bitmap of token
//     positions in LDS, kSpan positions at a time, from which the list of the next kList tokens is drawn as often as it
//     takes; all threads fetch the slices of the next kBatch token rows while the first wavefront adds the previous
//     ones, one column per lane, from LDS, where it reads 16 tokens ahead of the chain. That is bound by the latency
//     of add + round. A segment is read once per kSpan tokens of the batch, so its work grows with its tokens up to batches
//     of millions.
// Both live in one launch, the long segments' workgroups first. 32768 tokens x 1024 columns, ids Zipf distributed
// over 32000: 1846 -> 51 us (of which the most frequent id, 6.7 per cent of the tokens, sets the end).
constexpr unsigned int kShort = 64;      // tokens: one lane each
constexpr unsigned int kSlice = 64;      // columns of a long segment's workgroup: one lane each, one or two cache lines
constexpr unsigned int kBatch = 128;     // token rows per step of a long segment
constexpr unsigned int kSpan = 65536;    // token positions covered by the bitmap at a time
constexpr unsigned int kList = 4096;     // tokens ordered at a time

template <typename T, bool Vector>
__device__ __forceinline__ void embedding_short_row(T* __restrict__ row, const T* __restrict__ grad_output,
                                                    const unsigned int* __restrict__ segment, unsigned int tokens,
                                                    unsigned int hidden, bool accumulate) {
    constexpr int VEC = Vector ? kVec128<T> : 1;
    constexpr unsigned int kAhead = 8;
    using vec_f = vec_t<float, VEC>;
    const unsigned int lane = threadIdx.x & (kWave - 1);
    if (tokens == 0) {
        if (!accumulate)
            for (unsigned int col = lane * VEC; col < hidden; col += kWave * VEC) store_vec<T, VEC>(row + col, vec_t<T, VEC>(0));
        return;
    }
    const unsigned int mine = lane < tokens ? segment[lane] : 0xFFFFFFFFu;
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
    static constexpr unsigned int kVec = Vector ? kVec128<T> : 1;
    static constexpr unsigned int kChunks = kSlice / kVec;                    // loads per token and slice
    static constexpr unsigned int kPerThread = kBatch * kChunks / kThreads;   // loads per thread and batch
    struct Shared {
        alignas(16) T rows[kBatch][kSlice];
        alignas(16) unsigned int words[kSpan / 32];
        unsigned short list[kList];              // token positions of the window, ascending, relative to its start
        unsigned int wave_counts[kWavesPerBlock];
    };
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
    const unsigned int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave;
    const unsigned int col = col0 + lane;
    float acc = 0.0f;
    if (wave == 0 && accumulate && col < hidden) acc = to_f32(row[col]);
    for (unsigned int base = 0; base < count; base += kSpan) {
        // The window's tokens of this segment: a bit per position.
#pragma unroll
        for (unsigned int i = 0; i < kWords; i += 4) *reinterpret_cast<u32x4*>(&lds.words[tid * kWords + i]) = u32x4(0u);
        __syncthreads();
        for (unsigned int i = tid; i < tokens; i += kThreads) {
            const unsigned int position = segment[i] - base;  // wraps below the window
            if (position < kSpan) atomicOr(&lds.words[position / 32], 1u << (position % 32));
        }
        __syncthreads();
        unsigned int word[kWords], mine = 0;
#pragma unroll
        for (unsigned int i = 0; i < kWords; i += 4) {
            const u32x4 four = *reinterpret_cast<const u32x4*>(&lds.words[tid * kWords + i]);
#pragma unroll
            for (unsigned int e = 0; e < 4; ++e) mine += __popc(word[i + e] = four[e]);
        }
        unsigned int inclusive = mine;
#pragma unroll
        for (int offset = 1; offset < kWave; offset <<= 1) {
            const unsigned int other = __shfl_up(inclusive, offset, kWave);
            if (lane >= static_cast<unsigned int>(offset)) inclusive += other;
        }
        if (lane == kWave - 1) lds.wave_counts[wave] = inclusive;
        __syncthreads();
        unsigned int slot = inclusive - mine, window = 0;
        for (unsigned int w = 0; w < kWavesPerBlock; ++w) {
            if (w < wave) slot += lds.wave_counts[w];
            window += lds.wave_counts[w];
        }
        for (unsigned int listed = 0; listed < window; listed += kList) {
            // The next kList of them in ascending order.
            const unsigned int found = min(kList, window - listed);
#pragma unroll
            for (unsigned int i = 0; i < kWords; ++i) {
                while (word[i] != 0 && slot < listed + kList) {
                    lds.list[slot++ - listed] = static_cast<unsigned short>((tid * kWords + i) * 32 + __builtin_ctz(word[i]));
                    word[i] &= word[i] - 1;
                }
            }
            __syncthreads();
            // Loads of the batch that starts at list entry `first`, into registers.
            chunk_t held[L::kPerThread];
            auto fetch = [&](unsigned int first) {
#pragma unroll
                for (unsigned int u = 0; u < L::kPerThread; ++u) {
                    const unsigned int index = u * kThreads + tid;
                    const unsigned int entry = first + index / L::kChunks, column = col0 + index % L::kChunks * L::kVec;
                    if (entry < found && column < hidden)
                        held[u] = load_vec<T, static_cast<int>(L::kVec)>(
                            grad_output + static_cast<std::size_t>(base + lds.list[entry]) * hidden + column);
                }
            };
            fetch(0);
            for (unsigned int first = 0; first < found; first += kBatch) {
#pragma unroll
                for (unsigned int u = 0; u < L::kPerThread; ++u) {
                    const unsigned int index = u * kThreads + tid;
                    store_vec<T, static_cast<int>(L::kVec)>(&lds.rows[index / L::kChunks][index % L::kChunks * L::kVec], held[u]);
                }
                __syncthreads();
                if (first + kBatch < found) fetch(first + kBatch);
                if (wave == 0) {
                    const unsigned int n = min(kBatch, found - first);
                    T even[16], odd[16];
                    auto read = [&](T(&dy)[16], unsigned int j) {
                        const unsigned int from = min(j, kBatch - 16);
#pragma unroll
                        for (unsigned int u = 0; u < 16; ++u) dy[u] = lds.rows[from + u][lane];
                    };
                    auto add = [&](const T(&dy)[16], unsigned int j) {
                        if (j + 16 <= n) {
#pragma unroll
                            for (unsigned int u = 0; u < 16; ++u) acc = add_rounded<T>(acc, dy[u]);
                        } else {
#pragma unroll
                            for (unsigned int u = 0; u < 16; ++u)
                                if (j + u < n) acc = add_rounded<T>(acc, dy[u]);
                        }
                    };
                    read(even, 0);
                    for (unsigned int j = 0; j < n; j += 32) {
                        read(odd, j + 16);
                        add(even, j);
                        read(even, j + 32);
                        add(odd, j + 16);
                    }
                }
                __syncthreads();
            }
        }
    }
    if (wave == 0 && col < hidden) row[col] = from_f32<T>(acc);
}

// Workgroups [0, long_groups): long segments. A segment of more than kShort = 64 tokens contains a position of
// `order` that is a multiple of 64; the first one in it names the segment, so candidate j is the id of the token at
// position 64 j if that id's segment is long and 64 j its first multiple. Each of these workgroups lists the long
// ids itself, one candidate per thread at a time, and takes every long_groups-th (id, slice) of the list: a workgroup
// for every candidate and slice would mostly find that there is nothing to do, after four dependent loads
// (with the wider bitmap and the shorter chain 64 -> 51 us). The remaining workgroups take kWavesPerBlock ids each and leave the long ones out.
template <typename T, bool Vector>
__global__ __launch_bounds__(kThreads) void embedding_rows_kernel(T* __restrict__ grad_weight,
                                                                 const T* __restrict__ grad_output,
                                                                 const std::uint32_t* __restrict__ ids,
                                                                 const unsigned int* __restrict__ offsets,
                                                                 const unsigned int* __restrict__ order,
                                                                 unsigned int count, unsigned int vocab,
                                                                 unsigned int hidden, unsigned int slices,
                                                                 unsigned int long_groups, bool accumulate) {
    __shared__ typename LongRow<T, Vector>::Shared lds;
    __shared__ unsigned int long_ids[kThreads], wave_longs[kWavesPerBlock];
    if (blockIdx.x < long_groups) {
        const unsigned int tid = threadIdx.x, wave = tid / kWave;
        const unsigned int placed = offsets[vocab];  // ids past the vocabulary have no place in `order`
        const unsigned int candidates = (placed + kShort - 1) / kShort;
        unsigned int next_item = blockIdx.x;  // among the items of the candidates from `first` on
        for (unsigned int first = 0; first < candidates; first += kThreads) {
            const unsigned int position = (first + tid) * kShort;
            unsigned int id = 0;
            bool is_long = false;
            if (first + tid < candidates) {
                id = ids[order[position]];
                const unsigned int begin = offsets[id];
                is_long = offsets[id + 1] - begin > kShort && position - begin < kShort;
            }
            const unsigned long long mask = __ballot(is_long);
            if ((tid & (kWave - 1)) == 0) wave_longs[wave] = __popcll(mask);
            __syncthreads();
            unsigned int slot = __popcll(mask & ((1ull << (tid & (kWave - 1))) - 1)), found = 0;
            for (unsigned int w = 0; w < kWavesPerBlock; ++w) {
                if (w < wave) slot += wave_longs[w];
                found += wave_longs[w];
            }
            if (is_long) long_ids[slot] = id;
            __syncthreads();
            const unsigned int items = found * slices;
            for (; next_item < items; next_item += long_groups) {
                const unsigned int entry = next_item / slices, row = long_ids[entry];
                const unsigned int begin = offsets[row], tokens = offsets[row + 1] - begin;
                embedding_long_row<T, Vector>(lds, grad_weight + static_cast<std::size_t>(row) * hidden, grad_output, order + begin,
                                              tokens, count, (next_item - entry * slices) * kSlice, hidden, accumulate);
            }
            next_item -= items;
            __syncthreads();  // the list is written again
        }
        return;
    }
    const unsigned int id = (blockIdx.x - long_groups) * kWavesPerBlock + threadIdx.x / kWave;
    if (id >= vocab) return;
    const unsigned int begin = offsets[id], tokens = offsets[id + 1] - begin;
    if (tokens <= kShort)
        embedding_short_row<T, Vector>(grad_weight + static_cast<std::size_t>(id) * hidden, grad_output, order + begin, tokens,
                                       hidden, accumulate);
}

template <typename T, bool Vector>
__global__ __launch_bounds__(kThreads) void embedding_gather_kernel(T* __restrict__ out,
                                                                   const std::uint32_t* __restrict__ ids,
                                                                   const T* __restrict__ weight, unsigned int count,
                                                                   unsigned int vocab, unsigned int hidden) {
    constexpr int VEC = Vector ? kVec128<T> : 1;
    const unsigned int lane = threadIdx.x & (kWave - 1);
    const unsigned int token = blockIdx.x * kWavesPerBlock + threadIdx.x / kWave;
    if (token >= count) return;
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

}  // namespace
}  // namespace cgptx

extern "C" int cgptx_embedding_backward(void* grad_weight, const void* grad_output, const uint32_t* token_ids,
                                        size_t token_count, size_t vocab, size_t hidden, int bounds_check,
                                        int accumulate_weight, int dtype, cgptx_stream stream_) {
    using namespace cgptx;
    (void)bounds_check;  // out-of-range ids are skipped either way
    const char* name = "embedding_backward";
    if (!valid_dtype(dtype)) return fail(CGPTX_INVALID_ARGUMENT, std::string(name) + ": unsupported dtype");
    if (grad_weight == nullptr || grad_output == nullptr || token_ids == nullptr || token_count == 0 || vocab == 0 ||
        hidden == 0)
        return fail(CGPTX_INVALID_ARGUMENT, std::string(name) + ": incompatible tensors or token count");
    constexpr std::size_t u32max = std::numeric_limits<std::uint32_t>::max();
    if (token_count >= u32max / 2 || vocab >= u32max || hidden > u32max)
        return fail(CGPTX_OVERFLOW, std::string(name) + ": dimension exceeds uint32_t range");
    auto stream = static_cast<hipStream_t>(stream_);
    const auto count = static_cast<unsigned int>(token_count);
    const auto v = static_cast<unsigned int>(vocab);

    // Scratch: offsets[vocab + 1] | order[token_count].
    const std::size_t offsets_bytes = ((vocab + 1) * sizeof(unsigned int) + 255) & ~std::size_t{255};
    void* mem = nullptr;
    if (int s = scratch(stream, offsets_bytes + token_count * sizeof(unsigned int), &mem)) return s;
    auto* offsets = static_cast<unsigned int*>(mem);
    auto* order = reinterpret_cast<unsigned int*>(static_cast<char*>(mem) + offsets_bytes);
    // Ranges of at least 1024 ids, at most one workgroup per compute unit, each histogram within the LDS.
    unsigned int ids_per_group = 1024;
    const unsigned int units = static_cast<unsigned int>(compute_units());
    while (ids_per_group < kGroupMaxIds && (v + ids_per_group - 1) / ids_per_group > units) ids_per_group *= 2;
    const unsigned int groups = (v + ids_per_group - 1) / ids_per_group;
    const std::size_t group_lds = ids_per_group * sizeof(unsigned int);
    {
        static bool configured = false;
        if (!configured) {
            CGPTX_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(embedding_group_kernel),
                                          hipFuncAttributeMaxDynamicSharedMemorySize,
                                          static_cast<int>(kGroupMaxIds * sizeof(unsigned int))));
            configured = true;
        }
    }
    hipLaunchKernelGGL(embedding_group_kernel, dim3(groups), dim3(kGroupThreads), group_lds, stream, offsets, order, token_ids,
                       count, v, ids_per_group, is_aligned16(token_ids));
    CGPTX_LAUNCH_CHECK();
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
        const std::size_t short_groups = (vocab + kWavesPerBlock - 1) / kWavesPerBlock;
        if (long_groups + short_groups > static_cast<std::size_t>(std::numeric_limits<int>::max()))
            return fail(CGPTX_OVERFLOW, std::string(name) + ": too many workgroups");
        const dim3 grid(static_cast<unsigned int>(long_groups + short_groups));
        auto kernel = vector_ok ? embedding_rows_kernel<T, true> : embedding_rows_kernel<T, false>;
        hipLaunchKernelGGL(kernel, grid, dim3(kThreads), 0, stream, dw, dy, token_ids, offsets, order, count, v, h,
                           static_cast<unsigned int>(slices), static_cast<unsigned int>(long_groups), accumulate_weight != 0);
        CGPTX_LAUNCH_CHECK();
        return CGPTX_OK;
    });
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
