// Small contractions: K split between the wavefronts of a workgroup.
//
// C of at most a few hundred tiles (short sequences, narrow layers, the weight gradients of a small batch) leaves the
// persistent kernels of gemm.hip with little to do per K tile and a workgroup barrier around each: what such a call costs
// is the latency of its start and of its serial K loop. Here a workgroup owns one 64 x 64 or 32 x 32 tile and its four
// wavefronts take every fourth K tile each, the whole C tile of it: the loop is four times shorter and has no barrier,
// since a wavefront loads its K tiles into LDS stages of its own (global -> LDS) and waits for nobody. Fragments of the
// next K tile are read, and the loads of the one STAGES further issued, between the MFMAs of the present one. At the end
// the four partial tiles meet in LDS and are added in wavefront order. Same swizzled operand tiles and same edges (buffer
// range checks) as the persistent kernels.
//
// What bounds it: with few workgroups the latency of the loads, i.e. the K bytes of a workgroup over the bytes it keeps
// in flight (64 or 128 KiB), which is why short rows of tiles take 32 x 32 ones; with a full chip the L2's bandwidth
// (64 bytes per CU and cycle against 8 KiB per 16 MFMAs), where larger tiles win.
#pragma once

#include "gemm_small.hpp"
#include "gemm_tiles.hpp"

namespace cgptx {
namespace {

template <int COUNT>
__device__ __forceinline__ void wait_loads() {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(COUNT) : "memory");
}

__device__ __forceinline__ SegmentPick pick_small_segment(const SmallSegments& seg, int col) {
    KernelSegments s;
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        s.ptr[i] = seg.ptr[i];
        s.ld[i] = seg.ld[i];
        s.cols[i] = seg.cols[i];
    }
    s.count = seg.count;
    return pick_segment(s, col);
}

template <int TILE, bool DEEP>
constexpr int small_smem_bytes() { return DEEP ? 128 * 1024 : 64 * 1024; }

template <typename T, int TILE, bool DEEP, bool A_K, bool B_K, SmallEpilogue EPILOGUE, bool SEGMENTED>
__global__ __launch_bounds__(kThreads) void gemm_small_kernel(SmallArgs p) {
    using frag_t = typename Mfma<T>::frag;
    using ATile = std::conditional_t<A_K, KTile<T, TILE>, NTile<T, TILE>>;
    using BTile = std::conditional_t<B_K, KTile<T, TILE>, NTile<T, TILE>>;
    constexpr int kBlocks = TILE / 16;                  // 16 x 16 MFMA blocks along an edge
    constexpr int kOperandBytes = TILE * 64;            // 64 bytes along K per row, or the same bytes k-strided
    constexpr int kStageBytes = 2 * kOperandBytes;      // [A | B]
    constexpr int kLoadBytes = 1024, kOperandLoads = kOperandBytes / kLoadBytes, kLoads = 2 * kOperandLoads;
    constexpr int STAGES = small_smem_bytes<TILE, DEEP>() / (kWaves * kStageBytes);
    static_assert(STAGES >= 2 && STAGES * kLoads < 64, "the loads in flight are counted by vmcnt");
    extern __shared__ __align__(1024) unsigned char smem_raw[];
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);

    // Workgroups go to the XCDs round-robin, tile rows first: an XCD reads its share of A's panels and all of B.
    const int m0 = blockIdx.x * TILE, n0 = blockIdx.y * TILE, slice = blockIdx.z;
    const int kt_begin = slice * p.k_tiles_per_slice, kt_end = min(p.k_tiles, kt_begin + p.k_tiles_per_slice);
    const int steps = max(0, (kt_end - kt_begin - wave + kWaves - 1) / kWaves);  // K tiles kt_begin + wave + kWaves i

    // Sources. A in column segments: along K (k-contiguous) the segment is picked per K tile, along M once.
    ATile a_src;
    BTile b_src;
    if constexpr (A_K) {
        if (!SEGMENTED || p.a_seg.count == 0)
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
    // Step i's loads; past the last one they read zeros from beyond the buffers, so that every step issues the same number.
    unsigned int a_soffset = 0, b_soffset = 0;
    auto aim = [&](int i) __attribute__((always_inline)) {
        const unsigned int past_end = i >= steps ? 0x80000000u : 0u;
        const int k0 = min(kt_begin + wave + kWaves * i, p.k_tiles - 1) * kBK<T>;
        a_soffset = a_src.first_offset(k0, 0) | past_end;
        if constexpr (A_K && SEGMENTED) {
            if (p.a_seg.count > 0) {
                const SegmentPick pick = pick_small_segment(p.a_seg, k0);
                a_src.init(static_cast<const T*>(pick.ptr) + static_cast<long>(m0) * pick.ld, pick.ld, p.m - m0, pick.cols, 0);
                a_soffset = a_src.first_offset(k0 - pick.first, 0) | past_end;
            }
        }
        b_soffset = b_src.first_offset(k0, 0) | past_end;
    };
    auto issue = [&](auto index, unsigned int stage_lds) __attribute__((always_inline)) {
        constexpr int l = decltype(index)::value;
        if constexpr (l < kOperandLoads)
            a_soffset = load_to_lds<l * kLoadBytes>(a_src.rsrc, stage_lds, a_src.load_voffset(l), a_soffset, a_src.group_bytes);
        else
            b_soffset = load_to_lds<l * kLoadBytes>(b_src.rsrc, stage_lds, b_src.load_voffset(l - kOperandLoads), b_soffset, b_src.group_bytes);
    };

    static_for<0, STAGES>([&](auto s) {
        aim(decltype(s)::value);
        static_for<0, kLoads>([&](auto l) { issue(l, lds_wave + decltype(s)::value * kStageBytes); });
    });

    constexpr int kAOffsets = A_K ? 1 : kBlocks, kBOffsets = B_K ? 1 : kBlocks;
    int a_off[kAOffsets], b_off[kBOffsets];
    if constexpr (A_K) a_off[0] = ATile::lane_offset(lane);
    else static_for<0, kBlocks>([&](auto i) { a_off[decltype(i)::value] = ATile::lane_offset(lane, decltype(i)::value * 16); });
    if constexpr (B_K) b_off[0] = BTile::lane_offset(lane);
    else static_for<0, kBlocks>([&](auto i) { b_off[decltype(i)::value] = BTile::lane_offset(lane, decltype(i)::value * 16); });
    frag_t af[2][kBlocks], bf[2][kBlocks];
    auto read_frag = [&]<int BUFFER, int F>(const T* stage) __attribute__((always_inline)) {
        if constexpr (F < kBlocks) {
            if constexpr (A_K) af[BUFFER][F] = ATile::frag(stage, F * 16, a_off[0]);
            else af[BUFFER][F] = ATile::frag(stage, a_off[F]);
        } else {
            constexpr int j = F - kBlocks;
            if constexpr (B_K) bf[BUFFER][j] = BTile::frag(stage + kOperandElems, j * 16, b_off[0]);
            else bf[BUFFER][j] = BTile::frag(stage + kOperandElems, b_off[j]);
        }
    };

    acc_t acc[kBlocks][kBlocks];
#pragma unroll
    for (int i = 0; i < kBlocks; ++i)
#pragma unroll
        for (int j = 0; j < kBlocks; ++j) acc[i][j] = acc_t(0.0f);
    wait_loads<(STAGES - 1) * kLoads>();
    static_for<0, 2 * kBlocks>([&](auto f) { read_frag.template operator()<0, decltype(f)::value>(wave_stages); });
    int stage = 0;
    auto step = [&]<int BUFFER>(int i) __attribute__((always_inline)) {
        const int next_stage = (stage + 1) % STAGES;
        aim(i + STAGES);
        // This step's fragments are in registers, so its stage can be refilled; the next step's K tile has landed.
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        wait_loads<(STAGES - 2) * kLoads>();
        constexpr int kMfmas = kBlocks * kBlocks, kReads = 2 * kBlocks;
        static_for<0, kMfmas>([&](auto index) {
            constexpr int m = decltype(index)::value, row = m / kBlocks, column = (row & 1) ? kBlocks - 1 - m % kBlocks : m % kBlocks;
            Mfma<T>::run(acc[row][column], bf[BUFFER][column], af[BUFFER][row]);
            // The fragment reads in the first half of the MFMAs, the loads in the second.
            if constexpr (m < kMfmas / 2) {
                static_for<m * kReads / (kMfmas / 2), (m + 1) * kReads / (kMfmas / 2)>(
                    [&](auto f) { read_frag.template operator()<BUFFER ^ 1, decltype(f)::value>(wave_stages + next_stage * kStageElems); });
            } else {
                constexpr int h = m - kMfmas / 2;
                static_for<h * kLoads / (kMfmas / 2), (h + 1) * kLoads / (kMfmas / 2)>(
                    [&](auto l) { issue(l, lds_wave + stage * kStageBytes); });
            }
            __builtin_amdgcn_sched_barrier(0);
        });
        stage = next_stage;
    };
    for (int i = 0; i < steps; i += 2) {
        step.template operator()<0>(i);
        if (i + 1 < steps) step.template operator()<1>(i + 1);
    }

    // The partial tiles, [wavefront][row][column] in fp32. Everybody's loads (of zeros, past the end) have to be through
    // before the stages are reused; the waits also separate the last MFMA from the reads of its accumulator.
    constexpr int kPitch = TILE + 4;
    static_assert(kWaves * TILE * kPitch * 4 <= kWaves * STAGES * kStageBytes + 8192, "partial tiles fit where the stages were");
    float* const partial = reinterpret_cast<float*>(smem_raw);
    wait_loads<0>();
    asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
    __syncthreads();
    {
        float* mine = partial + wave * TILE * kPitch + (lane & 15) * kPitch + (lane >> 4) * 4;
#pragma unroll
        for (int i = 0; i < kBlocks; ++i)
#pragma unroll
            for (int j = 0; j < kBlocks; ++j) *reinterpret_cast<acc_t*>(mine + i * 16 * kPitch + j * 16) = acc[i][j];
    }
    __syncthreads();
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
