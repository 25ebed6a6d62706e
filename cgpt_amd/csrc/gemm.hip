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
// Operands whose rows are not whole aligned 16-byte chunks are copied to padded rows first;
// C may have any width and alignment (a store per element). fp32 storage takes the same kernels
// with v_mfma_f32_16x16x4_f32 and K steps of 16. Operands beyond 32-bit offsets, and unaligned ones
// of a caller that owns the arena or whose padded copies the arena has no room for, run on a general fp32 matrix-core kernel
// (v_mfma_f32_32x32x2_f32, register-staged operand tiles) with the same semantics.
#include "gemm_large.hpp"
#include "gemm_small.hpp"
#include "gemm_tiles.hpp"

#include <algorithm>
#include <cmath>
#include <cstdlib>

namespace cgptx {
namespace {

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

// Copies [rows, cols] matrices to rows of `pitch` elements (whole 16-byte chunks), zeros past cols: the streamed kernels
// read whole chunks. One chunk per thread; a source may start anywhere. Two copies, those of a product of odd K, share a launch: the first
// first_blocks workgroups take one, the others the other.
struct PadJob {
    void* dst;
    const void* src;
    long rows, ld;
    int cols, pitch;
};
template <typename E>
__global__ __launch_bounds__(kThreads) void pad_rows_kernel(PadJob first, PadJob second, int first_blocks) {
    constexpr int VEC = kVec128<E>;
    const bool other = static_cast<int>(blockIdx.x) >= first_blocks;
    const PadJob job = other ? second : first;
    const long block = static_cast<int>(blockIdx.x) - (other ? first_blocks : 0);
    const long blocks = other ? static_cast<int>(gridDim.x) - first_blocks : first_blocks;
    const E* const src = static_cast<const E*>(job.src);
    E* const dst = static_cast<E*>(job.dst);
    const int chunks = job.pitch / VEC;
    const long total = job.rows * chunks;
    for (long q = block * kThreads + threadIdx.x; q < total; q += blocks * kThreads) {
        const long row = q / chunks;
        const int col = static_cast<int>(q - row * chunks) * VEC;
        const E* from = src + row * job.ld + col;
        vec_t<E, VEC> v;
        if (col + VEC <= job.cols) {
            __builtin_memcpy(&v, from, 16);
        } else {
#pragma unroll
            for (int e = 0; e < VEC; ++e) v[e] = col + e < job.cols ? from[e] : E{0};
        }
        store_vec<E, VEC>(dst + row * job.pitch + col, v);
    }
}
int launch_pad_rows(const PadJob& first, const PadJob* second, int dtype, hipStream_t stream) {
    auto blocks_of = [&](const PadJob& job) {
        const long chunks = job.rows * (job.pitch * static_cast<long>(dtype_size(dtype)) / 16);
        return static_cast<int>(std::min<long>((chunks + kThreads - 1) / kThreads, static_cast<long>(compute_units()) * 16));
    };
    const int blocks = blocks_of(first);
    const dim3 grid(static_cast<unsigned int>(blocks + (second != nullptr ? blocks_of(*second) : 0)));
    auto kernel = dtype == CGPTX_F32 ? pad_rows_kernel<std::uint32_t> : pad_rows_kernel<std::uint16_t>;
    hipLaunchKernelGGL(kernel, grid, dim3(kThreads), 0, stream, first, second != nullptr ? *second : first, blocks);
    CGPTX_LAUNCH_CHECK();
    return CGPTX_OK;
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

// Oblong tiles run one block per CU: us before and after a block's K loop, of a further one, of a K step on an idle chip and what a
// full one (whose clock and L2s are shared) adds. Measured as predicted_us says, K from 128 to 4096: within 8 per cent where one round of
// blocks is enough, and short by up to 20 where many rounds run at the power limit. How much less than the best square tiles or 256 x 192
// ones they have to be predicted to take is oblong_has_to_beat's. [M, N] x K, us, operands rotated,
// best of those and chosen: 5005 x 1024 x 1024 17.3 -> 14.6 (160 x 128), x 2048 27.4 -> 22.6; 7000 x 768 x 2048 27.9 -> 24.1 (192 x 128);
// 5005 x 2048 x 1024 26.4 -> 22.8 (160 x 256), 10000 x 1024 x 1024 26.8 -> 22.4; 13000 x 4096 x 1024 108 -> 98 (224 x 256). Full rounds
// of 256 x 128 gain little: 8192 x 1024 x 1024 19.1 - 20.7 and 18.6 - 20.2, its input gradient 19.6 - 20.7 and 19.3 - 20.1, 4096 x 2048 x 1024
// 19.3 - 19.9 and 19.0 - 20.3; with a bias, which square tiles add in their general epilogue, 21.3 - 22.6 and 19.2 - 20.3. Where square
// tiles fill the chip they stay: 16384 x 1024 x 1024 30.6 and 35.5 (256 x 128), 2000 x 2048 x 1024 12.0 (128 x 128) and 12.9.
struct OblongCost {
    int tile;
    double first, further, step, step_full;
};
constexpr OblongCost kOblongCosts[] = {{oblong_tile(160, 128), 5.6, 2.8, 0.165, 0.085}, {oblong_tile(192, 128), 5.8, 3.2, 0.20, 0.09},
                                       {oblong_tile(256, 128), 6.2, 4.0, 0.23, 0.13},   {oblong_tile(160, 256), 7.2, 4.2, 0.24, 0.19},
                                       {oblong_tile(192, 256), 7.5, 4.5, 0.32, 0.17},   {oblong_tile(224, 256), 7.8, 5.0, 0.37, 0.19}};
const OblongCost& oblong_cost(int tile) {
    for (const OblongCost& c : kOblongCosts)
        if (c.tile == tile) return c;
    return kOblongCosts[0];
}
// What square tiles have to be predicted to take at least for an oblong one to be taken: more where its prediction is known to be short. Of several
// rounds of tiles of 128 columns those predicted to gain 6 per cent lost 3 (19504 x 640 x 4096 100 -> 104 us, 33416 x 640 x 2048 93.5 -> 96), those
// predicted to gain 7 to 13 gained 2 to 8; beyond four rounds of sums longer than 512 5 to 7 per cent predicted were -2 to 0
// (28856 x 2048 x 2048 202 -> 205, 30304 x 4096 x 768 178 -> 180) and 15 were 3 to 8. With a bias all of these gain (19105 x 640 x 4096 90.3 -> 84.6).
double oblong_has_to_beat(int tile, double predicted, long tiles, long k_tiles, bool bias, long units) {
    if (bias) return 1.05 * predicted;
    if (tiles > 4 * units && k_tiles > 16) return 1.10 * predicted;
    return (tiles > units && tile_columns(tile) == 128 ? 1.07 : 1.05) * predicted;
}
// What a call of 128 x 128 tiles with a CU each takes, closer than predicted_us has it where K is long: many small blocks bring in more at once
// than few large ones. Of such calls 16 of 16 lost 2 to 10 per cent on oblong tiles (2000 x 1280 x 4096 29.0 -> 31.8, 3000 x 1024 x 4096 31.1 -> 32.8,
// its input gradient 32.3 -> 35.3, 1552 x 1536 x 1024 11.6 -> 12.4) unless a bias is added (1670 x 1280 x 1024 13.6 -> 12.8, 3000 x
// 1024 x 4096 32.0 -> 32.6). Within 6 per cent.
double lone_blocks_us(long tiles, long k_tiles, bool bias, long units) {
    const double load = static_cast<double>(tiles) / static_cast<double>(units);
    return 5.9 + static_cast<double>(k_tiles) * (0.15 + 0.06 * load) + (bias ? 2.0 : 0.0);
}

// CGPTX_GEMM_TILE=32|64|128|192|256|160128|... pins the tile size (for experiments); anything else = automatic, and so is a size that a call's
// kernels do not have (192 where takes_narrow_tiles says no, oblong ones where takes_oblong_tiles does, 256 in fp32).
int forced_tile() {
    static const int value = [] {
        const char* text = std::getenv("CGPTX_GEMM_TILE");
        if (text == nullptr) return 0;
        const int v = std::atoi(text);
        bool oblong = false;
        for (const OblongCost& c : kOblongCosts) oblong = oblong || c.tile == v;
        return (v == 32 || v == 64 || v == 128 || v == 192 || v == 256 || oblong) ? v : 0;
    }();
    return value;
}

std::size_t round_up(std::size_t v, std::size_t unit) { return (v + unit - 1) / unit * unit; }

// How a call of the streamed kernels is cut: tile, K slices per tile and K steps per slice.
struct Plan {
    int tile = 256;  // see tile_rows
    int replaced = 0;  // the tile that an oblong one took the place of
    static long tiles_of(const GemmArgs& g, int tile) {
        const std::size_t rows = tile_rows(tile), columns = tile_columns(tile);
        return static_cast<long>((g.m + rows - 1) / rows) * static_cast<long>((g.n + columns - 1) / columns);
    }
    int slices = 1;
    int k_tiles_per_slice = 1;
    bool deep = false;  // small tiles: all of a CU's LDS for one workgroup's stages
    std::size_t partial_bytes(const GemmArgs& g) const {
        return slices > 1 ? static_cast<std::size_t>(slices) * g.m * round_up(g.n, 8) * sizeof(float) : 0;
    }
};

// Predicted time of a call in microseconds, from launches measured on random bf16 data inside a graph (operands rotated
// through 64 MB; K tiles of 64 bytes): what a kernel costs before its K loop, plus the K loop of the busiest CU.
//   256: one block per CU, 8.5 us for filling its pipeline and storing its tile (6.8 where the next tile's loads run under
//        the store), 0.48 per K tile on an idle chip, 0.65 at the power limit of a full one
//   256 x 192: one block per CU, 10 us and 7.5 for a further one, 0.40 per K tile on an idle chip, 0.55 on a full one
//   128: 0.235 per K tile for a block that has a CU to itself, 0.17 each for two that share one where other CUs have less to
//        do, 0.22 where all of them load at once, up to 0.245 in calls long enough to meet the power limit
//    64: 0.09 - 0.13 per K tile with up to one block per CU, 0.11 per K tile and block with more
//    32: 0.07 - 0.1 per K tile (k-contiguous operands stream best), up to one block per CU
// A split along K adds a launch and the partial tiles' way to memory and back. fp32 K tiles hold 16 positions and take about
// as long as the fp32 matrix rate asks (0.93 per K tile of 128 x 128), smaller tiles somewhat longer for their share.
// [M, N] x K: 128 x 768 x 768 32/1 4.4, 64/1 5.4; 1000 x 1024 x 1024 64/1 7.5, 32/1 9.5; 2000 x 2048 x 1024 128/1 13.3, 64/1
// 17.2, 256/1 25.2; 5005 x 1024 x 1024 128/1 17.3, 256/1 25.6; 5005 x 2048 x 1024 128/1 26.4, 256/1 27.1; 16384 x 1024 x 1024
// 256/1 31.1, 128/1 35.6; 32768 x 768 x 768 128/1 41.5, 192/1 44.2, 256/1 46.3; 32768 x 768 x 2048 192/1 85.3, 128/1 91.1, 256/1 91.2; 2048 x 4096 x 4096 128/1 60.1, 256/1 77.5; 8192 x 4096 x 1024 256/1 62.5, 128/1 68.2 (tile / slices).
double predicted_us(int tile, long tiles, long slices, long k_tiles, double partial_mb, bool f32, bool a_k, bool b_k, long units) {
    const double kt = static_cast<double>((k_tiles + slices - 1) / slices);
    const double load = static_cast<double>(tiles * slices) / static_cast<double>(units);
    const double blocks = std::ceil(load);
    double time = 0.0;
    if (tile > 256) {
        const OblongCost& c = oblong_cost(tile);
        const double filled = load / blocks;
        time = c.first + 1.3 * filled + c.further * (blocks - 1.0) + blocks * kt * (c.step + c.step_full * filled);
    } else if (f32) {
        const double per_tile = tile == 32 ? 0.088 : tile == 64 ? 0.265 : 0.93;
        time = (tile == 32 ? 3.0 : tile == 64 ? 4.0 : 5.0) + kt * per_tile * (tile == 32 ? std::max(1.0, load) : blocks);
    } else if (tile == 192) {
        time = 10.0 + 7.5 * (blocks - 1.0) + blocks * kt * (0.40 + 0.15 * load / blocks);
    } else if (tile == 256) {
        time = 8.5 + 6.8 * (blocks - 1.0) + blocks * kt * (0.48 + 0.17 * load / blocks);
    } else if (tile == 128) {
        const double crowded = std::min(0.245, 0.21 + 0.005 * load);
        time = 5.9 + kt * (load <= 1.0 ? 0.235 : std::max(0.17 * blocks, crowded * load)) + 1.2 * std::max(0.0, std::ceil(blocks / 2.0) - 1.0);
    } else if (tile == 64) {
        time = load <= 1.0 ? 3.4 + kt * (0.09 + 0.04 * load)
                           : 3.4 + kt * 0.11 * blocks * (blocks > 4.0 ? 1.3 : 1.0);
    } else {
        time = 2.6 + kt * (!a_k ? 0.1 : b_k ? 0.07 : 0.085) * std::max(1.0, 0.92 * load);
    }
    return slices > 1 ? time + 3.0 + 0.45 * partial_mb + 0.3 * std::min(partial_mb, 8.0) : time;
}

bool c_streams(const GemmArgs& g, std::size_t elem);

// Whether 256 x 192 tiles take a call: 16-bit storage, nothing but products, a residual, an fp32 addend and what C holds added, C
// in one buffer, it and what is added in whole aligned chunks.
bool takes_narrow_tiles(const GemmArgs& g) {
    constexpr std::size_t kMostPitch = std::size_t{1} << 21;  // 32-bit offsets within a wavefront's 128 rows of fp32
    return g.dtype != CGPTX_F32 && g.bias == nullptr && g.a_sums == nullptr && g.swiglu_out == nullptr && g.swiglu_saved == nullptr &&
           g.c_segments.count == 0 && g.batch_rows == 0 && (g.a_k_contiguous || (!g.b_k_contiguous && g.a_segments.count == 0)) &&
           (g.a_segments.count == 0 || !g.b_k_contiguous) && !(g.residual != nullptr && (g.c_is_f32 || g.accumulate)) &&
           !(g.addend_f32 != nullptr && g.c_is_f32 && g.accumulate) && c_streams(g, 2) &&
           g.ldc < kMostPitch && g.ldr < kMostPitch && g.ld_addend < kMostPitch;
}

// Whether oblong tiles take a call: 16-bit storage, k-contiguous A, one sum over K, the result stored as it is, with a residual or
// what C holds added, or (a forward product) with a bias.
bool takes_oblong_tiles(const GemmArgs& g) {
    if (g.bias != nullptr && (!g.b_k_contiguous || g.residual != nullptr || g.accumulate)) return false;
    return g.dtype != CGPTX_F32 && g.a_k_contiguous && g.addend_f32 == nullptr && !g.c_is_f32 && g.a_sums == nullptr &&
           g.swiglu_out == nullptr && g.swiglu_saved == nullptr && g.batch_rows == 0 && !(g.a_segments.count > 0 && (g.b_k_contiguous || g.residual != nullptr || g.accumulate)) &&
           !(g.residual != nullptr && g.accumulate) && !(g.c_segments.count > 0 && (g.residual != nullptr || g.accumulate)) && c_streams(g, 2);
}

Plan make_plan(const GemmArgs& g) {
    Plan plan;
    const long units = compute_units();
    const bool f32 = g.dtype == CGPTX_F32;
    const long k_step = f32 ? kBK<float> : kBK<bf16_t>;
    const long k_tiles = (static_cast<long>(g.k) + k_step - 1) / k_step;
    auto tiles_of = [&](int tile) { return Plan::tiles_of(g, tile); };
    const bool may_split = (!g.no_split || g.split_workspace != nullptr) && g.residual == nullptr && g.addend_f32 == nullptr &&
                           g.swiglu_out == nullptr && g.swiglu_saved == nullptr && g.c_segments.count == 0 &&
                           !(g.a_k_contiguous && g.a_segments.count > 0);
    auto set_slices = [&](long slices) {
        plan.k_tiles_per_slice = static_cast<int>((k_tiles + slices - 1) / slices);
        // Slices of a k-contiguous operand begin at whole K tiles: its rows are read in whole cache lines. A K step of k-strided
        // operands is whole rows of memory wherever it begins, and their slices are as long as each other.
        if (slices > 1 && (g.a_k_contiguous || g.b_k_contiguous))
            plan.k_tiles_per_slice = (plan.k_tiles_per_slice + kSteps - 1) / kSteps * kSteps;
        plan.slices = static_cast<int>((k_tiles + plan.k_tiles_per_slice - 1) / plan.k_tiles_per_slice);
    };
    const int pinned = forced_tile();
    // Oblong tiles in place of plan.tile's, predicted to take `best`: the same sums in the same order.
    auto try_oblong = [&](double best) {
        plan.replaced = plan.tile;
        for (const OblongCost& c : kOblongCosts) {
            if (pinned > 256 && c.tile != pinned) continue;
            const double time = oblong_has_to_beat(c.tile, predicted_us(c.tile, tiles_of(c.tile), 1, k_tiles, 0.0, f32, true, g.b_k_contiguous, units),
                                                   tiles_of(c.tile), k_tiles, g.bias != nullptr, units);
            if (pinned == 0 && time >= best) continue;
            best = time;
            plan.tile = c.tile;
        }
    };
    if (g.swiglu_out != nullptr || g.swiglu_saved != nullptr || (!f32 && tiles_of(256) >= 3 * units && g.batch_rows == 0)) {
        // Of more rounds the last one is too small a part.
        if ((pinned == 0 || pinned > 256) && tiles_of(256) <= 8 * units && takes_oblong_tiles(g))
            try_oblong(predicted_us(256, tiles_of(256), 1, k_tiles, 0.0, f32, true, g.b_k_contiguous, units));
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
    const int forced = (pinned == 192 && !takes_narrow_tiles(g)) || (pinned > 256 && !takes_oblong_tiles(g)) || (f32 && pinned == 256) ? 0 : pinned;
    const double slice_bytes = static_cast<double>(g.m) * static_cast<double>(round_up(g.n, 8)) * sizeof(float);
    // Calls that 256 x 256 tiles spread over three quarters of the chip keep the order of additions of the kernels with a
    // SwiGLU epilogue, which take such calls only (one sum over all of K): the fused and the separate operators give the same
    // bits. A split would fill the last quarter, less the partial tiles' way: 16384 x 768 x 32000 688 us, in four slices 650.
    const bool whole_k = !f32 && tiles_of(256) * 4 >= units * 3;
    double best = -1.0;
    long best_slices = 1;
    for (int tile : {32, 64, 128, 256}) {
        if ((whole_k && tile < 128) || (forced != 0 && tile != forced) || (f32 && tile == 256)) continue;
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
    // 256 x 192 tiles where one sum over K on a large tile is best anyway: they add in the same order.
    const bool large = plan.tile >= 128 && best_slices == 1;
    if (takes_narrow_tiles(g) && (forced == 192 || (forced == 0 && large))) {
        const double time = predicted_us(192, tiles_of(192), 1, k_tiles, 0.0, f32, g.a_k_contiguous, g.b_k_contiguous, units);
        if (forced == 192 || time < best) {
            best = time;
            plan.tile = 192;
            best_slices = 1;
        }
    }
    if (takes_oblong_tiles(g) && (forced > 256 || (forced == 0 && large))) {
        try_oblong(tiles_of(128) <= units ? std::min(best, lone_blocks_us(tiles_of(128), k_tiles, g.bias != nullptr, units)) : best);
        best_slices = plan.tile > 256 ? 1 : best_slices;
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
    const int rows = tile_rows(plan.tile), columns = tile_columns(plan.tile);
    p.tiles_m = (p.m + rows - 1) / rows;
    p.tiles_n = (p.n + columns - 1) / columns;
    p.k_tiles_per_slice = plan.k_tiles_per_slice;
    auto launch = [&](const KernelArgs& args, bool split) -> int {
        if (plan.tile <= 64) return launch_small_call<T>(g, args, plan, split, stream);
        const LargeCall call{args, g.a_k_contiguous, g.b_k_contiguous, plan.tile, split, plan.slices};
        if constexpr (std::is_same_v<T, bf16_t>) return plan.tile > 256 ? gemm_oblong_bf16(call, stream) : gemm_large_bf16(call, stream);
        else if constexpr (std::is_same_v<T, f16_t>) return plan.tile > 256 ? gemm_oblong_f16(call, stream) : gemm_large_f16(call, stream);
        else return gemm_large_f32(call, stream);
    };
    if (plan.slices == 1) return launch(p, false);
    KernelArgs split = p;
    split.c = g.split_workspace;
    split.ld_partial = static_cast<long>(round_up(g.n, 8));
    if (int s = launch(split, true)) return s;
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
    // Both operands' copies in one launch, graphs of calls: bf16 16 x 1379 x 256 8.3 -> 6.5 us, 1000 x 1021 x 1024 14.1 -> 12.4.
    PadJob jobs[2];
    int copies = 0;
    auto copy = [&](void* to, const void* from, bool k_contiguous, std::size_t extent, std::size_t ld, std::size_t pitch) {
        jobs[copies++] = PadJob{to, from, static_cast<long>(k_contiguous ? extent : g.k), static_cast<long>(ld),
                                static_cast<int>(k_contiguous ? g.k : extent), static_cast<int>(pitch)};
    };
    if (pad_a) {
        padded.a = base;
        copy(base, g.a, g.a_k_contiguous, g.m, g.lda, padded.lda);
    }
    if (pad_b) {
        padded.b = base + a_bytes;
        copy(base + a_bytes, g.b, g.b_k_contiguous, g.n, g.ldb, padded.ldb);
    }
    if (int s = launch_pad_rows(jobs[0], copies > 1 ? &jobs[1] : nullptr, g.dtype, stream)) return s;
    padded.no_split = true;
    padded.split_workspace = split_bytes != 0 ? base + a_bytes + b_bytes : nullptr;
    padded.split_workspace_bytes = std::min(split_bytes, held - a_bytes - b_bytes);
    return run_typed<T>(padded, stream);
}

constexpr double kGroupBlocksPerUnit = 16.0;  // of a group, at most

// An input and a weight gradient that gemm_pair_kernel takes together (the small kernels' groups take more).
bool pairs(const GemmArgs* calls, int count) {
    return count == 2 && calls[0].dtype != CGPTX_F32 && calls[0].a_k_contiguous && !calls[0].b_k_contiguous && calls[0].a_segments.count == 0 &&
           !calls[1].a_k_contiguous && !calls[1].b_k_contiguous && calls[1].a_segments.count == 0;
}
long tiles_of_size(const GemmArgs& g, std::size_t rows, std::size_t columns) {
    return static_cast<long>((g.m + rows - 1) / rows) * static_cast<long>((g.n + columns - 1) / columns);
}
// The weight gradient's tile of a pair, by the input gradient's.
int pair_weight_rows(const GemmGroup& plan) { return plan.tile[0] > 256 ? kPairWeightRows : 128; }
int pair_weight_columns(const GemmGroup& plan) { return plan.tile[0] > 256 ? kPairWeightColumns : 128; }
long k_steps_16bit(const GemmArgs& g) { return static_cast<long>((g.k + kBK<bf16_t> - 1) / kBK<bf16_t>); }
// K steps of a slice: whole K tiles, as the kernels read them.
long slice_steps(long steps, long slices) { return ((steps + slices - 1) / slices + kSteps - 1) / kSteps * kSteps; }

// Predicted time of a pair in microseconds: the dispatch of its workgroups, the longer ones first, onto two slots per CU, in K steps
// (0.22 us of a workgroup that has a CU to itself, 0.47 each of two that share one, no CU faster than 0.237 a step), 5.6 before and
// after the K loops, and the way of the partial tiles to memory and back. Fitted to 33 shapes from 300 x 768 x 768 to 32768 x 768 x 768
// in up to 12 slices each: within 15 per cent where it matters, the slice count it picks within 6 of the best one. Both gradients
// of [rows, in] x out, us, calls of their own (or the small group) and a pair: 2000 x 1024 x 2048 34.3 -> 22.3, 5005 x 1024 x 1024 38.0 -> 29.6,
// 5005 x 1024 x 2048 59.0 -> 50.3, 4096 x 768 x 2048 45.0 -> 32.5, 8192 x 1024 x 2048 74.7 -> 65.0; 1000 x 1024 x 1024 12.4 and 13.0,
// 8192 x 256 x 256 17.0 and 20.6 (partial tiles), 16384 x 1024 x 4096 225 and 229 (256 x 256 tiles): those stay as they were.
// The slots are only walked where the answer can be below `worth`: a bound is returned where not (the walk is most of what planning a
// large call costs, up to 1.5 us).
double predicted_pair_us(long tiles_x, long steps_x, long tiles_w, long steps_w, long slices, long units, double worth) {
    const long kt = slices > 1 ? slice_steps(steps_w, slices) : steps_w, items_w = tiles_w * slices, items = tiles_x + items_w;
    const bool weight_first = kt >= steps_x;
    const long counts[2] = {weight_first ? items_w : tiles_x, weight_first ? tiles_x : items_w};
    const long lengths[2] = {weight_first ? kt : steps_x, weight_first ? steps_x : kt};
    const double work = static_cast<double>(tiles_x * steps_x + items_w * kt) / static_cast<double>(units);
    const double fold = slices > 1 ? 3.0 * static_cast<double>(items_w) / static_cast<double>(units) + 0.9 * static_cast<double>(slices) : 0.0;
    // K steps of the CU that ends last: of its longer slot, and of the one beside it.
    double longest = static_cast<double>(lengths[0]), beside = 0.0;
    auto time = [&]() { return 5.6 + std::max(0.22 * (longest - beside) + 0.47 * beside + fold, 0.237 * work); };
    if (items > 2 * units) {
        longest = std::max(longest, work / 2.0);  // no slot order has a shorter longest one
        beside = work / 2.0;
        if (time() >= worth) return time();
        // Slots by the steps they have been given: the least loaded ones take the next workgroups.
        struct Slots {
            long steps, count;
        } slots[64] = {{0, 2 * units}};
        int groups = 1;
        for (int kind = 0; kind < 2; ++kind) {
            for (long left = counts[kind]; left > 0;) {
                int least = 0;
                for (int i = 1; i < groups; ++i)
                    if (slots[i].steps < slots[least].steps) least = i;
                const long taken = std::min(left, slots[least].count), steps = slots[least].steps + lengths[kind];
                left -= taken;
                slots[least].count -= taken;
                if (slots[least].count == 0) slots[least] = slots[--groups];
                int same = 0;
                while (same < groups && slots[same].steps != steps) ++same;
                if (same == groups && groups < 64) slots[groups++] = {steps, 0};
                slots[std::min(same, groups - 1)].count += taken;
            }
        }
        long most = 0;
        for (int i = 0; i < groups; ++i) most = std::max(most, slots[i].steps);
        longest = static_cast<double>(most);
        beside = std::min(longest, work / 2.0);
    } else if (items > units) {
        beside = static_cast<double>(counts[0] > units ? lengths[0] : lengths[1]);
    }
    return time();
}

// What oblong pairs are held against: the same, closer, where all workgroups have a slot at once. Two that share a CU take 0.28 us a K step there
// and not 0.47. Fitted to 2472 launches of 1298 drawn shapes, three sets of operands in turn: 2 per cent short, standard deviation 6 (predicted_pair_us
// 9 per cent too long, 11).
double pair_us_of_one_round(long tiles_x, long steps_x, long tiles_w, long steps_w, long slices, long units) {
    const long kt = slices > 1 ? slice_steps(steps_w, slices) : steps_w, items_w = tiles_w * slices, items = tiles_x + items_w;
    const bool weight_first = kt >= steps_x;
    const long longest = weight_first ? kt : steps_x, most = weight_first ? items_w : tiles_x;
    const long beside = items <= units ? 0 : most > units ? longest : weight_first ? steps_x : kt;
    if (items <= units && slices > 1)  // few workgroups, in short slices: they do not slow each other down
        return 8.0 + 1.2 * static_cast<double>(slices) + static_cast<double>(longest) * (0.13 + 0.07 * static_cast<double>(items) / static_cast<double>(units));
    const double work = static_cast<double>(tiles_x * steps_x + items_w * kt) / static_cast<double>(units);
    return (slices > 1 ? 8.0 + 0.9 * static_cast<double>(slices) : 5.0) + 0.22 * static_cast<double>(longest - beside) + 0.28 * static_cast<double>(beside) +
           0.05 * work;
}

// A pair with an oblong tile for the input gradient and 256 x 128 for the weight gradient, where every workgroup has a CU to itself:
// the longer of the two, and what the shorter one takes of the L2s and the power meanwhile. Both operands of the weight gradient are read transposed
// from LDS, 0.30 - 0.39 us a K step; adding its slices up takes some 5 us, and longer the later the input gradient's tiles let go of the memory. Fitted to
// 6070 launches of 1510 drawn shapes: standard deviation 3 per cent in one slice, 5 in two and three. What several rounds take varies by a third with
// the order in which workgroups end, so those keep to 128 x 128 tiles.
double predicted_oblong_pair_us(const OblongCost& c, long tiles_x, long steps_x, long tiles_w, long steps_w, long slices, long units) {
    const long items = tiles_x + tiles_w * slices;
    // Workgroups go to the XCDs in turn and each call's tiles are dealt out to them by itself: one round is one that every XCD's share of
    // either fits. 3613 x 1408 x 1792 is 102 and 154 workgroups, 13 and 20 on some XCDs of 32 CUs: 39.5 us on 128 x 128 tiles, 66.6 on these.
    const long on_an_xcd = (tiles_x + kXcds - 1) / kXcds + (tiles_w * slices + kXcds - 1) / kXcds;
    if (on_an_xcd > units / kXcds) return std::numeric_limits<double>::infinity();
    const long kt = slices > 1 ? slice_steps(steps_w, slices) : steps_w;
    const double filled = static_cast<double>(items) / static_cast<double>(units);
    const double input = static_cast<double>(steps_x) * (1.09 * c.step + 0.565 * c.step_full * filled);
    const double weight = static_cast<double>(kt) * (0.30 + 0.087 * filled);
    const double longer = std::max(input, weight), shorter = std::min(input, weight);
    return slices == 1 ? 7.2 + 0.93 * longer + 0.20 * shorter
                       : 7.6 + 0.54 * static_cast<double>(slices) + 0.77 * longer + 0.30 * shorter + 15.7 * static_cast<double>(tiles_x) / static_cast<double>(units);
}

// What a pair on oblong tiles has to be predicted to take in place of one of 128 x 128 predicted at `pair_us`: 5 per cent less where all workgroups of that one
// have a slot at once, 12 where not (predicted_pair_us is longest there just where some CUs get one more). Of 1252 drawn shapes with such a pair 294 take oblong
// tiles, 0.90 of the time in the mean, and 5 lose 1 to 3 per cent; of 140 others 2, by 2 and 4. Asked for 6 per cent less than predicted_pair_us says, 114 of
// 270 lost, up to 20. us, 128 x 128 and chosen: 5005 x 1024 x 2048 50.5 -> 46.2, 6000 x 1024 x 2048 60.0 -> 52.1, 6983 x 760 x 2048 53.3 -> 48.6, 7000 x
// 768 x 2048 50.5 -> 48.5. That stay: 5005 x 1024 x 1024 30.4 and 31.5, 4096 x 768 x 2048 34.3 and 35.9, 2816 x 896 x 2944 36.2 and 41.7, 1615 x 1792 x
// 1472 24.5 and 28.6, 3357 x 1024 x 2688 41.3 and 48.1; and, for want of a closer prediction, 3000 x 1024 x 4096 50.8 and 46.9.
double oblong_pair_has_to_beat(double pair_us, long tiles_x, long steps_x, long tiles_w, long steps_w, long slices, long units) {
    if (tiles_x + tiles_w * slices > 2 * units) return pair_us / 1.12;
    return pair_us_of_one_round(tiles_x, steps_x, tiles_w, steps_w, slices, units) / 1.05;
}

// A group's tiles: those whose predicted time in one launch is least. The launch takes as long as its longest workgroup or
// as the busiest CU's share of the work, whatever is more (us per K tile and workgroup as in predicted_us; 3.5 us before and
// after the K loops). Two workgroups share a CU and its LDS, or, deep, each has one to itself: then the longest is not held
// up by another, but 3.5 us of start and end of every workgroup are in nobody's shadow. Joined if that is less than the calls'
// own predictions in turn. [M, N] x K measured apart and joined: dX and dW of 128 x 768 x 768 10.4 -> 7.4 us, of 2000 x 1024 x
// 2048 35.7 -> 32.3; 5005 x 1024 x 256, whose dW is better split along K, 23.7 -> 28.8: stays apart. fp32, 256 rows, 1024 wide, 8:2
// heads of 128, feed-forward of 2048: the gradients of gate|up, q, k and v in turn 83, joined 66; q, k, v and gate|up forward on 64 x 64
// tiles 42, gate|up on those and the others on 32 x 32 37.
GemmGroup plan_group(const GemmArgs* calls, int count, bool pair) {
    GemmGroup best_plan;
    const double units = static_cast<double>(compute_units());
    // Large calls are told apart by their tiles alone: whatever is spent here, they pay beside their own plans.
    double fewest = 0.0;
    for (int i = 0; i < count; ++i) fewest += static_cast<double>((calls[i].m + 63) / 64) * static_cast<double>((calls[i].n + 63) / 64);
    if (fewest > (pair ? 4.0 : 1.0) * kGroupBlocksPerUnit * units) return best_plan;
    double separate = 0.0;
    // fp32 pairs whose own plans have no K slices: a group gives neither a longer chain of additions. (Who makes larger groups of
    // gradients has looked at that, see gemm_adds_as_joined and gemm_segments_add_as_joined; the three forward projections, whose
    // chains are a layer's width, always shared a launch.)
    bool f32_group = calls[0].dtype == CGPTX_F32;
    for (int i = 0; i < count; ++i) {
        const GemmArgs& g = calls[i];
        const Plan plan = make_plan(g);
        f32_group = f32_group && (count > 2 || plan.slices == 1);
        // An input gradient by itself on oblong tiles counts with those that they replace: what they promise is less than the error of a pair's
        // prediction. Pairs given up for it lost 5 to 27 per cent (17175 x 256 x 640 31.2 -> 39.5 us, with the bias 4469 x 1728 x 2880 92 -> 114).
        const int tile = plan.tile > 256 ? plan.replaced : plan.tile;
        const long tiles = Plan::tiles_of(g, tile);
        const bool f32 = g.dtype == CGPTX_F32;
        const long k_step = f32 ? kBK<float> : kBK<bf16_t>, k_tiles = (static_cast<long>(g.k) + k_step - 1) / k_step;
        separate += predicted_us(tile, tiles, plan.slices, k_tiles, static_cast<double>(plan.partial_bytes(g)) * 1e-6, f32,
                                 g.a_k_contiguous, g.b_k_contiguous, compute_units());
        if (g.a_sums != nullptr) separate += 6.0;  // two launches of their own
    }
    double best = separate;
    if (pair) {
        const long tiles_x = tiles_of_size(calls[0], 128, 128), tiles_w = tiles_of_size(calls[1], 128, 128), steps_x = k_steps_16bit(calls[0]), steps_w = k_steps_16bit(calls[1]);
        for (long s = 1; s <= 16 && tiles_w <= kTickets && (s == 1 || steps_w / s >= 8); ++s) {
            if (slice_steps(steps_w, s) * (s - 1) >= steps_w) continue;
            const double time = predicted_pair_us(tiles_x, steps_x, tiles_w, steps_w, s, compute_units(), best);
            if (time < best) {
                best = time;
                best_plan.joined = best_plan.pair = true;
                best_plan.tile[0] = 128;
                best_plan.slices = static_cast<int>(s);
            }
        }
        if (takes_oblong_tiles(calls[0]) && calls[0].a_segments.count == 0 && c_streams(calls[1], 2)) {
            const long tiles = tiles_of_size(calls[1], kPairWeightRows, kPairWeightColumns);
            const double most = best_plan.pair ? oblong_pair_has_to_beat(best, tiles_x, steps_x, tiles_w, steps_w, best_plan.slices, compute_units()) : best / 1.08;
            double least = most;
            for (const OblongCost& c : kOblongCosts) {
                // Of two that are predicted within 2 per cent the larger one: 5005 x 1024 x 2048 47.1 us on 192 x 256, 46.2 on 224 x 256.
                double own = std::min(most, 1.02 * least);
                for (long s = 1; s <= 3; ++s) {
                    if (s > 1 && slice_steps(steps_w, s) * (s - 1) >= steps_w) continue;
                    const double time = predicted_oblong_pair_us(c, Plan::tiles_of(calls[0], c.tile), steps_x, tiles, steps_w, s, compute_units());
                    if (time >= own) continue;
                    own = time;
                    least = std::min(least, time);
                    best = std::min(best, 1.08 * time);
                    best_plan.joined = best_plan.pair = true;
                    best_plan.tile[0] = c.tile;
                    best_plan.slices = static_cast<int>(s);
                }
            }
        }
    }
    if (fewest > kGroupBlocksPerUnit * units) return best_plan;
    for (int choice = 0; choice < 1 << count; ++choice) {
        double longest = 0.0, work = 0.0, lone_work = 0.0, blocks = 0.0, loops[kGroupCalls], counts[kGroupCalls];
        for (int i = 0; i < count; ++i) {
            const GemmArgs& g = calls[i];
            const bool f32 = g.dtype == CGPTX_F32, small = ((choice >> i) & 1) != 0;
            const long edge = small ? 32 : 64, k_step = f32 ? kBK<float> : kBK<bf16_t>;
            const double kt = static_cast<double>((static_cast<long>(g.k) + k_step - 1) / k_step);
            const double tiles = static_cast<double>((g.m + edge - 1) / edge) * static_cast<double>((g.n + edge - 1) / edge);
            const double lone = f32 ? (small ? 0.088 : 0.265) : small ? (!g.a_k_contiguous ? 0.1 : g.b_k_contiguous ? 0.07 : 0.085) : 0.12;
            const double shared = f32 ? lone : small ? 0.92 * lone : 0.11;
            const double loop = kt * lone;
            longest = std::max(longest, loop);
            work += tiles * kt * shared;
            lone_work += tiles * (loop + 3.5);
            blocks += tiles;
            loops[i] = loop;
            counts[i] = tiles;
        }
        if (blocks > kGroupBlocksPerUnit * units) continue;
        const double load = blocks / units;
        double two = load <= 1.0 ? longest : std::max(1.4 * longest, work / units * std::ceil(load) / load * (load > 4.0 && !f32_group ? 1.3 : 1.0));
        // fp32: the matrix cores are what binds, two tiles on a CU take twice as long, and a CU that has one long tile more than the
        // others ends that much later.
        for (int i = 0; i < count && f32_group; ++i) {
            double as_long = 0.0;
            for (int j = 0; j < count; ++j) as_long += loops[j] >= loops[i] ? counts[j] : 0.0;
            two = std::max(two, std::ceil(as_long / units) * loops[i]);
        }
        const double one = load <= 1.0 ? longest : std::max(longest, lone_work / units * std::ceil(load) / load);
        if (3.5 + std::min(one, two) < best) {
            best = 3.5 + std::min(one, two);
            best_plan.joined = true;
            best_plan.pair = false;
            best_plan.deep = one <= two;
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
        (g.a_segments.count > 0 && (!g.a_k_contiguous || g.b_k_contiguous)))
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
        if (copy_segments(segments, g.k, kSteps * kBK<T>, p.a_seg) != CGPTX_OK || segments.cols[segments.count - 1] % kBK<T> != 0) {
            clear_error();
            return false;
        }
    }
    return true;
}

// What a pair's weight gradient in K slices needs: partial tiles and counters.
struct FoldRoom {
    void* partial = nullptr;
    unsigned int* counters = nullptr;
    bool enough = false;
};
int fold_room(const GemmArgs& g, const GemmGroup& plan, hipStream_t stream, FoldRoom* room) {
    const int rows = pair_weight_rows(plan), columns = pair_weight_columns(plan);
    const std::size_t wanted = static_cast<std::size_t>(tiles_of_size(g, rows, columns)) * static_cast<std::size_t>(plan.slices) * fold_tile_bytes(rows, columns);
    room->partial = g.split_workspace;
    std::size_t held = g.split_workspace_bytes;
    if (!g.no_split)
        if (int s = scratch_up_to(stream, wanted, &room->partial, &held)) return s;
    room->counters = tickets(stream);
    room->enough = room->partial != nullptr && held >= wanted && room->counters != nullptr;
    return CGPTX_OK;
}

template <typename T>
int run_pair(const GemmArgs* calls, const GemmGroup& plan, hipStream_t stream) {
    if constexpr (std::is_same_v<T, float>) {
        return fail(CGPTX_RUNTIME, "gemm: fp32 calls run in groups of small tiles");
    } else {
        PairArgs pair{};
        for (int i = 0; i < 2; ++i) {
            KernelArgs& p = i == 0 ? pair.input : pair.weight;
            if (!joinable<T>(calls[i], p)) return fail(CGPTX_RUNTIME, "gemm: this call cannot be part of a group");
            const int rows = i == 0 ? tile_rows(plan.tile[0]) : pair_weight_rows(plan), columns = i == 0 ? tile_columns(plan.tile[0]) : pair_weight_columns(plan);
            p.tiles_m = (p.m + rows - 1) / rows;
            p.tiles_n = (p.n + columns - 1) / columns;
            p.slices = 1;
            p.k_tiles_per_slice = p.k_tiles;
        }
        KernelArgs& w = pair.weight;
        const GemmArgs& g = calls[1];
        w.a_sums = g.a_sums;
        w.a_sums_accumulate = g.a_sums_accumulate ? 1 : 0;
        if (plan.slices > 1) {
            FoldRoom room;
            if (int s = fold_room(g, plan, stream, &room)) return s;
            if (!room.enough) return fail(CGPTX_RUNTIME, "gemm: no room for the partial tiles of a pair");
            w.fold_partial = static_cast<unsigned char*>(room.partial);
            w.fold_tickets = room.counters;
            w.k_tiles_per_slice = static_cast<int>(slice_steps(w.k_tiles, plan.slices));
            w.slices = (w.k_tiles + w.k_tiles_per_slice - 1) / w.k_tiles_per_slice;
        }
        pair.input_tile = plan.tile[0];
        const bool oblong = plan.tile[0] > 256;
        if constexpr (std::is_same_v<T, bf16_t>) return oblong ? gemm_oblong_pair_bf16(pair, stream) : gemm_pair_bf16(pair, stream);
        else return oblong ? gemm_oblong_pair_f16(pair, stream) : gemm_pair_f16(pair, stream);
    }
}

template <typename T, int CALLS>
int run_group(const GemmArgs* calls, int count, const GemmGroup& plan, hipStream_t stream) {
    SmallGroup<CALLS> group{};
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
    if constexpr (std::is_same_v<T, bf16_t>) return gemm_small_bf16(group, blocks, plan.deep, stream);
    else if constexpr (std::is_same_v<T, f16_t>) return gemm_small_f16(group, blocks, plan.deep, stream);
    else return gemm_small_f32(group, blocks, plan.deep, stream);
}

template <typename T>
int run_joined(const GemmArgs* calls, int count, const GemmGroup& plan, hipStream_t stream) {
    if (plan.pair) return run_pair<T>(calls, plan, stream);
    return plan.few ? run_group<T, kFewCalls>(calls, count, plan, stream) : run_group<T, kGroupCalls>(calls, count, plan, stream);
}

}  // namespace

GemmGroup gemm_joins(const GemmArgs* calls, int count, hipStream_t stream, bool large_pairs) {
    if (count < 2 || count > kGroupCalls || forced_tile() != 0) return {};
    for (int i = 0; i < count; ++i) {
        if (calls[i].dtype != calls[0].dtype || !valid_dtype(calls[i].dtype)) return {};
        KernelArgs p;
        const bool fits = calls[i].dtype == CGPTX_F32 ? joinable<float>(calls[i], p)
                          : calls[i].dtype == CGPTX_F16 ? joinable<f16_t>(calls[i], p) : joinable<bf16_t>(calls[i], p);
        if (!fits) return {};
    }
    const bool pair = large_pairs && pairs(calls, count);
    GemmGroup group = plan_group(calls, count, pair);
    if (group.pair && group.slices > 1) {
        FoldRoom room;
        if (fold_room(calls[1], group, stream, &room) != CGPTX_OK || !room.enough) {
            clear_error();
            group = plan_group(calls, count, false);
        }
    }
    group.few = large_pairs && count <= kFewCalls;
    return group;
}

bool gemm_adds_as_joined(const GemmArgs* calls, int count, hipStream_t stream) {
    if (gemm_joins(calls, count, stream, false).joined) return true;
    for (int i = 0; i < count; ++i) {
        const Plan plan = make_plan(calls[i]);
        if (plan.tile > 64 || plan.slices != 1) return false;
    }
    return true;
}

bool gemm_segments_add_as_joined(const GemmArgs* calls, hipStream_t stream) {
    const GemmSegments& segments = calls[0].a_segments;
    std::size_t first = 0;
    for (int i = 0; i < segments.count; ++i) {
        GemmArgs pair[2] = {calls[0], calls[1 + i]};
        pair[0].a_segments = GemmSegments{};
        pair[0].a = segments.ptr[i];
        pair[0].lda = segments.ld[i];
        pair[0].k = segments.cols[i];
        pair[0].b = static_cast<const char*>(calls[0].b) + first * calls[0].ldb * dtype_size(calls[0].dtype);
        if (!gemm_adds_as_joined(pair, 2, stream)) return false;
        first += segments.cols[i];
    }
    return true;
}

int gemm_joined(const GemmArgs* calls, int count, const GemmGroup& group, hipStream_t stream) {
    if (!group.joined || count < 2 || count > (group.few ? kFewCalls : kGroupCalls)) return fail(CGPTX_RUNTIME, "gemm: these calls cannot share a launch");
    return dispatch_dtype(calls[0].dtype, [&]<typename T>() -> int { return run_joined<T>(calls, count, group, stream); });
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
    return launch_pad_rows(PadJob{dst, src, static_cast<long>(rows), static_cast<long>(ld), static_cast<int>(cols), static_cast<int>(pitch)}, nullptr,
                           dtype, stream);
}

int pad_rows_of_two(void* dst0, const void* src0, std::size_t rows0, void* dst1, const void* src1, std::size_t rows1, std::size_t cols,
                    std::size_t pitch, int dtype, hipStream_t stream) {
    const PadJob second{dst1, src1, static_cast<long>(rows1), static_cast<long>(cols), static_cast<int>(cols), static_cast<int>(pitch)};
    return launch_pad_rows(PadJob{dst0, src0, static_cast<long>(rows0), static_cast<long>(cols), static_cast<int>(cols), static_cast<int>(pitch)}, &second,
                           dtype, stream);
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
