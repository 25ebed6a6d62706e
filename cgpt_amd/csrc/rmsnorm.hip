// RMSNorm forward and backward for gfx950.
//
// Backward (reference semantics: src/ops/cpu/backward/rmsnorm_backward_cpu.cpp:86-133,
// CUDA dispatch src/ops/backward/rmsnorm_backward.cu:445-547):
//   r = 1/sqrt(mean(x^2)+eps);  c = (sum_j dy_j w_j x_j) r^3 / H
//   dx = dy w r - x c;          dgamma_j = sum_rows dy x r
//
// Fast path: one pass over x and dy. A wavefront owns 64/LPR rows at a time
// (LPR lanes per row, 128-bit accesses), keeps the row in registers between the
// reduction and the dx store, and accumulates its dgamma columns in registers.
// Per-block dgamma partials go to scratch and a second small kernel sums them in
// a fixed order, so the result does not depend on scheduling. HBM traffic is
// read x + read dy + write dx (+ partials, ~2% at 32768x1024).
//
// Generic path (any H, any alignment): row kernel with a second, cache-served
// read, then a column kernel over saved 1/rms.
#include "common.hpp"
#include "reduce.hpp"
#include "swiglu.hpp"

#include <cmath>
#include <limits>
#include <mutex>
#include <unordered_map>

namespace cgptx {
namespace {

constexpr int kThreads = 256;
constexpr int kWavesPerBlock = kThreads / kWave;
// Groups of four rows a wavefront of the dense norm + rotary kernel requests at a time: the backward pass holds three
// times the registers per group, and more of them in flight cost it more in resident wavefronts than they bring.
template <bool Backward>
constexpr int kRopeDenseUnroll = Backward ? 2 : 4;

// Rotary embedding applied to the rows on the way (rows are heads of head_dim = hidden elements):
// forward  y = rope(round(rmsnorm(x)));  backward  the incoming gradient is rotated back (and
// rounded) first. The roundings are those of the separate operators' stores, so the fused pass gives
// bit for bit what rmsnorm and rope give one after the other.
struct RopeArgs {
    const void* cos_cache;  // [positions, rotary_dim/2], element type of the rows
    const void* sin_cache;
    int heads;      // rows per token
    int sequence;   // tokens per sequence: position = offset + token % sequence
    int rotary_dim;
    int position_offset;
};

// Rotation of the pair (x, y) by +angle (forward) or -angle (backward); the arithmetic of the
// separate rotary kernels.
template <bool Inverse>
__device__ __forceinline__ void rotate_pair(float x, float y, float c, float s, float& ox, float& oy) {
    if constexpr (Inverse) {
        ox = fmaf(y, s, x * c);
        oy = fmaf(-x, s, y * c);
    } else {
        ox = fmaf(-y, s, x * c);
        oy = fmaf(x, s, y * c);
    }
}

template <typename T, bool Inverse>
__device__ __forceinline__ vec_t<float, kVec128<T>> rope_vector(vec_t<float, kVec128<T>> v, const RopeArgs& rope, int row,
                                                                int col) {
    constexpr int VEC = kVec128<T>;
    constexpr int HALF = VEC / 2;
    // What the separate operator would have read back from memory.
    v = vec_to_f32<T, VEC>(vec_from_f32<T, VEC>(v));
    if (col >= rope.rotary_dim) return v;
    const int token = row / rope.heads;
    const int pos = rope.position_offset + token % rope.sequence;
    const std::size_t index = static_cast<std::size_t>(pos) * (rope.rotary_dim / 2) + col / 2;
    const vec_t<float, HALF> c = vec_to_f32<T, HALF>(load_vec<T, HALF>(static_cast<const T*>(rope.cos_cache) + index));
    const vec_t<float, HALF> s = vec_to_f32<T, HALF>(load_vec<T, HALF>(static_cast<const T*>(rope.sin_cache) + index));
    vec_t<float, VEC> r;
#pragma unroll
    for (int p = 0; p < HALF; ++p) {
        float a, b;
        rotate_pair<Inverse>(v[2 * p], v[2 * p + 1], c[p], s[p], a, b);
        r[2 * p] = a;
        r[2 * p + 1] = b;
    }
    return r;
}

// ------------------------------------------------------------------ fast path
// Workgroup `block` of `blocks`.
template <typename T, int LPR, int K, bool Backward, bool Rope>
__device__ __forceinline__ void rmsnorm_rows(
    T* out,                         // dx (backward) or y (forward)
    float* __restrict__ partial,    // [blocks, H] dgamma partials (backward)
    const T* dy,                    // backward only; may be out itself
    const T* residual,              // backward only, optional: added to dx (may be out itself)
    const T* __restrict__ x, const T* __restrict__ w, int rows, int hidden, float inv_hidden, float eps,
    const RopeArgs& rope, int block, int blocks) {
    constexpr int VEC = kVec128<T>;
    constexpr int RPW = kWave / LPR;  // rows per wavefront iteration
    using F = vec_t<float, VEC>;

    const int lane = threadIdx.x & (kWave - 1);
    const int wave = threadIdx.x / kWave;
    const int sub = lane % LPR;   // lane within the row
    const int rsel = lane / LPR;  // which of the RPW rows

    F wv[K];
    F acc[K];
    bool live[K];
#pragma unroll
    for (int c = 0; c < K; ++c) {
        const int col = (c * LPR + sub) * VEC;
        live[c] = col < hidden;
        wv[c] = live[c] ? vec_to_f32<T, VEC>(load_vec<T, VEC>(w + col)) : F(0.0f);
        acc[c] = F(0.0f);
    }

    const int groups = (rows + RPW - 1) / RPW;
    const int wave_global = block * kWavesPerBlock + wave;
    const int wave_count = blocks * kWavesPerBlock;
    for (int g = wave_global; g < groups; g += wave_count) {
        const int row = g * RPW + rsel;
        const bool row_live = row < rows;
        const std::size_t base = static_cast<std::size_t>(row) * hidden;
        F xv[K], gv[K];
        vec_t<T, VEC> rv[K];  // residual, requested with the other operands: one memory round trip per row
#pragma unroll
        for (int c = 0; c < K; ++c) {
            const int col = (c * LPR + sub) * VEC;
            if (row_live && live[c]) {
                xv[c] = vec_to_f32<T, VEC>(load_vec<T, VEC>(x + base + col));
                if constexpr (Backward) {
                    if (residual != nullptr) rv[c] = load_vec<T, VEC>(residual + base + col);
                    gv[c] = vec_to_f32<T, VEC>(load_vec<T, VEC>(dy + base + col));
                    if constexpr (Rope) gv[c] = vec_to_f32<T, VEC>(vec_from_f32<T, VEC>(rope_vector<T, true>(gv[c], rope, row, col)));
                }
            } else {
                xv[c] = F(0.0f);
                if constexpr (Backward) gv[c] = F(0.0f);
            }
        }
        float ss = 0.0f, dd = 0.0f;
#pragma unroll
        for (int c = 0; c < K; ++c) {
#pragma unroll
            for (int e = 0; e < VEC; ++e) {
                ss = fmaf(xv[c][e], xv[c][e], ss);
                if constexpr (Backward) dd = fmaf(gv[c][e] * wv[c][e], xv[c][e], dd);
            }
        }
        ss = wave_sum<LPR>(ss);
        const float inv = 1.0f / sqrtf(ss * inv_hidden + eps);
        if constexpr (Backward) {
            dd = wave_sum<LPR>(dd);
            const float corr = dd * inv * inv * inv * inv_hidden;
#pragma unroll
            for (int c = 0; c < K; ++c) {
                F r;
#pragma unroll
                for (int e = 0; e < VEC; ++e) {
                    r[e] = gv[c][e] * wv[c][e] * inv - xv[c][e] * corr;
                    acc[c][e] = fmaf(gv[c][e], xv[c][e] * inv, acc[c][e]);
                }
                const int col = (c * LPR + sub) * VEC;
                if (row_live && live[c]) {
                    if (residual != nullptr) r += vec_to_f32<T, VEC>(rv[c]);
                    store_vec<T, VEC>(out + base + col, vec_from_f32<T, VEC>(r));
                }
            }
        } else {
#pragma unroll
            for (int c = 0; c < K; ++c) {
                F r;
#pragma unroll
                for (int e = 0; e < VEC; ++e) r[e] = xv[c][e] * inv * wv[c][e];
                const int col = (c * LPR + sub) * VEC;
                if (row_live && live[c]) {
                    if constexpr (Rope) r = rope_vector<T, false>(r, rope, row, col);
                    store_vec<T, VEC>(out + base + col, vec_from_f32<T, VEC>(r));
                }
            }
        }
    }

    if constexpr (Backward) {
        // Fold the RPW row slots of the wavefront, then the block's wavefronts.
        __shared__ float stage[kWavesPerBlock][LPR * K * VEC];
#pragma unroll
        for (int c = 0; c < K; ++c) {
#pragma unroll
            for (int e = 0; e < VEC; ++e) {
                float v = acc[c][e];
#pragma unroll
                for (int offset = LPR; offset < kWave; offset <<= 1) v += __shfl_xor(v, offset, kWave);
                if (rsel == 0) stage[wave][(c * LPR + sub) * VEC + e] = v;
            }
        }
        __syncthreads();
        for (int col = threadIdx.x; col < hidden; col += kThreads) {
            float v = 0.0f;
#pragma unroll
            for (int s = 0; s < kWavesPerBlock; ++s) v += stage[s][col];
            partial[static_cast<std::size_t>(block) * hidden + col] = v;
        }
    }
}

template <typename T, int LPR, int K, bool Backward>
__global__ __launch_bounds__(kThreads) void rmsnorm_rows_kernel(T* out, float* __restrict__ partial, const T* dy, const T* residual,
                                                                const T* __restrict__ x, const T* __restrict__ w, int rows,
                                                                int hidden, float inv_hidden, float eps) {
    rmsnorm_rows<T, LPR, K, Backward, false>(out, partial, dy, residual, x, w, rows, hidden, inv_hidden, eps, RopeArgs{}, blockIdx.x,
                                             gridDim.x);
}

// The fused per-head norm + rotary pass at the shape a training step gives it: rows of exactly 16 vectors (head_dim 128
// in 16-bit storage), all of them rotated, a multiple of four rows, tensors and tables below 4 GiB. Same arithmetic,
// in the same order, as rmsnorm_rows<T, 16, 1, Backward, true>; what differs is the bookkeeping, which at 2 KiB
// of rows per wavefront and trip is what that kernel spends most of its instructions on: no per-lane predicates, 32-bit
// byte offsets that advance by a constant, and the token position carried from trip to trip (head index and position
// advance by constants with one carry each) instead of two integer divisions per trip. A trip requests U groups of
// four rows before it uses the first, so that a wavefront has U times the bytes in flight.
template <typename T, bool Backward, int U>
__device__ __forceinline__ void rmsnorm_rope_dense(
    T* out, float* __restrict__ partial, const T* dy /* may be out itself */, const T* __restrict__ x,
    const T* __restrict__ w, int rows, float inv_hidden, float eps, const RopeArgs& rope, int block, int blocks) {
    constexpr int VEC = kVec128<T>;
    constexpr int HALF = VEC / 2;
    constexpr int LPR = 16;
    constexpr int RPW = kWave / LPR;
    constexpr int HIDDEN = LPR * VEC;
    using F = vec_t<float, VEC>;
    using H = vec_t<float, HALF>;

    const int lane = threadIdx.x & (kWave - 1);
    const int wave = threadIdx.x / kWave;
    const int sub = lane % LPR;
    const int rsel = lane / LPR;
    const F wv = vec_to_f32<T, VEC>(load_vec<T, VEC>(w + sub * VEC));
    F acc(0.0f);

    const int groups = rows / RPW;
    const int wave_global = block * kWavesPerBlock + wave;
    const int wave_count = blocks * kWavesPerBlock;
    const int first_row = wave_global * RPW + rsel;
    const int stride_rows = wave_count * RPW;
    int head = first_row % rope.heads;
    int pos = (first_row / rope.heads) % rope.sequence;
    const int head_step = stride_rows % rope.heads;
    const int pos_step = (stride_rows / rope.heads) % rope.sequence;
    unsigned offset = (static_cast<unsigned>(first_row) * HIDDEN + sub * VEC) * static_cast<unsigned>(sizeof(T));
    const unsigned offset_step = static_cast<unsigned>(stride_rows) * HIDDEN * static_cast<unsigned>(sizeof(T));
    const unsigned table_lane = sub * HALF * static_cast<unsigned>(sizeof(T));
    constexpr unsigned kTableRow = (HIDDEN / 2) * sizeof(T);
    const auto at = [](const void* base, unsigned bytes) {
        return reinterpret_cast<const T*>(static_cast<const char*>(base) + bytes);
    };

    struct Fetched {
        vec_t<T, VEC> x, g;
        vec_t<T, HALF> c, s;
        unsigned offset;
    };
    // Requests the operands of the group at `offset` / `pos` and moves both on to the wavefront's next group.
    const auto fetch = [&]() {
        Fetched f;
        const unsigned table = static_cast<unsigned>(rope.position_offset + pos) * kTableRow + table_lane;
        f.c = load_vec<T, HALF>(at(rope.cos_cache, table));
        f.s = load_vec<T, HALF>(at(rope.sin_cache, table));
        f.x = load_vec<T, VEC>(at(x, offset));
        if constexpr (Backward) f.g = load_vec<T, VEC>(at(dy, offset));
        f.offset = offset;
        offset += offset_step;
        head += head_step;
        const int carry = head >= rope.heads ? 1 : 0;
        head -= carry ? rope.heads : 0;
        pos += pos_step + carry;
        pos -= pos >= rope.sequence ? rope.sequence : 0;
        return f;
    };
    const auto finish = [&](const Fetched& f) {
        const H c = vec_to_f32<T, HALF>(f.c);
        const H s = vec_to_f32<T, HALF>(f.s);
        const F xv = vec_to_f32<T, VEC>(f.x);
        F gv;
        if constexpr (Backward) {
            // The incoming gradient rotated back and rounded: what the separate rotary operator would have stored.
            const F raw = vec_to_f32<T, VEC>(f.g);
            F turned;
#pragma unroll
            for (int p = 0; p < HALF; ++p) {
                float a, b;
                rotate_pair<true>(raw[2 * p], raw[2 * p + 1], c[p], s[p], a, b);
                turned[2 * p] = a;
                turned[2 * p + 1] = b;
            }
            gv = vec_to_f32<T, VEC>(vec_from_f32<T, VEC>(turned));
        }
        float ss = 0.0f, dd = 0.0f;
#pragma unroll
        for (int e = 0; e < VEC; ++e) {
            ss = fmaf(xv[e], xv[e], ss);
            if constexpr (Backward) dd = fmaf(gv[e] * wv[e], xv[e], dd);
        }
        ss = wave_sum<LPR>(ss);
        const float inv = 1.0f / sqrtf(ss * inv_hidden + eps);
        F r;
        if constexpr (Backward) {
            dd = wave_sum<LPR>(dd);
            const float corr = dd * inv * inv * inv * inv_hidden;
#pragma unroll
            for (int e = 0; e < VEC; ++e) {
                r[e] = gv[e] * wv[e] * inv - xv[e] * corr;
                acc[e] = fmaf(gv[e], xv[e] * inv, acc[e]);
            }
        } else {
            F y;
#pragma unroll
            for (int e = 0; e < VEC; ++e) y[e] = xv[e] * inv * wv[e];
            y = vec_to_f32<T, VEC>(vec_from_f32<T, VEC>(y));  // the norm's own store, before the rotation
#pragma unroll
            for (int p = 0; p < HALF; ++p) {
                float a, b;
                rotate_pair<false>(y[2 * p], y[2 * p + 1], c[p], s[p], a, b);
                r[2 * p] = a;
                r[2 * p + 1] = b;
            }
        }
        store_vec<T, VEC>(const_cast<T*>(at(out, f.offset)), vec_from_f32<T, VEC>(r));
    };

    int g = wave_global;
    for (; g + (U - 1) * wave_count < groups; g += U * wave_count) {
        Fetched f[U];
#pragma unroll
        for (int u = 0; u < U; ++u) f[u] = fetch();
        __builtin_amdgcn_sched_barrier(0);  // every request of the trip goes out before the first use
#pragma unroll
        for (int u = 0; u < U; ++u) finish(f[u]);
    }
    for (; g < groups; g += wave_count) finish(fetch());

    if constexpr (Backward) {
        // Fold the four row slots of the wavefront, then the block's wavefronts.
        __shared__ float stage[kWavesPerBlock][HIDDEN];
#pragma unroll
        for (int e = 0; e < VEC; ++e) {
            float v = acc[e];
#pragma unroll
            for (int across = LPR; across < kWave; across <<= 1) v += __shfl_xor(v, across, kWave);
            if (rsel == 0) stage[wave][sub * VEC + e] = v;
        }
        __syncthreads();
        for (int col = threadIdx.x; col < HIDDEN; col += kThreads) {
            float v = 0.0f;
#pragma unroll
            for (int s = 0; s < kWavesPerBlock; ++s) v += stage[s][col];
            partial[static_cast<std::size_t>(block) * HIDDEN + col] = v;
        }
    }
}

// q and k in one launch: the first blocks_q workgroups take q's rows, the others k's. In a call of a few hundred tokens each of the
// two is a launch of 4.5 us for less than one of work.
template <typename T>
struct RopeRows {
    T* out;
    float* partial;
    const T* dy;
    const T* x;
    const T* w;
    int rows, heads;
};
// SWIGLU: the workgroups behind them take the SwiGLU product of the feed-forward branch or its gradient, which neither reads nor writes
// what the attention branch does: a step of 3 x 100 tokens gives each of the two launches 3 - 4 us for less than one of work.
template <typename T>
struct SwigluRows {
    T* out;
    const T* grad_activated;  // backward
    const T* gate_up;
    unsigned int rows, hidden;
};
// LPR: lanes per row, 16, or 32 for heads of 128 in fp32 (three launches before, q's norm, k's and the rotation: 14.4 us of a step of
// 256 tokens in each direction and layer, now 4.8).
template <typename T, int LPR, bool Backward, bool Dense, bool SWIGLU>
__global__ __launch_bounds__(kThreads) void rmsnorm_rope_pair_kernel(RopeRows<T> q, RopeRows<T> k, int blocks_q, int blocks_k, int hidden,
                                                                     float inv_hidden, float eps, RopeArgs rope, SwigluRows<T> swiglu) {
    if constexpr (SWIGLU) {
        const int block = static_cast<int>(blockIdx.x) - blocks_q - blocks_k, blocks = static_cast<int>(gridDim.x) - blocks_q - blocks_k;
        if (block >= 0) {
            const std::size_t row_elems = swiglu.hidden;
            const unsigned int row_vectors = swiglu.hidden / kVec128<T>;
            if constexpr (Backward)
                swiglu_backward_vectors<T, false, false, 1>(swiglu.out, swiglu.out + row_elems, swiglu.grad_activated, swiglu.gate_up,
                                                            swiglu.gate_up + row_elems, static_cast<std::size_t>(swiglu.rows) * row_vectors,
                                                            row_vectors, -1, 2 * row_elems, block, blocks);
            else
                swiglu_forward_packed_vectors<T>(swiglu.out, swiglu.gate_up, swiglu.rows, swiglu.hidden, block, blocks);
            return;
        }
    }
    const bool second = static_cast<int>(blockIdx.x) >= blocks_q;
    const int block = static_cast<int>(blockIdx.x) - (second ? blocks_q : 0);
    const int blocks = second ? blocks_k : blocks_q;
    const RopeRows<T> of = second ? k : q;
    rope.heads = of.heads;
    if constexpr (Dense)
        rmsnorm_rope_dense<T, Backward, kRopeDenseUnroll<Backward>>(of.out, of.partial, of.dy, of.x, of.w, of.rows, inv_hidden, eps, rope,
                                                                    block, blocks);
    else
        rmsnorm_rows<T, LPR, 1, Backward, true>(of.out, of.partial, of.dy, nullptr, of.x, of.w, of.rows, hidden, inv_hidden, eps, rope,
                                               block, blocks);
}

// Two RMSNorms of the same rows with different weights (the block's attention and feed-forward norms
// both read the block input): one pass reads x once.
//   forward   y_a = x r w_a,  y_f = x r w_f
//   backward  dx = g r - x (sum_j g_j x_j) r^3 / H + residual  with g = dy_a w_a + dy_f w_f  (the two
//             gradients add up before the row reduction: the norm is the same for both),
//             dgamma_a = sum_rows dy_a x r,  dgamma_f = sum_rows dy_f x r
template <typename T, int LPR, int K, bool Backward>
__global__ __launch_bounds__(kThreads) void rmsnorm_dual_rows_kernel(
    T* out_a,                       // y_a (forward) or dx (backward)
    T* out_f,                       // y_f (forward)
    float* __restrict__ partial_a,  // [gridDim.x, H] dgamma partials (backward)
    float* __restrict__ partial_f,
    const T* __restrict__ dy_a, const T* __restrict__ dy_f,  // backward only
    const T* residual,              // backward only, optional: added to dx (may be out_a itself)
    const T* __restrict__ x, const T* __restrict__ w_a, const T* __restrict__ w_f, int rows, int hidden,
    float inv_hidden, float eps) {
    constexpr int VEC = kVec128<T>;
    constexpr int RPW = kWave / LPR;
    using F = vec_t<float, VEC>;
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = threadIdx.x / kWave;
    const int sub = lane % LPR;
    const int rsel = lane / LPR;

    F wa[K], wf[K], acc_a[K], acc_f[K];
    bool live[K];
#pragma unroll
    for (int c = 0; c < K; ++c) {
        const int col = (c * LPR + sub) * VEC;
        live[c] = col < hidden;
        wa[c] = live[c] ? vec_to_f32<T, VEC>(load_vec<T, VEC>(w_a + col)) : F(0.0f);
        wf[c] = live[c] ? vec_to_f32<T, VEC>(load_vec<T, VEC>(w_f + col)) : F(0.0f);
        acc_a[c] = F(0.0f);
        acc_f[c] = F(0.0f);
    }
    const int groups = (rows + RPW - 1) / RPW;
    const int wave_global = blockIdx.x * kWavesPerBlock + wave;
    const int wave_count = gridDim.x * kWavesPerBlock;
    for (int g = wave_global; g < groups; g += wave_count) {
        const int row = g * RPW + rsel;
        const bool row_live = row < rows;
        const std::size_t base = static_cast<std::size_t>(row) * hidden;
        F xv[K], ga[K], gf[K];
        vec_t<T, VEC> rv[K];  // residual, requested with the other operands: one memory round trip per row
#pragma unroll
        for (int c = 0; c < K; ++c) {
            const int col = (c * LPR + sub) * VEC;
            const bool on = row_live && live[c];
            xv[c] = on ? vec_to_f32<T, VEC>(load_vec<T, VEC>(x + base + col)) : F(0.0f);
            if constexpr (Backward) {
                ga[c] = on ? vec_to_f32<T, VEC>(load_vec<T, VEC>(dy_a + base + col)) : F(0.0f);
                gf[c] = on ? vec_to_f32<T, VEC>(load_vec<T, VEC>(dy_f + base + col)) : F(0.0f);
                if (on && residual != nullptr) rv[c] = load_vec<T, VEC>(residual + base + col);
            }
        }
        float ss = 0.0f, dd = 0.0f;
#pragma unroll
        for (int c = 0; c < K; ++c) {
#pragma unroll
            for (int e = 0; e < VEC; ++e) {
                ss = fmaf(xv[c][e], xv[c][e], ss);
                if constexpr (Backward) dd = fmaf(fmaf(ga[c][e], wa[c][e], gf[c][e] * wf[c][e]), xv[c][e], dd);
            }
        }
        ss = wave_sum<LPR>(ss);
        const float inv = 1.0f / sqrtf(ss * inv_hidden + eps);
        if constexpr (Backward) {
            dd = wave_sum<LPR>(dd);
            const float corr = dd * inv * inv * inv * inv_hidden;
#pragma unroll
            for (int c = 0; c < K; ++c) {
                F r;
#pragma unroll
                for (int e = 0; e < VEC; ++e) {
                    const float scaled = xv[c][e] * inv;
                    r[e] = fmaf(ga[c][e], wa[c][e], gf[c][e] * wf[c][e]) * inv - xv[c][e] * corr;
                    acc_a[c][e] = fmaf(ga[c][e], scaled, acc_a[c][e]);
                    acc_f[c][e] = fmaf(gf[c][e], scaled, acc_f[c][e]);
                }
                const int col = (c * LPR + sub) * VEC;
                if (row_live && live[c]) {
                    if (residual != nullptr) r += vec_to_f32<T, VEC>(rv[c]);
                    store_vec<T, VEC>(out_a + base + col, vec_from_f32<T, VEC>(r));
                }
            }
        } else {
#pragma unroll
            for (int c = 0; c < K; ++c) {
                F ra, rf;
#pragma unroll
                for (int e = 0; e < VEC; ++e) {
                    ra[e] = xv[c][e] * inv * wa[c][e];
                    rf[e] = xv[c][e] * inv * wf[c][e];
                }
                const int col = (c * LPR + sub) * VEC;
                if (row_live && live[c]) {
                    store_vec<T, VEC>(out_a + base + col, vec_from_f32<T, VEC>(ra));
                    store_vec<T, VEC>(out_f + base + col, vec_from_f32<T, VEC>(rf));
                }
            }
        }
    }
    if constexpr (Backward) {
        // Fold the RPW row slots of the wavefront, then the block's wavefronts; first one weight, then the other.
        __shared__ float stage[kWavesPerBlock][LPR * K * VEC];
#pragma unroll
        for (int which = 0; which < 2; ++which) {
#pragma unroll
            for (int c = 0; c < K; ++c) {
#pragma unroll
                for (int e = 0; e < VEC; ++e) {
                    float v = which == 0 ? acc_a[c][e] : acc_f[c][e];
#pragma unroll
                    for (int offset = LPR; offset < kWave; offset <<= 1) v += __shfl_xor(v, offset, kWave);
                    if (rsel == 0) stage[wave][(c * LPR + sub) * VEC + e] = v;
                }
            }
            __syncthreads();
            float* partial = which == 0 ? partial_a : partial_f;
            for (int col = threadIdx.x; col < hidden; col += kThreads) {
                float v = 0.0f;
#pragma unroll
                for (int s = 0; s < kWavesPerBlock; ++s) v += stage[s][col];
                partial[static_cast<std::size_t>(blockIdx.x) * hidden + col] = v;
            }
            __syncthreads();
        }
    }
}

// --------------------------------------------------------------- generic path
template <typename T, bool Backward>
__global__ __launch_bounds__(kThreads) void rmsnorm_row_generic_kernel(
    T* out, float* __restrict__ inv_rms, const T* __restrict__ dy, const T* residual /* may be null or alias out */, const T* __restrict__ x,
    const T* __restrict__ w, int rows, int hidden, float inv_hidden, float eps) {
    __shared__ float red[2][kWavesPerBlock];
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = threadIdx.x / kWave;
    for (int row = blockIdx.x; row < rows; row += gridDim.x) {
        const std::size_t base = static_cast<std::size_t>(row) * hidden;
        float ss = 0.0f, dd = 0.0f;
        for (int col = threadIdx.x; col < hidden; col += kThreads) {
            const float xv = to_f32(x[base + col]);
            ss = fmaf(xv, xv, ss);
            if constexpr (Backward) dd = fmaf(to_f32(dy[base + col]) * to_f32(w[col]), xv, dd);
        }
        ss = wave_sum(ss);
        dd = wave_sum(dd);
        __syncthreads();  // protects red[] against the previous iteration's readers
        if (lane == 0) {
            red[0][wave] = ss;
            red[1][wave] = dd;
        }
        __syncthreads();
        ss = 0.0f;
        dd = 0.0f;
#pragma unroll
        for (int s = 0; s < kWavesPerBlock; ++s) {
            ss += red[0][s];
            dd += red[1][s];
        }
        const float inv = 1.0f / sqrtf(ss * inv_hidden + eps);
        if constexpr (Backward) {
            const float corr = dd * inv * inv * inv * inv_hidden;
            if (threadIdx.x == 0) inv_rms[row] = inv;
            for (int col = threadIdx.x; col < hidden; col += kThreads) {
                const float gradient = to_f32(dy[base + col]) * to_f32(w[col]) * inv - to_f32(x[base + col]) * corr;
                out[base + col] = from_f32<T>(residual != nullptr ? gradient + to_f32(residual[base + col]) : gradient);
            }
        } else {
            for (int col = threadIdx.x; col < hidden; col += kThreads) {
                out[base + col] = from_f32<T>(to_f32(x[base + col]) * inv * to_f32(w[col]));
            }
        }
    }
}

// partial[blockIdx.y, col] = sum over this block's row slice of dy*x*inv_rms.
template <typename T>
__global__ __launch_bounds__(kThreads) void rmsnorm_dgamma_generic_kernel(
    float* __restrict__ partial, const T* __restrict__ dy, const T* __restrict__ x,
    const float* __restrict__ inv_rms, int rows, int hidden, int rows_per_slice) {
    __shared__ float stage[kWavesPerBlock][kWave];
    const int lane = threadIdx.x & (kWave - 1);
    const int slice = threadIdx.x / kWave;
    const int col = blockIdx.x * kWave + lane;
    const int row_begin = blockIdx.y * rows_per_slice;
    const int row_end = min(rows, row_begin + rows_per_slice);
    float v = 0.0f;
    if (col < hidden) {
        for (int row = row_begin + slice; row < row_end; row += kWavesPerBlock) {
            const std::size_t index = static_cast<std::size_t>(row) * hidden + col;
            v = fmaf(to_f32(dy[index]), to_f32(x[index]) * inv_rms[row], v);
        }
    }
    stage[slice][lane] = v;
    __syncthreads();
    if (slice == 0 && col < hidden) {
        float total = 0.0f;
#pragma unroll
        for (int s = 0; s < kWavesPerBlock; ++s) total += stage[s][lane];
        partial[static_cast<std::size_t>(blockIdx.y) * hidden + col] = total;
    }
}

// ------------------------------------------------------------------- dispatch
struct FastShape {
    int lpr = 0;
    int k = 0;
};

template <typename T>
FastShape pick_fast_shape(int hidden) {
    constexpr int VEC = kVec128<T>;
    if (hidden % VEC != 0) return {};
    const int vecs = hidden / VEC;
    if (vecs <= 16) return {16, 1};
    if (vecs <= 32) return {32, 1};
    if (vecs <= 64) return {64, 1};
    if (vecs <= 128) return {64, 2};
    if (vecs <= 256) return {64, 4};
    return {};
}

// Whether rmsnorm_rope_dense serves the pass: rows of exactly 16 vectors, all of them rotated, whole groups of
// four rows, and every byte offset it forms (tensor and table) below 2^32.
template <typename T>
bool rope_dense(int rows, int hidden, const RopeArgs& rope) {
    constexpr int VEC = kVec128<T>;
    const unsigned long long tensor_bytes = static_cast<unsigned long long>(rows) * hidden * sizeof(T);
    const unsigned long long table_bytes =
        (static_cast<unsigned long long>(rope.position_offset) + rope.sequence) * (hidden / 2) * sizeof(T);
    return hidden == 16 * VEC && rope.rotary_dim == hidden && rows % 4 == 0 && tensor_bytes < (1ull << 32) &&
           table_bytes < (1ull << 32);
}

template <typename T, bool Backward>
int launch_fast(const FastShape shape, T* out, float* partial, const T* dy, const T* residual, const T* x, const T* w,
                int rows, int hidden, float eps, int blocks, hipStream_t stream) {
    const float inv_hidden = 1.0f / static_cast<float>(hidden);
#define CGPTX_RMS_CASE(L, KK)                                                                             \
    if (shape.lpr == L && shape.k == KK) {                                                                \
        hipLaunchKernelGGL((rmsnorm_rows_kernel<T, L, KK, Backward>), dim3(blocks), dim3(kThreads), 0,   \
                           stream, out, partial, dy, residual, x, w, rows, hidden, inv_hidden, eps);                \
        return CGPTX_OK;                                                                                  \
    }
    CGPTX_RMS_CASE(16, 1)
    CGPTX_RMS_CASE(32, 1)
    CGPTX_RMS_CASE(64, 1)
    CGPTX_RMS_CASE(64, 2)
    CGPTX_RMS_CASE(64, 4)
#undef CGPTX_RMS_CASE
    return fail(CGPTX_RUNTIME, "rmsnorm: no kernel for shape");
}

// The kernel launch_fast would launch (null when there is none).
template <typename T, bool Backward>
const void* fast_kernel(const FastShape shape) {
#define CGPTX_RMS_CASE(L, KK) \
    if (shape.lpr == L && shape.k == KK) return reinterpret_cast<const void*>(&rmsnorm_rows_kernel<T, L, KK, Backward>);
    CGPTX_RMS_CASE(16, 1)
    CGPTX_RMS_CASE(32, 1)
    CGPTX_RMS_CASE(64, 1)
    CGPTX_RMS_CASE(64, 2)
    CGPTX_RMS_CASE(64, 4)
#undef CGPTX_RMS_CASE
    return nullptr;
}

// Blocks of `kernel` the device holds at once. The row kernels are grid-stride loops with equal
// shares: launched with more blocks than fit, the surplus would run as a second, mostly idle round.
int resident_blocks(const void* kernel) {
    static std::mutex guard;
    static std::unordered_map<const void*, int> known;
    std::lock_guard<std::mutex> lock(guard);
    auto found = known.find(kernel);
    if (found == known.end()) {
        int per_cu = 0;
        if (kernel == nullptr || hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, kThreads, 0) != hipSuccess ||
            per_cu < 1) {
            (void)hipGetLastError();
            per_cu = 1;
        }
        found = known.emplace(kernel, per_cu).first;
    }
    return found->second * compute_units();
}

int fast_blocks(const FastShape shape, int rows, const void* kernel) {
    const int rpw = kWave / shape.lpr;
    const long groups = (static_cast<long>(rows) + rpw - 1) / rpw;
    const long wanted = (groups + kWavesPerBlock - 1) / kWavesPerBlock;
    const long cap = resident_blocks(kernel);
    return static_cast<int>(wanted < cap ? wanted : cap);
}

int validate(const void* a, const void* b, const void* c, std::size_t rows, std::size_t hidden, float eps, int dtype,
             const char* name) {
    if (!valid_dtype(dtype)) return fail(CGPTX_INVALID_ARGUMENT, std::string(name) + ": unsupported dtype");
    if (!std::isfinite(eps) || eps <= 0.0f)
        return fail(CGPTX_INVALID_ARGUMENT, std::string(name) + ": epsilon must be finite and positive");
    if (a == nullptr || b == nullptr || c == nullptr)
        return fail(CGPTX_INVALID_ARGUMENT, std::string(name) + ": null tensor");
    if (rows == 0 || hidden == 0) return fail(CGPTX_INVALID_ARGUMENT, std::string(name) + ": empty shape");
    if (rows > static_cast<std::size_t>(std::numeric_limits<int>::max()) ||
        hidden > static_cast<std::size_t>(std::numeric_limits<int>::max()))
        return fail(CGPTX_INVALID_ARGUMENT, std::string(name) + ": dimensions exceed supported range");
    return CGPTX_OK;
}

// Lanes per row of the norm + rotary kernels (0: not served): rows of up to 16 vectors, in fp32 of up to 32.
template <typename T>
int pair_lanes(int head_dim) {
    const FastShape shape = pick_fast_shape<T>(head_dim);
    return shape.k == 1 && (shape.lpr == 16 || (shape.lpr == 32 && std::is_same_v<T, float>)) ? shape.lpr : 0;
}
}  // namespace

bool rmsnorm_rope_fusable(const void* a, const void* b, const void* c, const void* weight, const void* cos_cache,
                          const void* sin_cache, std::size_t head_dim, std::size_t rotary_dim, int dtype) {
    if (!valid_dtype(dtype) || head_dim == 0 || head_dim > 4096) return false;
    const std::size_t elem = dtype_size(dtype), vec = 16 / elem;
    bool shape_ok = false;
    dispatch_dtype(dtype, [&]<typename T>() -> int {
        shape_ok = pair_lanes<T>(static_cast<int>(head_dim)) != 0;
        return CGPTX_OK;
    });
    const auto half_aligned = [&](const void* p) { return (reinterpret_cast<std::uintptr_t>(p) % (vec / 2 * elem)) == 0; };
    return shape_ok && rotary_dim % vec == 0 && rotary_dim <= head_dim && is_aligned16(a) && is_aligned16(b) &&
           (c == nullptr || is_aligned16(c)) && is_aligned16(weight) && half_aligned(cos_cache) && half_aligned(sin_cache);
}

namespace {
RopeArgs make_rope(const void* cos_cache, const void* sin_cache, std::size_t heads, std::size_t sequence,
                   std::size_t rotary_dim, std::size_t position_offset) {
    return RopeArgs{cos_cache, sin_cache, static_cast<int>(heads), static_cast<int>(sequence), static_cast<int>(rotary_dim),
                    static_cast<int>(position_offset)};
}
}  // namespace

// Memory for a pass's partial sums: from the sink when one is given and has room (the reductions are then recorded
// and run later by the caller), else from the per-stream arena (the reductions then run at once).
int partial_memory(ColumnReduceSink* sink, hipStream_t stream, std::size_t bytes, void** out, bool* deferred) {
    *out = sink != nullptr ? sink->take(bytes) : nullptr;
    *deferred = *out != nullptr;
    return *deferred ? CGPTX_OK : scratch(stream, bytes, out);
}

// dw[h] = column sums of partial[blocks, h]: a small launch now, or an entry in the sink.
template <typename T>
int reduce_columns(ColumnReduceSink* sink, bool deferred, T* dw, const float* partial, int blocks, int h, int dtype,
                   hipStream_t stream) {
    if (deferred) {
        sink->entries.push_back(ColumnReduceEntry{partial, dw, blocks, h, dtype});
        return CGPTX_OK;
    }
    launch_column_partial_reduce<T>(dw, partial, blocks, h, 0, stream);
    CGPTX_LAUNCH_CHECK();
    return CGPTX_OK;
}

int run_column_reductions(const ColumnReduceEntry* table, const std::vector<ColumnReduceEntry>& entries, const MeanEntry& mean, hipStream_t stream) {
    if (entries.empty()) return mean.rows != 0 ? mean_reduce(mean.loss, mean.row_losses, mean.rows, stream) : CGPTX_OK;
    int groups = 1;
    for (const ColumnReduceEntry& e : entries) groups = std::max(groups, (e.hidden + finish_columns(e.hidden) - 1) / finish_columns(e.hidden));
    const auto count = static_cast<unsigned int>(entries.size());
    hipLaunchKernelGGL(column_partial_reduce_table_kernel, dim3(groups, count + (mean.rows != 0 ? 1u : 0u)), dim3(kFinishThreads), 0, stream, table,
                       static_cast<int>(count), compute_units(), mean);
    CGPTX_LAUNCH_CHECK();
    return CGPTX_OK;
}

namespace {
// Workgroups that the rows fill, 64 / lanes of them a wavefront.
int pair_blocks(int rows, int lanes) {
    const long rows_per_block = kWave / lanes * kWavesPerBlock;
    return static_cast<int>((static_cast<long>(rows) + rows_per_block - 1) / rows_per_block);
}
template <typename T, bool Backward>
using PairKernel = void (*)(RopeRows<T>, RopeRows<T>, int, int, int, float, float, RopeArgs, SwigluRows<T>);
template <typename T, bool Backward>
PairKernel<T, Backward> pair_kernel(int lanes, bool dense, bool swiglu) {
    if constexpr (std::is_same_v<T, float>) {
        if (lanes == 32) return swiglu ? rmsnorm_rope_pair_kernel<T, 32, Backward, false, true> : rmsnorm_rope_pair_kernel<T, 32, Backward, false, false>;
    }
    if (dense) return swiglu ? rmsnorm_rope_pair_kernel<T, 16, Backward, true, true> : rmsnorm_rope_pair_kernel<T, 16, Backward, true, false>;
    return swiglu ? rmsnorm_rope_pair_kernel<T, 16, Backward, false, true> : rmsnorm_rope_pair_kernel<T, 16, Backward, false, false>;
}

// The pair kernel's form for these rows, and how many workgroups each of the two takes: as many as in a launch of its own, up to
// what the chip holds, since each leaves one partial sum of the weight gradient and their number is the order of its additions.
// More than the chip holds together, k's start as q's end; shared out in the ratio of their rows instead, all resident at once, the
// launches took longer: backward of 32768 tokens, 8:2 heads of 128, 45.6 us and 42.5 so, forward 31.9 and 29.5; 12:4 heads of 64,
// 50.4 and 45.7, 38.9 and 35.0.
template <typename T, bool Backward>
struct PairPlan {
    int lanes;
    bool dense;
    int blocks_q, blocks_k;
    PairPlan(int rows_q, int rows_k, int head_dim, RopeArgs rope) : lanes(pair_lanes<T>(head_dim)), dense(rope_dense<T>(std::max(rows_q, rows_k), head_dim, rope) &&
                                                                                                         rows_q % 4 == 0 && rows_k % 4 == 0) {
        const int cap = resident_blocks(reinterpret_cast<const void*>(pair_kernel<T, Backward>(lanes, dense, false)));
        blocks_q = std::min(pair_blocks(rows_q, lanes), cap);
        blocks_k = std::min(pair_blocks(rows_k, lanes), cap);
    }
};
template <typename T, bool Backward>
int launch_pair(const PairPlan<T, Backward>& plan, const RopeRows<T>& q, const RopeRows<T>& k, int head_dim, float epsilon,
                const RopeArgs& rope, const SwigluTensors* beside, hipStream_t stream) {
    SwigluRows<T> swiglu{};
    int blocks_s = 0;
    if (beside != nullptr) {
        swiglu = {static_cast<T*>(beside->output), static_cast<const T*>(beside->grad_activated), static_cast<const T*>(beside->gate_up),
                  static_cast<unsigned int>(beside->rows), static_cast<unsigned int>(beside->hidden)};
        const std::size_t vectors = beside->rows * (beside->hidden / kVec128<T>);
        blocks_s = static_cast<int>(std::min<std::size_t>((vectors + kThreads - 1) / kThreads, static_cast<std::size_t>(compute_units()) * 16));
        auto kernel = pair_kernel<T, Backward>(plan.lanes, plan.dense, true);
        hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned int>(plan.blocks_q + plan.blocks_k + blocks_s)), dim3(kThreads), 0, stream, q, k,
                           plan.blocks_q, plan.blocks_k, head_dim, 1.0f / static_cast<float>(head_dim), epsilon, rope, swiglu);
        CGPTX_LAUNCH_CHECK();
        return CGPTX_OK;
    }
    auto kernel = pair_kernel<T, Backward>(plan.lanes, plan.dense, false);
    hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned int>(plan.blocks_q + plan.blocks_k)), dim3(kThreads), 0, stream, q, k,
                       plan.blocks_q, plan.blocks_k, head_dim, 1.0f / static_cast<float>(head_dim), epsilon, rope, swiglu);
    CGPTX_LAUNCH_CHECK();
    return CGPTX_OK;
}
}  // namespace

bool swiglu_beside_norms(const SwigluTensors& s, int dtype) {
    constexpr std::size_t limit = std::size_t{1} << 31;
    return s.output != nullptr && s.gate_up != nullptr && is_aligned16(s.output) && is_aligned16(s.grad_activated) && is_aligned16(s.gate_up) &&
           s.rows != 0 && s.rows < limit && s.hidden != 0 && s.hidden < limit && s.hidden % (16 / dtype_size(dtype)) == 0;
}

int rmsnorm_rope_forward(const NormRopeTensors& q, const NormRopeTensors& k, const void* cos_cache, const void* sin_cache,
                         std::size_t tokens, std::size_t head_dim, std::size_t sequence, std::size_t rotary_dim,
                         std::size_t position_offset, float epsilon, int dtype, hipStream_t stream, const SwigluTensors* swiglu) {
    if (swiglu != nullptr && !swiglu_beside_norms(*swiglu, dtype))
        return fail(CGPTX_INVALID_ARGUMENT, "rmsnorm_rope_forward: SwiGLU tensors that the fused pass does not serve");
    for (const NormRopeTensors* t : {&q, &k}) {
        if (int s = validate(t->output, t->input, t->weight, tokens * t->heads, head_dim, epsilon, dtype, "rmsnorm_rope_forward")) return s;
        if (cos_cache == nullptr || sin_cache == nullptr || sequence == 0 ||
            !rmsnorm_rope_fusable(t->output, t->input, nullptr, t->weight, cos_cache, sin_cache, head_dim, rotary_dim, dtype))
            return fail(CGPTX_INVALID_ARGUMENT, "rmsnorm_rope_forward: shape or alignment not served by the fused pass");
    }
    const int h = static_cast<int>(head_dim);
    const RopeArgs rope = make_rope(cos_cache, sin_cache, 0, sequence, rotary_dim, position_offset);
    return dispatch_dtype(dtype, [&]<typename T>() -> int {
        const auto rows = [&](const NormRopeTensors& t) {
            return RopeRows<T>{static_cast<T*>(t.output), nullptr, nullptr, static_cast<const T*>(t.input),
                               static_cast<const T*>(t.weight), static_cast<int>(tokens * t.heads), static_cast<int>(t.heads)};
        };
        const RopeRows<T> of_q = rows(q), of_k = rows(k);
        return launch_pair<T, false>(PairPlan<T, false>(of_q.rows, of_k.rows, h, rope), of_q, of_k, h, epsilon, rope, swiglu, stream);
    });
}

int rmsnorm_rope_backward(const NormRopeTensors& q, const NormRopeTensors& k, const void* cos_cache, const void* sin_cache,
                          std::size_t tokens, std::size_t head_dim, std::size_t sequence, std::size_t rotary_dim,
                          std::size_t position_offset, float epsilon, int dtype, hipStream_t stream, ColumnReduceSink* sink,
                          const SwigluTensors* swiglu) {
    if (swiglu != nullptr && (!swiglu_beside_norms(*swiglu, dtype) || swiglu->grad_activated == nullptr))
        return fail(CGPTX_INVALID_ARGUMENT, "rmsnorm_rope_backward: SwiGLU tensors that the fused pass does not serve");
    for (const NormRopeTensors* t : {&q, &k}) {
        if (int s = validate(t->output, t->grad_output, t->input, tokens * t->heads, head_dim, epsilon, dtype, "rmsnorm_rope_backward"))
            return s;
        if (t->grad_weight == nullptr || t->weight == nullptr || cos_cache == nullptr || sin_cache == nullptr || sequence == 0 ||
            !rmsnorm_rope_fusable(t->output, t->grad_output, t->input, t->weight, cos_cache, sin_cache, head_dim, rotary_dim, dtype))
            return fail(CGPTX_INVALID_ARGUMENT, "rmsnorm_rope_backward: shape or alignment not served by the fused pass");
    }
    const int h = static_cast<int>(head_dim);
    const RopeArgs rope = make_rope(cos_cache, sin_cache, 0, sequence, rotary_dim, position_offset);
    return dispatch_dtype(dtype, [&]<typename T>() -> int {
        const PairPlan<T, true> plan(static_cast<int>(tokens * q.heads), static_cast<int>(tokens * k.heads), h, rope);
        void* mem = nullptr;
        bool deferred = false;
        if (int s = partial_memory(sink, stream, static_cast<std::size_t>(plan.blocks_q + plan.blocks_k) * head_dim * sizeof(float), &mem,
                                   &deferred))
            return s;
        auto* partial_q = static_cast<float*>(mem);
        float* partial_k = partial_q + static_cast<std::size_t>(plan.blocks_q) * head_dim;
        const auto rows = [&](const NormRopeTensors& t, float* partial) {
            return RopeRows<T>{static_cast<T*>(t.output), partial, static_cast<const T*>(t.grad_output), static_cast<const T*>(t.input),
                               static_cast<const T*>(t.weight), static_cast<int>(tokens * t.heads), static_cast<int>(t.heads)};
        };
        if (int s = launch_pair<T, true>(plan, rows(q, partial_q), rows(k, partial_k), h, epsilon, rope, swiglu, stream)) return s;
        if (int s = reduce_columns<T>(sink, deferred, static_cast<T*>(q.grad_weight), partial_q, plan.blocks_q, h, dtype, stream)) return s;
        return reduce_columns<T>(sink, deferred, static_cast<T*>(k.grad_weight), partial_k, plan.blocks_k, h, dtype, stream);
    });
}

bool rmsnorm_dual_fusable(const void* a, const void* b, const void* c, const void* d, const void* e, std::size_t hidden,
                          int dtype) {
    if (!valid_dtype(dtype) || hidden == 0 || hidden > (1u << 20)) return false;
    bool shape_ok = false;
    dispatch_dtype(dtype, [&]<typename T>() -> int {
        shape_ok = pick_fast_shape<T>(static_cast<int>(hidden)).lpr != 0;
        return CGPTX_OK;
    });
    return shape_ok && is_aligned16(a) && is_aligned16(b) && is_aligned16(c) && is_aligned16(d) && is_aligned16(e);
}

namespace {
template <typename T, bool Backward>
int launch_dual(const FastShape shape, T* out_a, T* out_f, float* partial_a, float* partial_f, const T* dy_a, const T* dy_f,
                const T* residual, const T* x, const T* w_a, const T* w_f, int rows, int hidden, float eps, int blocks,
                hipStream_t stream) {
    const float inv_hidden = 1.0f / static_cast<float>(hidden);
#define CGPTX_RMS_CASE(L, KK)                                                                                         \
    if (shape.lpr == L && shape.k == KK) {                                                                            \
        hipLaunchKernelGGL((rmsnorm_dual_rows_kernel<T, L, KK, Backward>), dim3(blocks), dim3(kThreads), 0, stream,   \
                           out_a, out_f, partial_a, partial_f, dy_a, dy_f, residual, x, w_a, w_f, rows, hidden,      \
                           inv_hidden, eps);                                                                          \
        return CGPTX_OK;                                                                                              \
    }
    CGPTX_RMS_CASE(16, 1)
    CGPTX_RMS_CASE(32, 1)
    CGPTX_RMS_CASE(64, 1)
    CGPTX_RMS_CASE(64, 2)
    CGPTX_RMS_CASE(64, 4)
#undef CGPTX_RMS_CASE
    return fail(CGPTX_RUNTIME, "rmsnorm: no kernel for shape");
}
}  // namespace

namespace {
template <typename T, bool Backward>
const void* dual_kernel(const FastShape shape) {
#define CGPTX_RMS_CASE(L, KK) \
    if (shape.lpr == L && shape.k == KK) return reinterpret_cast<const void*>(&rmsnorm_dual_rows_kernel<T, L, KK, Backward>);
    CGPTX_RMS_CASE(16, 1)
    CGPTX_RMS_CASE(32, 1)
    CGPTX_RMS_CASE(64, 1)
    CGPTX_RMS_CASE(64, 2)
    CGPTX_RMS_CASE(64, 4)
#undef CGPTX_RMS_CASE
    return nullptr;
}
}  // namespace

int rmsnorm_forward_dual(void* output_a, void* output_f, const void* input, const void* weight_a, const void* weight_f,
                         std::size_t rows, std::size_t hidden, float epsilon, int dtype, hipStream_t stream) {
    if (int s = validate(output_a, output_f, input, rows, hidden, epsilon, dtype, "rmsnorm_forward_dual")) return s;
    if (weight_a == nullptr || weight_f == nullptr ||
        !rmsnorm_dual_fusable(output_a, output_f, input, weight_a, weight_f, hidden, dtype))
        return fail(CGPTX_INVALID_ARGUMENT, "rmsnorm_forward_dual: shape or alignment not served by the fused pass");
    const int r = static_cast<int>(rows), h = static_cast<int>(hidden);
    return dispatch_dtype(dtype, [&]<typename T>() -> int {
        const FastShape shape = pick_fast_shape<T>(h);
        if (int s = launch_dual<T, false>(shape, static_cast<T*>(output_a), static_cast<T*>(output_f), nullptr, nullptr, nullptr,
                                          nullptr, nullptr, static_cast<const T*>(input), static_cast<const T*>(weight_a),
                                          static_cast<const T*>(weight_f), r, h, epsilon,
                                          fast_blocks(shape, r, dual_kernel<T, false>(shape)), stream))
            return s;
        CGPTX_LAUNCH_CHECK();
        return CGPTX_OK;
    });
}

int rmsnorm_backward_dual(void* grad_input, void* grad_weight_a, void* grad_weight_f, const void* grad_output_a,
                          const void* grad_output_f, const void* input, const void* weight_a, const void* weight_f,
                          const void* residual, std::size_t rows, std::size_t hidden, float epsilon, int dtype,
                          hipStream_t stream, ColumnReduceSink* sink) {
    if (int s = validate(grad_input, grad_output_a, input, rows, hidden, epsilon, dtype, "rmsnorm_backward_dual")) return s;
    if (grad_weight_a == nullptr || grad_weight_f == nullptr || weight_a == nullptr || weight_f == nullptr ||
        grad_output_f == nullptr ||
        !rmsnorm_dual_fusable(grad_input, grad_output_a, grad_output_f, input, residual, hidden, dtype) ||
        !is_aligned16(weight_a) || !is_aligned16(weight_f))
        return fail(CGPTX_INVALID_ARGUMENT, "rmsnorm_backward_dual: shape or alignment not served by the fused pass");
    const int r = static_cast<int>(rows), h = static_cast<int>(hidden);
    return dispatch_dtype(dtype, [&]<typename T>() -> int {
        const FastShape shape = pick_fast_shape<T>(h);
        const int blocks = fast_blocks(shape, r, dual_kernel<T, true>(shape));
        void* mem = nullptr;
        bool deferred = false;
        const std::size_t partial_bytes = static_cast<std::size_t>(blocks) * hidden * sizeof(float);
        if (int s = partial_memory(sink, stream, 2 * partial_bytes, &mem, &deferred)) return s;
        auto* partial_a = static_cast<float*>(mem);
        auto* partial_f = reinterpret_cast<float*>(static_cast<char*>(mem) + partial_bytes);
        if (int s = launch_dual<T, true>(shape, static_cast<T*>(grad_input), nullptr, partial_a, partial_f,
                                         static_cast<const T*>(grad_output_a), static_cast<const T*>(grad_output_f),
                                         static_cast<const T*>(residual), static_cast<const T*>(input),
                                         static_cast<const T*>(weight_a), static_cast<const T*>(weight_f), r, h, epsilon, blocks,
                                         stream))
            return s;
        CGPTX_LAUNCH_CHECK();
        if (int s = reduce_columns<T>(sink, deferred, static_cast<T*>(grad_weight_a), partial_a, blocks, h, dtype, stream))
            return s;
        return reduce_columns<T>(sink, deferred, static_cast<T*>(grad_weight_f), partial_f, blocks, h, dtype, stream);
    });
}

namespace {
// Where rmsnorm_backward's partial sums go: the per-stream arena (fixed == nullptr), or a caller-provided block
// of `fixed_bytes` that is never exceeded (a larger need is an error, nothing is allocated).
struct Workspace {
    hipStream_t stream;
    void* fixed;
    std::size_t fixed_bytes;
    ColumnReduceSink* sink = nullptr;  // when given and roomy enough, the weight-gradient reduction is recorded there
    int get(std::size_t bytes, void** out) const {
        if (fixed == nullptr) return scratch(stream, bytes, out);
        if (bytes > fixed_bytes)
            return fail(CGPTX_INVALID_ARGUMENT, "rmsnorm_backward_static: the shape needs " + std::to_string(bytes) +
                                                    " bytes of working memory, the built-in block holds " +
                                                    std::to_string(fixed_bytes));
        *out = fixed;
        return CGPTX_OK;
    }
};

int rmsnorm_backward_impl(void* grad_input, void* grad_weight, const void* grad_output, const void* input,
                          const void* weight, const void* residual, std::size_t rows, std::size_t hidden,
                          float epsilon, int dtype, hipStream_t stream, const Workspace& workspace) {
    if (int s = validate(grad_input, grad_output, input, rows, hidden, epsilon, dtype, "rmsnorm_backward")) return s;
    if (grad_weight == nullptr || weight == nullptr)
        return fail(CGPTX_INVALID_ARGUMENT, "rmsnorm_backward: null weight tensor");
    const int r = static_cast<int>(rows), h = static_cast<int>(hidden);
    return dispatch_dtype(dtype, [&]<typename T>() -> int {
        auto* dx = static_cast<T*>(grad_input);
        auto* res = static_cast<const T*>(residual);
        auto* dw = static_cast<T*>(grad_weight);
        auto* dy = static_cast<const T*>(grad_output);
        auto* x = static_cast<const T*>(input);
        auto* w = static_cast<const T*>(weight);
        const FastShape shape = pick_fast_shape<T>(h);
        const bool aligned = is_aligned16(dx) && is_aligned16(dy) && is_aligned16(x) && is_aligned16(w) && is_aligned16(res);
        const int reduce_blocks = (h + kWave - 1) / kWave;
        if (shape.lpr != 0 && aligned) {
            const int blocks = fast_blocks(shape, r, fast_kernel<T, true>(shape));
            void* mem = nullptr;
            const std::size_t bytes = static_cast<std::size_t>(blocks) * hidden * sizeof(float);
            if (workspace.sink != nullptr) mem = workspace.sink->take(bytes);
            const bool deferred = mem != nullptr;
            if (!deferred) {
                if (int s = workspace.get(bytes, &mem)) return s;
            }
            auto* partial = static_cast<float*>(mem);
            if (int s = launch_fast<T, true>(shape, dx, partial, dy, res, x, w, r, h, epsilon, blocks, stream)) return s;
            CGPTX_LAUNCH_CHECK();
            return reduce_columns<T>(workspace.sink, deferred, dw, partial, blocks, h, dtype, stream);
        }
        const int slices = r < 256 ? 1 : (r < 65536 ? 64 : 256);
        const int rows_per_slice = (r + slices - 1) / slices;
        void* mem = nullptr;
        const std::size_t inv_bytes = (rows * sizeof(float) + 255) & ~std::size_t{255};
        if (int s = workspace.get(inv_bytes + static_cast<std::size_t>(slices) * hidden * sizeof(float), &mem))
            return s;
        auto* inv_rms = static_cast<float*>(mem);
        auto* partial = reinterpret_cast<float*>(static_cast<char*>(mem) + inv_bytes);
        const int row_blocks = r < compute_units() * 8 ? r : compute_units() * 8;
        hipLaunchKernelGGL((rmsnorm_row_generic_kernel<T, true>), dim3(row_blocks), dim3(kThreads), 0, stream, dx,
                           inv_rms, dy, res, x, w, r, h, 1.0f / static_cast<float>(h), epsilon);
        CGPTX_LAUNCH_CHECK();
        hipLaunchKernelGGL((rmsnorm_dgamma_generic_kernel<T>), dim3(reduce_blocks, slices), dim3(kThreads), 0, stream,
                           partial, dy, x, inv_rms, r, h, rows_per_slice);
        CGPTX_LAUNCH_CHECK();
        launch_column_partial_reduce<T>(dw, partial, slices, h, 0, stream);
        CGPTX_LAUNCH_CHECK();
        return CGPTX_OK;
    });
}
}  // namespace

// What one backward pass takes from a ColumnReduceSink (0 when the shape runs on kernels that do not defer their
// reduction). The same arithmetic as in the passes below; a caller sizes its sink with it before the first pass.
std::size_t rmsnorm_backward_sink_bytes(NormPass pass, std::size_t rows, std::size_t hidden, int dtype) {
    if (!valid_dtype(dtype) || rows == 0 || hidden == 0 || rows > (1u << 30) || hidden > (1u << 20)) return 0;
    const int r = static_cast<int>(rows), h = static_cast<int>(hidden);
    std::size_t bytes = 0;
    dispatch_dtype(dtype, [&]<typename T>() -> int {
        const FastShape shape = pick_fast_shape<T>(h);
        if (shape.lpr == 0) return CGPTX_OK;
        int blocks = 0;
        if (pass == NormPass::with_rope) {
            // The pass picks between two kernels by properties of its rotary tables that are not known here: room
            // for whichever of them takes more. q's and k's last workgroups may both be partly filled.
            const int lanes = pair_lanes<T>(h);
            if (lanes == 0) return CGPTX_OK;
            for (const bool dense : {false, true})
                blocks = std::max(blocks, std::min(pair_blocks(r, lanes) + 1,
                                                   2 * resident_blocks(reinterpret_cast<const void*>(pair_kernel<T, true>(lanes, dense, false)))));
        } else {
            const void* kernel = pass == NormPass::dual ? dual_kernel<T, true>(shape) : fast_kernel<T, true>(shape);
            if (kernel == nullptr) return CGPTX_OK;
            blocks = fast_blocks(shape, r, kernel);
        }
        const std::size_t partial_bytes = static_cast<std::size_t>(blocks) * hidden * sizeof(float);
        bytes = pass == NormPass::dual ? 2 * partial_bytes : partial_bytes;
        bytes = (bytes + 255) & ~std::size_t{255};  // ColumnReduceSink::take hands out multiples of 256
        return CGPTX_OK;
    });
    return bytes;
}

int rmsnorm_backward_residual(void* grad_input, void* grad_weight, const void* grad_output, const void* input,
                              const void* weight, const void* residual, std::size_t rows, std::size_t hidden,
                              float epsilon, int dtype, hipStream_t stream, ColumnReduceSink* sink) {
    return rmsnorm_backward_impl(grad_input, grad_weight, grad_output, input, weight, residual, rows, hidden, epsilon, dtype,
                                 stream, Workspace{stream, nullptr, 0, sink});
}

}  // namespace cgptx

// ---- rmsnorm_backward without any allocation ------------------------------------------------------------------
// The partial sums of the weight gradient live in a block that is part of the library's device image: every
// GPU the library runs on holds its own copy, at its own address, until the process ends. Host code reaches it
// only through the address hipGetSymbolAddress returns for the current device (the array's name is a host-side
// stand-in, not a device address), looked up once per device and kept.
namespace {
constexpr std::size_t kStaticScratchBytes = std::size_t{16} << 20;
static __device__ __align__(256) unsigned char g_static_scratch[kStaticScratchBytes];

constexpr int kMaxDevices = 64;
std::mutex g_static_scratch_mutex;
void* g_static_scratch_address[kMaxDevices] = {};  // per device; null until first use on that device

int static_scratch_address(void** out) {
    int device = 0;
    CGPTX_HIP(hipGetDevice(&device));
    if (device < 0 || device >= kMaxDevices) return cgptx::fail(CGPTX_RUNTIME, "rmsnorm_backward_static: device index out of range");
    std::lock_guard<std::mutex> lock(g_static_scratch_mutex);
    if (g_static_scratch_address[device] == nullptr) {
        void* address = nullptr;
        CGPTX_HIP(hipGetSymbolAddress(&address, HIP_SYMBOL(g_static_scratch)));
        if (address == nullptr) return cgptx::fail(CGPTX_RUNTIME, "rmsnorm_backward_static: no device address for the working block");
        g_static_scratch_address[device] = address;
    }
    *out = g_static_scratch_address[device];
    return CGPTX_OK;
}
}  // namespace

extern "C" int cgptx_rmsnorm_backward_static(void* grad_input, void* grad_weight, const void* grad_output, const void* input,
                                             const void* weight, size_t rows, size_t hidden, float epsilon, int dtype,
                                             cgptx_stream stream_) {
    void* block = nullptr;
    if (int s = static_scratch_address(&block)) return s;
    auto stream = static_cast<hipStream_t>(stream_);
    // Nothing in the block has to start at zero: the row kernel writes every partial-sum row it is launched
    // with before the reduction kernels, later on the same stream, read them.
    return cgptx::rmsnorm_backward_impl(grad_input, grad_weight, grad_output, input, weight, nullptr, rows, hidden, epsilon,
                                        dtype, stream, cgptx::Workspace{stream, block, kStaticScratchBytes});
}

extern "C" int cgptx_rmsnorm_backward(void* grad_input, void* grad_weight, const void* grad_output, const void* input,
                                      const void* weight, size_t rows, size_t hidden, float epsilon, int dtype,
                                      cgptx_stream stream) {
    return cgptx::rmsnorm_backward_residual(grad_input, grad_weight, grad_output, input, weight, nullptr, rows, hidden,
                                            epsilon, dtype, static_cast<hipStream_t>(stream));
}

extern "C" int cgptx_rmsnorm_forward(void* output, const void* input, const void* weight, size_t rows, size_t hidden,
                                     float epsilon, int dtype, cgptx_stream stream_) {
    using namespace cgptx;
    if (int s = validate(output, input, weight, rows, hidden, epsilon, dtype, "rmsnorm_forward")) return s;
    auto stream = static_cast<hipStream_t>(stream_);
    const int r = static_cast<int>(rows), h = static_cast<int>(hidden);
    return dispatch_dtype(dtype, [&]<typename T>() -> int {
        auto* y = static_cast<T*>(output);
        auto* x = static_cast<const T*>(input);
        auto* w = static_cast<const T*>(weight);
        const FastShape shape = pick_fast_shape<T>(h);
        if (shape.lpr != 0 && is_aligned16(y) && is_aligned16(x) && is_aligned16(w)) {
            const int blocks = fast_blocks(shape, r, fast_kernel<T, false>(shape));
            if (int s = launch_fast<T, false>(shape, y, nullptr, nullptr, nullptr, x, w, r, h, epsilon, blocks, stream)) return s;
            CGPTX_LAUNCH_CHECK();
            return CGPTX_OK;
        }
        const int row_blocks = r < compute_units() * 8 ? r : compute_units() * 8;
        hipLaunchKernelGGL((rmsnorm_row_generic_kernel<T, false>), dim3(row_blocks), dim3(kThreads), 0, stream, y,
                           nullptr, nullptr, nullptr, x, w, r, h, 1.0f / static_cast<float>(h), epsilon);
        CGPTX_LAUNCH_CHECK();
        return CGPTX_OK;
    });
}
