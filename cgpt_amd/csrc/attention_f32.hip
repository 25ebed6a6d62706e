// Causal grouped-query attention, fp32 storage and arithmetic, forward and backward, on v_mfma_f32_16x16x4_f32.
//
// Formulas as in attention.hip. The scheme is the same, too: the score tile is produced so that the stationary index is
// the lane (l % 16) and the streamed index lives in the accumulator's four registers (4 (l / 16) + r), and with a k step
// of 4 those registers are, without any conversion, the k-operand of the second product: step r contracts over the
// streamed rows 4 g + r of the four lane groups g. Its other operand is read along the head dimension, 16 bytes per lane
// of row 4 g + r; the four elements belong to four different accumulator blocks, which only permutes the head dimension
// over the blocks. Nothing passes through LDS.
//
// What bounds it: fp32 is for checks on short sequences, where a serial walk over the streamed rows by one wavefront per
// output row (the scalar family of attention.hip) was latency, and the matrix rate is a sixteenth of the 16-bit one. So
// one workgroup of eight wavefronts owns 16 stationary rows only, and the wavefronts split the streamed tiles between
// them (tile t to wavefront t mod 8); their partial results meet in LDS at the end, in wavefront order: no atomics,
// results independent of scheduling. Few key tiles are shared by several workgroups in the dK/dV pass (the caller decides
// and adds their sums up). A query touches no key that the causal mask hides from it, as in a walk over single rows: see
// non_finite(). One sequence of 256 tokens, 8:2 heads of 128, causal: forward 151 -> 14 us, dQ
// 239 -> 21, dK/dV 295 -> 20.
#include "attention_f32.hpp"

#include <cmath>

namespace cgptx {
namespace {

constexpr int kWaves = 8;
constexpr int kThreads = kWaves * kWave;
constexpr int kTile = 16;  // stationary rows of a workgroup, streamed rows of a step

using acc_t = vec_t<float, 4>;
using f32x4 = vec_t<float, 4>;

__device__ __forceinline__ acc_t mfma(float a, float b, acc_t c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

// A row of a tensor as an operand that is contracted over the head dimension: lane l holds row l % 16's elements
// 16 c + 4 (l / 16) .. + 3 of chunk c. Rows that do not exist and elements past the head dimension are zeros.
template <int D>
struct RowOperand {
    f32x4 chunk[D / 16];
    __device__ __forceinline__ void load(const float* row, bool live, int d) {
        const int at = ((threadIdx.x & (kWave - 1)) >> 4) * 4;
#pragma unroll
        for (int c = 0; c < D / 16; ++c) chunk[c] = live && 16 * c + at < d ? load_vec<float, 4>(row + 16 * c + at) : f32x4(0.0f);
    }
};
template <int D>
__device__ __forceinline__ acc_t product(const RowOperand<D>& a, const RowOperand<D>& b) {
    acc_t sum[2] = {acc_t(0.0f), acc_t(0.0f)};  // two chains: consecutive MFMAs do not wait for each other
#pragma unroll
    for (int c = 0; c < D / 16; ++c)
#pragma unroll
        for (int e = 0; e < 4; ++e) sum[e & 1] = mfma(a.chunk[c][e], b.chunk[c][e], sum[e & 1]);
    return sum[0] + sum[1];
}

// Rows of a tile as the operand of a product over the rows: lane l holds, for each r, elements 64 b + 4 (l % 16) .. + 3 of
// row 4 (l / 16) + r.
template <int D>
struct ColumnOperand {
    f32x4 part[4][D / 64];
    // row0: first row of the tile; rows from `limit` on are zeros.
    __device__ __forceinline__ void load(const float* base, long row_stride, int row0, int limit, int d) {
        const int lane = threadIdx.x & (kWave - 1), at = (lane & 15) * 4;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int row = row0 + 4 * (lane >> 4) + r;
#pragma unroll
            for (int b = 0; b < D / 64; ++b)
                part[r][b] = row < limit && 64 * b + at < d ? load_vec<float, 4>(base + row * row_stride + 64 * b + at) : f32x4(0.0f);
        }
    }
};
// result[b][e] += rows^T x values: block (b, e) holds the head dimension's elements 64 b + 4 m + e, m = 0 .. 15.
template <int D>
__device__ __forceinline__ void accumulate(acc_t (&result)[D / 64][4], const ColumnOperand<D>& rows, const acc_t& values) {
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int b = 0; b < D / 64; ++b)
#pragma unroll
            for (int e = 0; e < 4; ++e) result[b][e] = mfma(rows.part[r][b][e], values[r], result[b][e]);
}

// Whether the tile holds an Inf or a NaN (the same answer in all lanes): 0 x is 0 for every other x. A tile on the causal
// diagonal has rows that some stationary rows do not see. Their values are 0, but the matrix instruction multiplies them
// all the same, and 0 x Inf is NaN. Such a tile with such a row is left out of the walk and added row by row behind it, in
// a pass of its own so that the walk's registers do not pay for it.
template <int D>
__device__ __forceinline__ bool non_finite(const ColumnOperand<D>& rows) {
    float sum = 0.0f;
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int b = 0; b < D / 64; ++b)
#pragma unroll
            for (int e = 0; e < 4; ++e) sum = fmaf(rows.part[r][b][e], 0.0f, sum);
    return __ballot(!(sum == 0.0f)) != 0;
}
// accumulate() over the rows row0 + i, below `limit`, that this lane's stationary row sees (visible(i)); no other row is
// multiplied.
template <int D, typename Visible>
__device__ __forceinline__ void accumulate_visible(acc_t (&result)[D / 64][4], const float* base, long row_stride, int row0, int limit,
                                                   int d, const acc_t& values, Visible&& visible) {
    const int lane = threadIdx.x & (kWave - 1), at = (lane >> 4) * 16;  // the head dimension's elements of a lane: see deposit()
#pragma unroll 1
    for (int i = 0; i < kTile; ++i) {
        const int r = i & 3;
        const float value = __shfl(r == 0 ? values[0] : r == 1 ? values[1] : r == 2 ? values[2] : values[3], (lane & 15) + 16 * (i >> 2), kWave);
        if (row0 + i >= limit || !visible(i)) continue;
#pragma unroll
        for (int b = 0; b < D / 64; ++b)
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                if (64 * b + at + 4 * c >= d) continue;
                const f32x4 row = load_vec<float, 4>(base + (row0 + i) * row_stride + 64 * b + at + 4 * c);
#pragma unroll
                for (int e = 0; e < 4; ++e) result[b][e][c] = fmaf(row[e], value, result[b][e][c]);
            }
    }
}

// Sums over the four lane groups of a stationary row.
__device__ __forceinline__ float row_sum(float v) {
    v += __shfl_xor(v, 16, kWave);
    return v + __shfl_xor(v, 32, kWave);
}

// The wavefronts' partial results [kWaves][16 rows][D] in LDS; rows are padded by one 16-byte chunk.
template <int D>
constexpr int kPitch = D + 4;
template <int D>
constexpr int kSmemBytes = kWaves * kTile * kPitch<D> * 4;
template <int D>
__device__ __forceinline__ void deposit(float* lds, int wave, const acc_t (&result)[D / 64][4], float factor) {
    const int lane = threadIdx.x & (kWave - 1);
    float* row = lds + (wave * kTile + (lane & 15)) * kPitch<D> + (lane >> 4) * 16;
#pragma unroll
    for (int b = 0; b < D / 64; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r)
            *reinterpret_cast<f32x4*>(row + 64 * b + 4 * r) =
                f32x4{result[b][0][r], result[b][1][r], result[b][2][r], result[b][3][r]} * factor;
}
// Adds the partial results up and hands thread t four consecutive elements: store(row, first element, sum).
template <int D, typename Store>
__device__ __forceinline__ void collect(const float* lds, int d, Store&& store) {
    const int row = threadIdx.x / (D / 4), at = (threadIdx.x % (D / 4)) * 4;
    if (row >= kTile || at >= d) return;
    f32x4 sum = *reinterpret_cast<const f32x4*>(lds + row * kPitch<D> + at);
#pragma unroll
    for (int w = 1; w < kWaves; ++w) sum += *reinterpret_cast<const f32x4*>(lds + (w * kTile + row) * kPitch<D> + at);
    store(row, at, sum);
}

template <int D>
__global__ __launch_bounds__(kThreads) void attention_f32_forward_kernel(AttentionF32Args p) {
    extern __shared__ __align__(16) float lds[];
    __shared__ float wave_max[kWaves][kTile], wave_total[kWaves][kTile];
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave, g = lane >> 4;
    const int q0 = (gridDim.x - 1 - blockIdx.x) * kTile, h = blockIdx.y, b = blockIdx.z, kvh = h / (p.hq / p.hkv);  // longest first
    const int query = q0 + (lane & 15);
    const long q_stride = static_cast<long>(p.hq) * p.d, kv_stride = static_cast<long>(p.hkv) * p.d;
    const float* k_base = p.k + static_cast<long>(b) * p.ks * kv_stride + static_cast<long>(kvh) * p.d;
    const float* v_base = p.v + static_cast<long>(b) * p.ks * kv_stride + static_cast<long>(kvh) * p.d;
    RowOperand<D> q;
    q.load(p.q + (static_cast<long>(b) * p.qs + query) * q_stride + static_cast<long>(h) * p.d, query < p.qs, p.d);
    const int last_key = p.causal ? min(p.ks - 1, p.offset + min(q0 + kTile, p.qs) - 1) : p.ks - 1;
    const int tiles = last_key / kTile + 1;
    const int my_last = p.causal ? min(p.ks - 1, p.offset + query) : p.ks - 1;

    float m = -INFINITY, total = 0.0f;
    acc_t o[D / 64][4];
#pragma unroll
    for (int c = 0; c < D / 64; ++c)
#pragma unroll
        for (int e = 0; e < 4; ++e) o[c][e] = acc_t(0.0f);
    auto key_rows = [&](RowOperand<D>& k, int t) {
        const int key = t * kTile + (lane & 15);
        k.load(k_base + key * kv_stride, key < p.ks && t < tiles, p.d);
    };
    const int first_masked = p.causal ? (p.offset + q0 + 1) / kTile : tiles;  // tile with a key that a query of the block does not see
    bool left_out = false;
    RowOperand<D> k, ahead;
    key_rows(k, wave);
    for (int t = wave; t < tiles; t += kWaves) {
        ColumnOperand<D> v;
        v.load(v_base, kv_stride, t * kTile, p.ks, p.d);
        key_rows(ahead, t + kWaves);
        acc_t s = product<D>(k, q);  // lane: query l % 16, keys 4 g + r
        float peak = -INFINITY;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            s[r] = t * kTile + 4 * g + r <= my_last ? s[r] * p.scale : -INFINITY;
            peak = fmaxf(peak, s[r]);
        }
        peak = fmaxf(peak, __shfl_xor(peak, 16, kWave));
        peak = fmaxf(peak, __shfl_xor(peak, 32, kWave));
        const float next = fmaxf(m, peak);
        const float base = next == -INFINITY ? 0.0f : next;  // no key visible so far: all terms below are 0
        const float alpha = expf(m - base);
        float sum = 0.0f;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            s[r] = expf(s[r] - base);
            sum += s[r];
        }
        total = total * alpha + row_sum(sum);
        m = next;
#pragma unroll
        for (int c = 0; c < D / 64; ++c)
#pragma unroll
            for (int e = 0; e < 4; ++e) o[c][e] *= alpha;
        if (t >= first_masked && non_finite<D>(v)) left_out = true;
        else accumulate<D>(o, v, s);
        k = ahead;
    }
    if (left_out) {
        for (int t = wave; t < tiles; t += kWaves) {
            ColumnOperand<D> v;
            v.load(v_base, kv_stride, t * kTile, p.ks, p.d);
            if (t < first_masked || !non_finite<D>(v)) continue;
            key_rows(k, t);
            acc_t s = product<D>(k, q);
#pragma unroll
            for (int r = 0; r < 4; ++r) s[r] = expf(s[r] * p.scale - (m == -INFINITY ? 0.0f : m));
            accumulate_visible<D>(o, v_base, kv_stride, t * kTile, p.ks, p.d, s, [&](int i) { return t * kTile + i <= my_last; });
        }
    }
    // Common maximum over the wavefronts, then the weighted sums.
    if (lane < kTile) {
        wave_max[wave][lane] = m;
        wave_total[wave][lane] = total;
    }
    __syncthreads();
    float peak = wave_max[0][lane & 15];
#pragma unroll
    for (int w = 1; w < kWaves; ++w) peak = fmaxf(peak, wave_max[w][lane & 15]);
    const float base = peak == -INFINITY ? 0.0f : peak;
    deposit<D>(lds, wave, o, expf(m - base));
    __syncthreads();
    auto denominator = [&](int row, float& top) {
        top = wave_max[0][row];
        for (int w = 1; w < kWaves; ++w) top = fmaxf(top, wave_max[w][row]);
        if (top == -INFINITY) return NAN;  // every query sees a key, so all its scores are -Inf or NaN
        float sum = 0.0f;
        for (int w = 0; w < kWaves; ++w) sum += wave_total[w][row] * expf(wave_max[w][row] - top);
        return sum;
    };
    collect<D>(lds, p.d, [&](int row, int at, const f32x4& sum) {
        if (q0 + row >= p.qs) return;
        float top;
        const float l = denominator(row, top);
        store_vec<float, 4>(p.out + (static_cast<long>(b) * p.qs + q0 + row) * q_stride + static_cast<long>(h) * p.d + at,
                            sum * (1.0f / l));  // l is NaN or, with the maximum's own term, at least 1
        if (at == 0 && p.lse_out != nullptr) p.lse_out[(static_cast<long>(b) * p.qs + q0 + row) * p.hq + h] = top + logf(l);
    });
}

template <int D>
__global__ __launch_bounds__(kThreads) void attention_f32_dq_kernel(AttentionF32Args p) {
    extern __shared__ __align__(16) float lds[];
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave, g = lane >> 4;
    const int q0 = (gridDim.x - 1 - blockIdx.x) * kTile, h = blockIdx.y, b = blockIdx.z, kvh = h / (p.hq / p.hkv);
    const int query = q0 + (lane & 15);
    const bool live = query < p.qs;
    const long q_stride = static_cast<long>(p.hq) * p.d, kv_stride = static_cast<long>(p.hkv) * p.d;
    const float* k_base = p.k + static_cast<long>(b) * p.ks * kv_stride + static_cast<long>(kvh) * p.d;
    const float* v_base = p.v + static_cast<long>(b) * p.ks * kv_stride + static_cast<long>(kvh) * p.d;
    const long q_row = (static_cast<long>(b) * p.qs + query) * q_stride + static_cast<long>(h) * p.d;
    const long stat = (static_cast<long>(b) * p.qs + query) * p.hq + h;
    RowOperand<D> q, dout;
    q.load(p.q + q_row, live, p.d);
    dout.load(p.dout + q_row, live, p.d);
    float delta = 0.0f;  // rowsum(dO o O)
    {
        RowOperand<D> o;
        o.load(p.o + q_row, live, p.d);
#pragma unroll
        for (int c = 0; c < D / 16; ++c)
#pragma unroll
            for (int e = 0; e < 4; ++e) delta = fmaf(dout.chunk[c][e], o.chunk[c][e], delta);
        delta = row_sum(delta);
    }
    if (wave == 0 && lane < kTile && live) p.delta[stat] = delta;
    const float lse = live ? p.lse[stat] : 0.0f;
    const int last_key = p.causal ? min(p.ks - 1, p.offset + min(q0 + kTile, p.qs) - 1) : p.ks - 1;
    const int my_last = p.causal ? min(p.ks - 1, p.offset + query) : p.ks - 1;

    acc_t dq[D / 64][4];
#pragma unroll
    for (int c = 0; c < D / 64; ++c)
#pragma unroll
        for (int e = 0; e < 4; ++e) dq[c][e] = acc_t(0.0f);
    const int first_masked = p.causal ? (p.offset + q0 + 1) / kTile : last_key / kTile + 1;
    bool left_out = false;
    auto score_gradient = [&](int t) {  // lane: query l % 16, keys 4 g + r
        const int key = t * kTile + (lane & 15);
        RowOperand<D> k, v;
        k.load(k_base + key * kv_stride, key < p.ks, p.d);
        v.load(v_base + key * kv_stride, key < p.ks, p.d);
        const acc_t s = product<D>(k, q), dp = product<D>(v, dout);
        acc_t ds;
#pragma unroll
        for (int r = 0; r < 4; ++r) ds[r] = t * kTile + 4 * g + r <= my_last ? expf(s[r] * p.scale - lse) * (dp[r] - delta) : 0.0f;
        return ds;
    };
    for (int t = wave; t <= last_key / kTile; t += kWaves) {
        ColumnOperand<D> columns;
        columns.load(k_base, kv_stride, t * kTile, p.ks, p.d);
        const acc_t ds = score_gradient(t);
        if (t >= first_masked && non_finite<D>(columns)) left_out = true;
        else accumulate<D>(dq, columns, ds);
    }
    if (left_out) {
        for (int t = wave; t <= last_key / kTile; t += kWaves) {
            ColumnOperand<D> columns;
            columns.load(k_base, kv_stride, t * kTile, p.ks, p.d);
            if (t < first_masked || !non_finite<D>(columns)) continue;
            accumulate_visible<D>(dq, k_base, kv_stride, t * kTile, p.ks, p.d, score_gradient(t),
                                  [&](int i) { return t * kTile + i <= my_last; });
        }
    }
    deposit<D>(lds, wave, dq, p.scale);
    __syncthreads();
    collect<D>(lds, p.d, [&](int row, int at, f32x4 sum) {
        if (q0 + row >= p.qs) return;
        float* to = p.dq + (static_cast<long>(b) * p.qs + q0 + row) * q_stride + static_cast<long>(h) * p.d + at;
        if (p.accumulate) sum += load_vec<float, 4>(to);
        store_vec<float, 4>(to, sum);
    });
}

// Four wavefronts per SIMD, two workgroups per CU, with heads of 64: the compiler's own choice is four registers over that.
template <int D>
__global__ __launch_bounds__(kThreads, D == 64 ? 4 : 2) void attention_f32_dkv_kernel(AttentionF32Args p) {
    extern __shared__ __align__(16) float lds[];
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave, g = lane >> 4;
    const int part = blockIdx.x % p.parts, k0 = blockIdx.x / p.parts * kTile;  // the first keys have most queries
    const int kvh = blockIdx.y, b = blockIdx.z, group = p.hq / p.hkv;
    const int key = k0 + (lane & 15);
    const long q_stride = static_cast<long>(p.hq) * p.d, kv_stride = static_cast<long>(p.hkv) * p.d;
    const long kv_row = (static_cast<long>(b) * p.ks + key) * kv_stride + static_cast<long>(kvh) * p.d;
    RowOperand<D> k, v;
    k.load(p.k + kv_row, key < p.ks, p.d);
    v.load(p.v + kv_row, key < p.ks, p.d);
    const int first_query = p.causal ? max(0, key - p.offset) : 0;  // that sees this lane's key
    const int first_tile = p.causal ? max(0, k0 - p.offset) / kTile : 0;
    const int tiles = max(0, (p.qs + kTile - 1) / kTile - first_tile);

    acc_t dk[D / 64][4], dv[D / 64][4];
#pragma unroll
    for (int c = 0; c < D / 64; ++c)
#pragma unroll
        for (int e = 0; e < 4; ++e) dk[c][e] = dv[c][e] = acc_t(0.0f);
    const int begin = part * (tiles * group) / p.parts + wave, end = (part + 1) * (tiles * group) / p.parts;
    bool left_out = false;
    // Item i is (head of the group, query tile): step(its head's Q and dO, first query, probabilities and score gradients of
    // queries 4 g + r).
    auto walk = [&](auto&& step) __attribute__((always_inline)) {
        for (int i = begin; i < end; i += kWaves) {
            const int head = i / tiles, row0 = (first_tile + i - head * tiles) * kTile, h = kvh * group + head;
            const float* q_base = p.q + static_cast<long>(b) * p.qs * q_stride + static_cast<long>(h) * p.d;
            const float* do_base = p.dout + static_cast<long>(b) * p.qs * q_stride + static_cast<long>(h) * p.d;
            const int query = row0 + (lane & 15);
            acc_t s, dp;
            {
                RowOperand<D> q, dout;
                q.load(q_base + query * q_stride, query < p.qs, p.d);
                dout.load(do_base + query * q_stride, query < p.qs, p.d);
                s = product<D>(q, k);  // lane: key l % 16, queries 4 g + r
                dp = product<D>(dout, v);
            }
            acc_t prob, ds;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int row = row0 + 4 * g + r;
                const bool seen = row >= first_query && row < p.qs && key < p.ks;
                const long stat = (static_cast<long>(b) * p.qs + min(row, p.qs - 1)) * p.hq + h;
                prob[r] = seen ? expf(s[r] * p.scale - p.lse[stat]) : 0.0f;
                ds[r] = seen ? prob[r] * (dp[r] - p.delta[stat]) : 0.0f;
            }
            step(q_base, do_base, row0, prob, ds);
        }
    };
    auto masked = [&](int row0) { return p.causal && row0 < k0 + kTile - 1 - p.offset; };  // a query that does not see a key of the block
    walk([&](const float* q_base, const float* do_base, int row0, const acc_t& prob, const acc_t& ds) __attribute__((always_inline)) {
        ColumnOperand<D> columns;
        columns.load(do_base, q_stride, row0, p.qs, p.d);
        if (masked(row0) && non_finite<D>(columns)) left_out = true;
        else accumulate<D>(dv, columns, prob);
        columns.load(q_base, q_stride, row0, p.qs, p.d);
        if (masked(row0) && non_finite<D>(columns)) left_out = true;
        else accumulate<D>(dk, columns, ds);
    });
    if (left_out) {
        walk([&](const float* q_base, const float* do_base, int row0, const acc_t& prob, const acc_t& ds) __attribute__((always_inline)) {
            if (!masked(row0)) return;
            auto visible = [&](int i) { return row0 + i >= first_query; };
            ColumnOperand<D> columns;
            columns.load(do_base, q_stride, row0, p.qs, p.d);
            if (non_finite<D>(columns)) accumulate_visible<D>(dv, do_base, q_stride, row0, p.qs, p.d, prob, visible);
            columns.load(q_base, q_stride, row0, p.qs, p.d);
            if (non_finite<D>(columns)) accumulate_visible<D>(dk, q_base, q_stride, row0, p.qs, p.d, ds, visible);
        });
    }
    const long count = static_cast<long>(p.batch) * p.ks * kv_stride;
    float* const dk_out = p.parts == 1 ? p.dk : p.partial + 2 * part * count;
    float* const dv_out = p.parts == 1 ? p.dv : p.partial + (2 * part + 1) * count;
    auto store_to = [&](float* out) {
        return [&, out](int row, int at, f32x4 sum) {
            if (k0 + row >= p.ks) return;
            float* to = out + (static_cast<long>(b) * p.ks + k0 + row) * kv_stride + static_cast<long>(kvh) * p.d + at;
            if (p.accumulate && p.parts == 1) sum += load_vec<float, 4>(to);
            store_vec<float, 4>(to, sum);
        };
    };
    deposit<D>(lds, wave, dk, p.scale);
    __syncthreads();
    collect<D>(lds, p.d, store_to(dk_out));
    __syncthreads();
    deposit<D>(lds, wave, dv, 1.0f);
    __syncthreads();
    collect<D>(lds, p.d, store_to(dv_out));
}

template <auto Kernel, int SMEM>
int launch(dim3 grid, const AttentionF32Args& args, hipStream_t stream) {
    if (grid.y > 65535u || grid.z > 65535u) return fail(CGPTX_OVERFLOW, "attention: grid too large");
    static const hipError_t status =
        hipFuncSetAttribute(reinterpret_cast<const void*>(Kernel), hipFuncAttributeMaxDynamicSharedMemorySize, SMEM);
    CGPTX_HIP(status);
    hipLaunchKernelGGL(Kernel, grid, dim3(kThreads), SMEM, stream, args);
    CGPTX_LAUNCH_CHECK();
    return CGPTX_OK;
}

dim3 grid_over(int rows, int heads, int batch) {
    return dim3(static_cast<unsigned int>((rows + kTile - 1) / kTile), static_cast<unsigned int>(heads), static_cast<unsigned int>(batch));
}

}  // namespace

bool attention_f32_takes(std::size_t head_dim, bool aligned) { return aligned && head_dim % 4 == 0 && head_dim <= 128; }

int attention_f32_forward(const AttentionF32Args& a, hipStream_t stream) {
    const dim3 grid = grid_over(a.qs, a.hq, a.batch);
    return a.d <= 64 ? launch<attention_f32_forward_kernel<64>, kSmemBytes<64>>(grid, a, stream)
                     : launch<attention_f32_forward_kernel<128>, kSmemBytes<128>>(grid, a, stream);
}

int attention_f32_backward(const AttentionF32Args& a, hipStream_t stream) {
    const dim3 q_grid = grid_over(a.qs, a.hq, a.batch);
    dim3 k_grid = grid_over(a.ks, a.hkv, a.batch);
    k_grid.x *= static_cast<unsigned int>(a.parts);
    if (int s = a.d <= 64 ? launch<attention_f32_dq_kernel<64>, kSmemBytes<64>>(q_grid, a, stream)
                          : launch<attention_f32_dq_kernel<128>, kSmemBytes<128>>(q_grid, a, stream))
        return s;
    return a.d <= 64 ? launch<attention_f32_dkv_kernel<64>, kSmemBytes<64>>(k_grid, a, stream)
                     : launch<attention_f32_dkv_kernel<128>, kSmemBytes<128>>(k_grid, a, stream);
}

}  // namespace cgptx
