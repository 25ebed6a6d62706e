// The projections of q, k and v as the step of a small model makes them: several contractions in one launch
// (cgpt_amd/csrc/gemm.hpp), forward as a group of three, backward as one of four whose input gradient reads its operand from
// three buffers. Operands of -1 .. 1: sums of at most 8192 products are exact in fp32 in any order, so every result is the
// rounded exact value. Built by `python -m cgpt_amd.build`; run by tests/test_cpp_interface.py on the GPU. Also what else of a step's parts no
// entry point of the library reaches: a norm's gradient added to the residual stream's.
#include <cmath>
#include <cstdio>
#include <cstring>
#include <random>
#include <stdexcept>
#include <string>
#include <vector>

#include "gemm.hpp"

namespace {

using cgptx::GemmArgs;
using Bits = std::vector<std::uint16_t>;

int failures = 0;
void expect(bool ok, const std::string& what) {
    if (!ok) {
        ++failures;
        std::printf("FAIL %s\n", what.c_str());
    }
}
void hip_ok(hipError_t status, const char* what) {
    if (status != hipSuccess) throw std::runtime_error(std::string(what) + ": " + hipGetErrorString(status));
}

// Nearest even, of whole numbers far from either type's limits.
std::uint16_t rounded(int value, int dtype) {
    std::uint16_t out;
    if (dtype == CGPTX_F16) {
        const auto half = static_cast<_Float16>(value);
        std::memcpy(&out, &half, 2);
        return out;
    }
    const auto f = static_cast<float>(value);
    std::uint32_t bits;
    std::memcpy(&bits, &f, 4);
    return static_cast<std::uint16_t>((bits + 0x7fff + (bits >> 16 & 1)) >> 16);
}

struct Matrix {
    std::size_t rows, cols;
    std::vector<int> values;
    int at(std::size_t r, std::size_t c) const { return values[r * cols + c]; }
};
Matrix random_matrix(std::size_t rows, std::size_t cols, std::mt19937& rng) {
    Matrix m{rows, cols, std::vector<int>(rows * cols)};
    for (int& v : m.values) v = static_cast<int>(rng() % 3) - 1;
    return m;
}
// Sum over t of a(t) b(t), for element (i, j) of a result.
template <typename A, typename B>
Bits product(std::size_t m, std::size_t n, std::size_t k, int dtype, A&& a, B&& b) {
    Bits out(m * n);
    for (std::size_t i = 0; i < m; ++i)
        for (std::size_t j = 0; j < n; ++j) {
            int sum = 0;
            for (std::size_t t = 0; t < k; ++t) sum += a(i, t) * b(t, j);
            out[i * n + j] = rounded(sum, dtype);
        }
    return out;
}

// Device memory with guards before and behind it.
class Buffer {
public:
    explicit Buffer(std::size_t count) : count_(count), host_(count + 2 * kGuard, kPoison) { allocate(); }
    Buffer(const Matrix& m, int dtype) : count_(m.values.size()), host_(count_ + 2 * kGuard, kPoison) {
        for (std::size_t i = 0; i < count_; ++i) host_[kGuard + i] = rounded(m.values[i], dtype);
        allocate();
    }
    Buffer(const Buffer&) = delete;
    ~Buffer() { (void)hipFree(base_); }
    std::uint16_t* data() const { return base_ + kGuard; }
    // What the buffer holds; false if a guard does not.
    bool copy(Bits& out) {
        hip_ok(hipMemcpy(host_.data(), base_, host_.size() * 2, hipMemcpyDeviceToHost), "hipMemcpy");
        for (std::size_t i = 0; i < kGuard; ++i)
            if (host_[i] != kPoison || host_[kGuard + count_ + i] != kPoison) return false;
        out.assign(host_.begin() + kGuard, host_.begin() + kGuard + static_cast<std::ptrdiff_t>(count_));
        return true;
    }
    bool holds(const Bits& want) {
        Bits held;
        return copy(held) && held == want;
    }

private:
    void allocate() {
        hip_ok(hipMalloc(reinterpret_cast<void**>(&base_), host_.size() * 2), "hipMalloc");
        hip_ok(hipMemcpy(base_, host_.data(), host_.size() * 2, hipMemcpyHostToDevice), "hipMemcpy");
    }
    static constexpr std::size_t kGuard = 512;
    static constexpr std::uint16_t kPoison = 0x7fc1;  // no number in either type
    std::size_t count_;
    std::vector<std::uint16_t> host_;
    std::uint16_t* base_ = nullptr;
};

void check(std::size_t rows, std::size_t hidden, std::size_t q, std::size_t k, std::size_t v, int dtype, hipStream_t stream) {
    const std::string name = std::to_string(rows) + " x " + std::to_string(hidden) + ", " + std::to_string(q) + " + " +
                             std::to_string(k) + " + " + std::to_string(v) + (dtype == CGPTX_F16 ? " f16" : " bf16");
    std::printf("%s\n", name.c_str());
    std::fflush(stdout);
    std::mt19937 rng(static_cast<unsigned int>(rows + hidden + q + v));
    const std::size_t width[3] = {q, k, v}, total = q + k + v;
    const Matrix x = random_matrix(rows, hidden, rng), w = random_matrix(total, hidden, rng);
    const Matrix dy[3] = {random_matrix(rows, q, rng), random_matrix(rows, k, rng), random_matrix(rows, v, rng)};
    const Buffer on_x(x, dtype), on_w(w, dtype), on_dq(dy[0], dtype), on_dk(dy[1], dtype), on_dv(dy[2], dtype);
    const Buffer* on_dy[3] = {&on_dq, &on_dk, &on_dv};
    Buffer y_q(rows * q), y_k(rows * k), y_v(rows * v), dw_q(q * hidden), dw_k(k * hidden), dw_v(v * hidden), dx(rows * hidden);
    Buffer *y[3] = {&y_q, &y_k, &y_v}, *dw[3] = {&dw_q, &dw_k, &dw_v};

    GemmArgs forward[3], backward[4];
    GemmArgs& input = backward[0];  // dX = [dq | dk | dv]·W
    input.b = on_w.data();
    input.c = dx.data();
    input.m = rows;
    input.n = input.ldb = input.ldc = hidden;
    input.k = total;
    input.b_k_contiguous = false;
    input.dtype = dtype;
    input.a_segments.count = 3;
    std::size_t first[3] = {0, q, q + k};
    for (int i = 0; i < 3; ++i) {
        GemmArgs& f = forward[i];  // Y = X·Wᵀ
        f.a = on_x.data();
        f.b = on_w.data() + first[i] * hidden;
        f.c = y[i]->data();
        f.m = rows;
        f.n = f.ldc = width[i];
        f.k = f.lda = f.ldb = hidden;
        f.dtype = dtype;
        GemmArgs& b = backward[i + 1];  // dW = dYᵀ·X
        b.a = on_dy[i]->data();
        b.b = on_x.data();
        b.c = dw[i]->data();
        b.m = b.lda = width[i];
        b.n = b.ldb = b.ldc = hidden;
        b.k = rows;
        b.a_k_contiguous = b.b_k_contiguous = false;
        b.dtype = dtype;
        input.a_segments.ptr[i] = on_dy[i]->data();
        input.a_segments.ld[i] = input.a_segments.cols[i] = width[i];
    }
    const cgptx::GemmGroup forward_group = cgptx::gemm_joins(forward, 3), backward_group = cgptx::gemm_joins(backward, 4);
    expect(forward_group.joined, name + ": the projections share no launch");
    expect(backward_group.joined, name + ": the gradients share no launch");
    if (!forward_group.joined || !backward_group.joined) return;
    expect(cgptx::gemm_joined(forward, 3, forward_group, stream) == CGPTX_OK, name + ": forward launch");
    expect(cgptx::gemm_joined(backward, 4, backward_group, stream) == CGPTX_OK, name + ": backward launch");
    hip_ok(hipStreamSynchronize(stream), "hipStreamSynchronize");

    const auto dy_at = [&](std::size_t r, std::size_t c) { return c < q ? dy[0].at(r, c) : c < q + k ? dy[1].at(r, c - q) : dy[2].at(r, c - q - k); };
    expect(dx.holds(product(rows, hidden, total, dtype, dy_at, [&](std::size_t t, std::size_t j) { return w.at(t, j); })), name + ": dX");
    for (int i = 0; i < 3; ++i) {
        expect(y[i]->holds(product(rows, width[i], hidden, dtype, [&](std::size_t r, std::size_t t) { return x.at(r, t); },
                                   [&](std::size_t t, std::size_t j) { return w.at(first[i] + j, t); })),
               name + ": Y " + std::to_string(i));
        expect(dw[i]->holds(product(width[i], hidden, rows, dtype, [&](std::size_t c, std::size_t t) { return dy[i].at(t, c); },
                                    [&](std::size_t t, std::size_t j) { return x.at(t, j); })),
               name + ": dW " + std::to_string(i));
    }
}

// The input gradient of q, k and v over many rows, whose operand comes from three buffers: few enough columns and rows that tiles of
// 256 x 192 fill the chip where 256 x 256 do not, ragged both ways. Some rows are compared, the last ones among them.
void check_many_rows(std::size_t rows, std::size_t hidden, std::size_t q, std::size_t k, std::size_t v, int dtype, hipStream_t stream) {
    const std::string name = "input gradient of " + std::to_string(rows) + " rows" + (dtype == CGPTX_F16 ? " f16" : " bf16");
    std::printf("%s\n", name.c_str());
    std::fflush(stdout);
    std::mt19937 rng(static_cast<unsigned int>(rows + hidden));
    const std::size_t width[3] = {q, k, v}, total = q + k + v;
    const Matrix w = random_matrix(total, hidden, rng);
    const Matrix dy[3] = {random_matrix(rows, q, rng), random_matrix(rows, k, rng), random_matrix(rows, v, rng)};
    const Buffer on_w(w, dtype), on_dq(dy[0], dtype), on_dk(dy[1], dtype), on_dv(dy[2], dtype);
    const Buffer* on_dy[3] = {&on_dq, &on_dk, &on_dv};
    Buffer dx(rows * hidden);
    GemmArgs input;
    input.b = on_w.data();
    input.c = dx.data();
    input.m = rows;
    input.n = input.ldb = input.ldc = hidden;
    input.k = total;
    input.b_k_contiguous = false;
    input.dtype = dtype;
    input.a_segments.count = 3;
    for (int i = 0; i < 3; ++i) {
        input.a_segments.ptr[i] = on_dy[i]->data();
        input.a_segments.ld[i] = input.a_segments.cols[i] = width[i];
    }
    expect(cgptx::gemm(input, stream) == CGPTX_OK, name + ": launch");
    hip_ok(hipStreamSynchronize(stream), "hipStreamSynchronize");
    std::vector<std::size_t> some;
    for (std::size_t r = 0; r < rows; r += 331) some.push_back(r);
    for (std::size_t r = rows - 3; r < rows; ++r) some.push_back(r);
    const auto dy_at = [&](std::size_t i, std::size_t c) {
        return c < q ? dy[0].at(some[i], c) : c < q + k ? dy[1].at(some[i], c - q) : dy[2].at(some[i], c - q - k);
    };
    const Bits want = product(some.size(), hidden, total, dtype, dy_at, [&](std::size_t t, std::size_t j) { return w.at(t, j); });
    Bits got(rows * hidden);
    expect(dx.copy(got), name + ": guards");
    for (std::size_t i = 0; i < some.size(); ++i)
        expect(std::memcmp(&got[some[i] * hidden], &want[i * hidden], hidden * 2) == 0, name + ": row " + std::to_string(some[i]));
}

class Floats {
public:
    explicit Floats(std::size_t count) : count_(count) { hip_ok(hipMalloc(reinterpret_cast<void**>(&data_), count * 4), "hipMalloc"); }
    explicit Floats(const std::vector<float>& from) : Floats(from.size()) {
        hip_ok(hipMemcpy(data_, from.data(), count_ * 4, hipMemcpyHostToDevice), "hipMemcpy");
    }
    Floats(const Floats&) = delete;
    ~Floats() { (void)hipFree(data_); }
    float* data() const { return data_; }
    std::vector<float> copy() const {  // after all that was launched
        std::vector<float> out(count_);
        hip_ok(hipDeviceSynchronize(), "hipDeviceSynchronize");
        hip_ok(hipMemcpy(out.data(), data_, count_ * 4, hipMemcpyDeviceToHost), "hipMemcpy");
        return out;
    }

private:
    std::size_t count_;
    float* data_ = nullptr;
};

// The same input gradient in fp32, where the group is launched for its one call in segments: its error against 64 bits is that of
// three calls which add to each other's result, not that of one sum over all segments. A sum's error grows with its length: one
// chain of three equal parts has some 1.7 times the error of three.
void check_segment_sums(std::size_t rows, std::size_t hidden, std::size_t q, std::size_t k, hipStream_t stream) {
    const std::string name = "fp32 input gradient, " + std::to_string(rows) + " x " + std::to_string(hidden) + ", " + std::to_string(q) + " + 2 x " + std::to_string(k);
    std::printf("%s\n", name.c_str());
    std::fflush(stdout);
    std::mt19937 rng(static_cast<unsigned int>(rows + q));
    std::normal_distribution<float> normal;
    const std::size_t width[3] = {q, k, k}, total = q + 2 * k;
    auto random = [&](std::size_t count) {
        std::vector<float> v(count);
        for (float& x : v) x = normal(rng);
        return v;
    };
    const std::vector<float> w = random(total * hidden), x = random(rows * hidden), dy[3] = {random(rows * q), random(rows * k), random(rows * k)};
    Floats on_w(w), on_x(x), dx(rows * hidden), dw(total * hidden);
    Floats on_dy[3] = {Floats(dy[0]), Floats(dy[1]), Floats(dy[2])};
    GemmArgs calls[4];
    GemmArgs& input = calls[0];
    input.b = on_w.data();
    input.c = dx.data();
    input.m = rows;
    input.n = input.ldb = input.ldc = hidden;
    input.k = total;
    input.b_k_contiguous = false;
    input.dtype = CGPTX_F32;
    input.a_segments.count = 3;
    std::size_t first = 0;
    for (int i = 0; i < 3; ++i) {
        GemmArgs& b = calls[1 + i];
        b.a = on_dy[i].data();
        b.b = on_x.data();
        b.c = dw.data() + first * hidden;
        b.m = b.lda = width[i];
        b.n = b.ldb = b.ldc = hidden;
        b.k = rows;
        b.a_k_contiguous = b.b_k_contiguous = false;
        b.dtype = CGPTX_F32;
        input.a_segments.ptr[i] = on_dy[i].data();
        input.a_segments.ld[i] = input.a_segments.cols[i] = width[i];
        first += width[i];
    }
    // Root mean square of the error of some rows.
    auto error = [&](const std::vector<float>& got) {
        double sum = 0.0;
        for (std::size_t r = 0; r < rows; r += 7)
            for (std::size_t c = 0; c < hidden; ++c) {
                double exact = 0.0;
                std::size_t t = 0;
                for (int i = 0; i < 3; ++i)
                    for (std::size_t j = 0; j < width[i]; ++j, ++t) exact += static_cast<double>(dy[i][r * width[i] + j]) * w[t * hidden + c];
                sum += (got[r * hidden + c] - exact) * (got[r * hidden + c] - exact);
            }
        return std::sqrt(sum / static_cast<double>((rows + 6) / 7 * hidden));
    };
    cgptx::GemmGroup group = cgptx::gemm_joins(calls, 4, stream);
    expect(group.joined, name + ": the gradients share no launch");
    if (!group.joined) return;
    for (const int tile : {32, 64})
        for (const bool deep : {false, true}) {
            for (int& t : group.tile) t = tile;
            group.deep = deep;
            expect(cgptx::gemm_joined(calls, 4, group, stream) == CGPTX_OK, name + ": launch");
            const double joined = error(dx.copy());
            // What it stands for, in the same tiles: each projection's pair of gradients, the input gradients added up.
            first = 0;
            for (int i = 0; i < 3; ++i) {
                GemmArgs pair[2] = {input, calls[1 + i]};
                pair[0].a_segments = {};
                pair[0].a = on_dy[i].data();
                pair[0].lda = pair[0].k = width[i];
                pair[0].b = on_w.data() + first * hidden;
                pair[0].accumulate = i > 0;
                first += width[i];
                expect(cgptx::gemm_joined(pair, 2, group, stream) == CGPTX_OK, name + ": launch of a pair");
            }
            const double apart = error(dx.copy());
            std::printf("  tiles of %d%s: error %.3g, apart %.3g\n", tile, deep ? ", deep" : "", joined, apart);
            expect(joined <= 1.1 * apart, name + ": larger error in one launch");
        }
}

// Y = X·Wᵀ on tiles of 256 x 192, ragged both ways, with all that their epilogue adds: a residual, sums in fp32, what C holds, into C of
// either kind. Whole numbers, exact in fp32 whatever the order. Some rows are compared, and the guards around C.
void check_narrow_epilogue(int dtype, hipStream_t stream) {
    const std::size_t rows = 16300, columns = 760, k = 1024;
    std::mt19937 rng(7);
    const Matrix x = random_matrix(rows, k, rng), w = random_matrix(columns, k, rng);
    auto wide = [&](int most) {
        Matrix m{rows, columns, std::vector<int>(rows * columns)};
        for (int& v : m.values) v = static_cast<int>(rng() % (2 * most + 1)) - most;
        return m;
    };
    const Matrix residual = wide(100), addend = wide(1000), old = wide(100);
    const Buffer on_x(x, dtype), on_w(w, dtype), on_residual(residual, dtype);
    const Floats on_addend(std::vector<float>(addend.values.begin(), addend.values.end()));
    std::vector<std::size_t> some;
    for (std::size_t r = 0; r < rows; r += 331) some.push_back(r);
    for (std::size_t r = rows - 3; r < rows; ++r) some.push_back(r);
    std::vector<int> products;
    for (const std::size_t r : some)
        for (std::size_t c = 0; c < columns; ++c) {
            int sum = 0;
            for (std::size_t t = 0; t < k; ++t) sum += x.at(r, t) * w.at(c, t);
            products.push_back(sum);
        }
    struct Form {
        const char* name;
        bool residual, addend, accumulate, f32;
    };
    for (const Form form : {Form{"residual", true, false, false, false}, {"addend", false, true, false, false}, {"addend and residual", true, true, false, false},
                            {"old C", false, false, true, false}, {"addend and old C", false, true, true, false}, {"fp32", false, false, false, true},
                            {"fp32, old C", false, false, true, true}, {"fp32, addend", false, true, false, true}}) {
        const std::string name = std::string("256 x 192 tiles, ") + form.name + (dtype == CGPTX_F16 ? " f16" : " bf16");
        std::printf("%s\n", name.c_str());
        std::fflush(stdout);
        Buffer c16(old, dtype);
        Floats c32(std::vector<float>(old.values.begin(), old.values.end()));
        GemmArgs g;
        g.a = on_x.data();
        g.b = on_w.data();
        g.c = form.f32 ? static_cast<void*>(c32.data()) : c16.data();
        g.m = rows;
        g.n = g.ldc = columns;
        g.k = g.lda = g.ldb = k;
        g.dtype = dtype;
        g.c_is_f32 = form.f32;
        g.accumulate = form.accumulate;
        if (form.residual) g.residual = on_residual.data(), g.ldr = columns;
        if (form.addend) g.addend_f32 = on_addend.data(), g.ld_addend = columns;
        expect(cgptx::gemm(g, stream) == CGPTX_OK, name + ": launch");
        hip_ok(hipStreamSynchronize(stream), "hipStreamSynchronize");
        Bits got;
        expect(c16.copy(got), name + ": guards");
        const std::vector<float> got32 = c32.copy();
        for (std::size_t i = 0; i < some.size(); ++i)
            for (std::size_t c = 0; c < columns; ++c) {
                const std::size_t at = some[i] * columns + c;
                const int want = products[i * columns + c] + (form.residual ? residual.values[at] : 0) + (form.addend ? addend.values[at] : 0) +
                                 (form.accumulate ? old.values[at] : 0);
                const bool same = form.f32 ? got32[at] == static_cast<float>(want) : got[at] == rounded(want, dtype);
                if (same) continue;
                expect(false, name + ": row " + std::to_string(some[i]) + ", column " + std::to_string(c));
                break;
            }
    }
}

// What oblong tiles take beside plain products, ragged both ways and along K: an input gradient whose operand comes from three buffers, a forward
// product into three, and a residual that is not C. The shapes' tiles are held by gemm_plan_test.cpp. Some rows are compared, and all guards.
void check_oblong_forms(std::size_t rows, std::size_t columns, std::size_t k, int dtype, hipStream_t stream) {
    const std::string name = "oblong tiles, " + std::to_string(rows) + " x " + std::to_string(columns) + " x " + std::to_string(k) + (dtype == CGPTX_F16 ? " f16" : " bf16");
    std::printf("%s\n", name.c_str());
    std::fflush(stdout);
    std::mt19937 rng(static_cast<unsigned int>(rows + k));
    std::vector<std::size_t> some;
    for (std::size_t r = 0; r < rows; r += 997) some.push_back(r);
    for (std::size_t r = rows - 3; r < rows; ++r) some.push_back(r);
    auto expect_rows = [&](const Bits& got, std::size_t width, const Bits& want, std::size_t want_width, std::size_t first, const char* what) {
        for (std::size_t i = 0; i < some.size(); ++i)
            expect(std::memcmp(&got[some[i] * width], &want[i * want_width + first], width * 2) == 0, name + ", " + what + ": row " + std::to_string(some[i]));
    };
    auto launch = [&](const GemmArgs& g, const char* what) {
        expect(cgptx::gemm(g, stream) == CGPTX_OK, name + ", " + what + ": launch");
        hip_ok(hipStreamSynchronize(stream), "hipStreamSynchronize");
    };
    {
        const std::size_t n = columns - 8, width[3] = {k / 2, k / 4, k / 4}, first[3] = {0, k / 2, k / 4 * 3};
        const Matrix w = random_matrix(k, n, rng), dy[3] = {random_matrix(rows, width[0], rng), random_matrix(rows, width[1], rng), random_matrix(rows, width[2], rng)};
        const Buffer on_w(w, dtype), on_dq(dy[0], dtype), on_dk(dy[1], dtype), on_dv(dy[2], dtype);
        const Buffer* on_dy[3] = {&on_dq, &on_dk, &on_dv};
        Buffer dx(rows * n);
        GemmArgs g;
        g.b = on_w.data();
        g.c = dx.data();
        g.m = rows;
        g.n = g.ldb = g.ldc = n;
        g.k = k;
        g.b_k_contiguous = false;
        g.dtype = dtype;
        g.a_segments.count = 3;
        for (int i = 0; i < 3; ++i) {
            g.a_segments.ptr[i] = on_dy[i]->data();
            g.a_segments.ld[i] = g.a_segments.cols[i] = width[i];
        }
        launch(g, "three operands");
        const Bits want = product(some.size(), n, k, dtype, [&](std::size_t i, std::size_t t) {
            const int s = t < first[1] ? 0 : t < first[2] ? 1 : 2;
            return dy[s].at(some[i], t - first[s]);
        }, [&](std::size_t t, std::size_t j) { return w.at(t, j); });
        Bits got;
        expect(dx.copy(got), name + ", three operands: guards");
        expect_rows(got, n, want, n, 0, "three operands");
    }
    const std::size_t short_k = k - 32;  // ends inside a K tile
    const Matrix x = random_matrix(rows, short_k, rng), w = random_matrix(columns, short_k, rng);
    const Buffer on_x(x, dtype), on_w(w, dtype);
    GemmArgs forward;
    forward.a = on_x.data();
    forward.b = on_w.data();
    forward.m = rows;
    forward.k = forward.lda = forward.ldb = short_k;
    forward.dtype = dtype;
    const Bits want = product(some.size(), columns, short_k, dtype, [&](std::size_t i, std::size_t t) { return x.at(some[i], t); },
                              [&](std::size_t t, std::size_t j) { return w.at(j, t); });
    {
        const std::size_t q = columns - 512;
        Buffer y_q(rows * q), y_k(rows * 256), y_v(rows * 256);
        Buffer* const y[3] = {&y_q, &y_k, &y_v};
        const std::size_t width[3] = {q, 256, 256}, first[3] = {0, q, q + 256};
        GemmArgs g = forward;
        g.n = columns;
        g.c_segments.count = 3;
        for (int i = 0; i < 3; ++i) {
            g.c_segments.ptr[i] = y[i]->data();
            g.c_segments.ld[i] = g.c_segments.cols[i] = width[i];
        }
        launch(g, "three results");
        for (int i = 0; i < 3; ++i) {
            Bits got;
            expect(y[i]->copy(got), name + ", three results: guards");
            expect_rows(got, width[i], want, columns, first[i], "three results");
        }
    }
    {
        const std::size_t n = columns - 8;
        const Matrix residual = random_matrix(rows, n, rng);
        const Buffer on_residual(residual, dtype);
        Buffer y(rows * n);
        GemmArgs g = forward;
        g.n = g.ldc = g.ldr = n;
        g.c = y.data();
        g.residual = on_residual.data();
        launch(g, "residual");
        Bits got, sum(some.size() * n);
        expect(y.copy(got), name + ", residual: guards");
        for (std::size_t i = 0; i < some.size(); ++i)
            for (std::size_t j = 0; j < n; ++j) {
                int exact = residual.at(some[i], j);
                for (std::size_t t = 0; t < short_k; ++t) exact += x.at(some[i], t) * w.at(j, t);
                sum[i * n + j] = rounded(exact, dtype);
            }
        expect_rows(got, n, sum, n, 0, "residual");
    }
}

// A norm's input gradient on top of the residual stream's: into a buffer of its own, and in place of it, as a step's blocks add their
// second branch. Without an output gradient the residual comes out as it went in; with one, both ways give the same bits.
void check_residual_in_place(std::size_t rows, std::size_t hidden, int dtype, hipStream_t stream) {
    const std::string name = "norm gradient on a residual, " + std::to_string(rows) + " x " + std::to_string(hidden) + ", type " + std::to_string(dtype);
    std::printf("%s\n", name.c_str());
    std::fflush(stdout);
    const std::size_t elem = dtype == CGPTX_F32 ? 4 : 2, count = rows * hidden;
    std::mt19937 rng(static_cast<unsigned int>(rows + hidden));
    using Bytes = std::vector<unsigned char>;
    auto numbers = [&](std::size_t n, int most) {
        Bytes bytes(n * elem);
        for (std::size_t i = 0; i < n; ++i) {
            const int value = static_cast<int>(rng() % (2 * most + 1)) - most;
            const auto f = static_cast<float>(value);
            const std::uint16_t half = rounded(value, dtype);
            std::memcpy(&bytes[i * elem], elem == 4 ? static_cast<const void*>(&f) : &half, elem);
        }
        return bytes;
    };
    std::vector<void*> held;
    auto on_device = [&](const Bytes& bytes) {
        void* p = nullptr;
        hip_ok(hipMalloc(&p, bytes.size()), "hipMalloc");
        hip_ok(hipMemcpy(p, bytes.data(), bytes.size(), hipMemcpyHostToDevice), "hipMemcpy");
        held.push_back(p);
        return p;
    };
    const Bytes residual = numbers(count, 100), nothing(count * elem);
    void* const x = on_device(numbers(count, 5));
    void* const w = on_device(numbers(hidden, 3));
    void* const dw = on_device(Bytes(hidden * elem));
    void* const apart = on_device(residual);
    for (const Bytes& gradient : {nothing, numbers(count, 7)}) {
        void* const dy = on_device(gradient);
        void* const out = on_device(nothing);
        void* const in_place = on_device(residual);
        expect(cgptx::rmsnorm_backward_residual(out, dw, dy, x, w, apart, rows, hidden, 1e-5f, dtype, stream) == CGPTX_OK, name + ": launch");
        expect(cgptx::rmsnorm_backward_residual(in_place, dw, dy, x, w, in_place, rows, hidden, 1e-5f, dtype, stream) == CGPTX_OK, name + ": launch in place");
        hip_ok(hipStreamSynchronize(stream), "hipStreamSynchronize");
        Bytes got(count * elem), got_in_place(count * elem);
        hip_ok(hipMemcpy(got.data(), out, got.size(), hipMemcpyDeviceToHost), "hipMemcpy");
        hip_ok(hipMemcpy(got_in_place.data(), in_place, got.size(), hipMemcpyDeviceToHost), "hipMemcpy");
        expect(got == got_in_place, name + ": in place");
        if (gradient == nothing) expect(got == residual, name + ": no gradient");
        else if (hidden > 1) expect(got != residual, name + ": a gradient");  // of one column it is next to nothing
    }
    for (void* p : held) (void)hipFree(p);
}

}  // namespace

int main() {
    try {
        hipStream_t stream = nullptr;
        hip_ok(hipStreamCreate(&stream), "hipStreamCreate");
        for (const int dtype : {CGPTX_F16, CGPTX_BF16}) {
            check(1, 64, 64, 64, 32, dtype, stream);        // the last segment is half a K tile
            check(33, 96, 128, 64, 96, dtype, stream);      // one row behind a 32-wide tile, a step more than whole K tiles
            check(100, 256, 256, 128, 128, dtype, stream);  // 3 x 100 tokens' kind: segments of whole K tiles
            check(131, 224, 192, 64, 160, dtype, stream);   // ragged rows and columns, five steps in the last segment
            check(300, 512, 512, 64, 224, dtype, stream);   // more rows than one tile of either size
            check_many_rows(16300, 760, 1024, 512, 512, dtype, stream);
            check_narrow_epilogue(dtype, stream);
            check_oblong_forms(5003, 1024, 1024, dtype, stream);   // 160 x 128
            check_oblong_forms(6999, 768, 2048, dtype, stream);    // 192 x 128
            check_oblong_forms(8161, 1024, 4096, dtype, stream);   // 256 x 128
            check_oblong_forms(9999, 1024, 1024, dtype, stream);   // 160 x 256
            check_oblong_forms(11871, 1024, 1024, dtype, stream);  // 192 x 256
            check_oblong_forms(12470, 1024, 1024, dtype, stream);  // 224 x 256
        }
        for (const int dtype : {CGPTX_F32, CGPTX_F16, CGPTX_BF16})
            for (const std::size_t hidden : {1, 18, 20, 36, 64, 180, 1021, 1024, 5003})  // rows of whole vectors and others
                for (const std::size_t rows : {1, 130, 2500}) check_residual_in_place(rows, hidden, dtype, stream);
        check_segment_sums(300, 512, 512, 512, stream);
        check_segment_sums(131, 768, 768, 256, stream);
        check_segment_sums(70, 224, 96, 32, stream);  // wavefronts without a K tile of some segments
        hip_ok(hipStreamDestroy(stream), "hipStreamDestroy");
    } catch (const std::exception& e) {
        std::printf("FAIL %s\n", e.what());
        ++failures;
    }
    std::printf("%d failure(s)\n", failures);
    return failures == 0 ? 0 : 1;
}
