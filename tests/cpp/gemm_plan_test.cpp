// How contractions are cut and which of them share a launch: the rules of cgpt_amd/csrc/gemm.hip, read where they stand. Host code
// only, no GPU needed. Built by `python -m cgpt_amd.build`; run by tests/test_cpp_interface.py.
#include <algorithm>
#include <cstdio>
#include <cstring>
#include <random>
#include <string>
#include <vector>

#include "cross_entropy.hpp"
#include "gemm.hip"

namespace {

using namespace cgptx;

int failures = 0;
void expect(bool ok, const std::string& what) {
    if (!ok) {
        ++failures;
        std::printf("FAIL %s\n", what.c_str());
    }
}

// An aligned address that nothing reads.
void* address(std::size_t offset = 0) { return reinterpret_cast<void*>(std::size_t{1} << 40 | offset); }

enum class Kind { forward, input_gradient, weight_gradient };

GemmArgs contraction(Kind kind, std::size_t m, std::size_t n, std::size_t k, int dtype) {
    GemmArgs g;
    g.a = address();
    g.b = address();
    g.c = address();
    g.m = m;
    g.n = n;
    g.k = k;
    g.a_k_contiguous = kind != Kind::weight_gradient;
    g.b_k_contiguous = kind == Kind::forward;
    g.lda = g.a_k_contiguous ? k : m;
    g.ldb = g.b_k_contiguous ? k : n;
    g.ldc = n;
    g.dtype = dtype;
    return g;
}

std::string name_of(const GemmArgs& g) {
    return std::string(g.dtype == CGPTX_F32 ? "f32" : g.dtype == CGPTX_F16 ? "f16" : "bf16") + " [" + std::to_string(g.m) + ", " +
           std::to_string(g.n) + "] x " + std::to_string(g.k) + (g.a_k_contiguous ? g.b_k_contiguous ? " Y" : " dX" : " dW");
}

// CGPTX_GEMM_TILE=192: a call that has no kernel of 256 x 192 tiles is planned for one that it has.
void check_pinned() {
    expect(forced_tile() == 192, "started without CGPTX_GEMM_TILE=192");
    for (const Kind kind : {Kind::forward, Kind::input_gradient, Kind::weight_gradient})
        for (const std::size_t m : {33, 300, 5005, 16384})
            for (const std::size_t n : {96, 760, 2048})
                for (const std::size_t k : {64, 1024, 8192}) {
                    const GemmArgs f32 = contraction(kind, m, n, k, CGPTX_F32);
                    const Plan plan = make_plan(f32);
                    expect(plan.tile == 32 || plan.tile == 64 || plan.tile == 128, name_of(f32) + ": tiles of " + std::to_string(plan.tile));
                    GemmArgs bf16 = contraction(kind, m, n, k, CGPTX_BF16);
                    const bool many = Plan::tiles_of(bf16, 256) >= 3 * compute_units();
                    expect(make_plan(bf16).tile == (many ? 256 : 192), name_of(bf16) + ": not as pinned");
                    bf16.bias = address();
                    expect(make_plan(bf16).tile != 192, name_of(bf16) + ": 256 x 192 tiles add no bias");
                }
}

// Calls whose columns leave square tiles idle take 256 x 192 ones where C and all that is added lie in whole aligned chunks: those
// tiles have no other epilogue. The rest is served by square tiles, element by element.
void check_narrow() {
    for (const int dtype : {CGPTX_BF16, CGPTX_F16})
        for (const Kind kind : {Kind::forward, Kind::input_gradient}) {
            const GemmArgs plain = contraction(kind, 16384, 768, 4096, dtype);
            auto expect_tile = [&](const GemmArgs& g, bool narrow, const char* what) {
                expect((make_plan(g).tile == 192) == narrow, name_of(g) + ", " + what + ": tiles of " + std::to_string(make_plan(g).tile));
                expect(make_plan(g).tile != 192 || c_streams(g, 2), name_of(g) + ", " + what + ": tiles without an epilogue for it");
            };
            expect_tile(plain, true, "plain");
            for (const std::size_t offset : {0, 2, 8}) {  // residuals are read four elements at a time
                GemmArgs g = plain;
                g.residual = address(offset);
                g.ldr = 768;
                expect_tile(g, offset != 2, "residual");
                g.ldr = 770;
                expect_tile(g, false, "residual in rows of 770");
            }
            for (const std::size_t offset : {0, 4, 8}) {
                GemmArgs g = plain;
                g.addend_f32 = static_cast<const float*>(address(offset));
                g.ld_addend = 768;
                expect_tile(g, offset == 0, "addend");
                g.ld_addend = 770;
                expect_tile(g, false, "addend in rows of 770");
            }
            GemmArgs g = plain;
            g.c = address(8);
            expect_tile(g, false, "C on 8 bytes");
            g.c = address();
            g.ldc = 772;
            expect_tile(g, false, "C in rows of 772");
        }
}

// Oblong tiles take the place of large square ones only, where the call is one sum over K and has nothing but a residual, its own C or (a forward
// product) a bias added: results keep their bits, and every such plan has a kernel.
void check_oblong() {
    int taken = 0;
    for (const int dtype : {CGPTX_BF16, CGPTX_F16, CGPTX_F32})
        for (const Kind kind : {Kind::forward, Kind::input_gradient, Kind::weight_gradient})
            for (std::size_t m = 100; m <= 40000; m += m / 7)
                for (const std::size_t n : {640, 768, 1000, 1024, 1536, 2048, 4096})
                    for (const std::size_t k : {64, 768, 1024, 4096})
                        for (const int extra : {0, 1, 2, 3, 4, 5}) {
                            GemmArgs g = contraction(kind, m, n, k, dtype);
                            if (extra == 1) g.residual = address(), g.ldr = n;
                            if (extra == 2) g.accumulate = true;
                            if (extra == 3) g.bias = address();
                            if (extra == 4) g.c = address(8);
                            if (extra == 5) g.c_is_f32 = true;
                            const Plan plan = make_plan(g);
                            if (plan.tile <= 256) continue;
                            ++taken;
                            const std::string name = name_of(g) + ": tiles of " + std::to_string(plan.tile);
                            expect((extra < 3 || (extra == 3 && kind == Kind::forward)) && dtype != CGPTX_F32 && kind != Kind::weight_gradient && plan.slices == 1, name);
                            expect(tile_rows(plan.tile) % 32 == 0 && tile_columns(plan.tile) % 128 == 0, name);
                            expect(Plan::tiles_of(g, 128) > compute_units() || g.bias != nullptr, name + " where every square one has a CU");
                            GemmArgs square = g;  // as it was planned without them
                            square.c = address(8);
                            const Plan other = make_plan(square);
                            expect(other.slices == 1 && other.tile >= 128, name + " for " + std::to_string(other.tile) + " in " + std::to_string(other.slices));
                        }
    expect(taken > 500, std::to_string(taken) + " calls on oblong tiles");
    // Measured (see kOblongCosts, oblong_has_to_beat, lone_blocks_us): who gains and who loses by them.
    struct {
        std::size_t m, n, k;
        bool gains, gains_with_bias;
    } const measured[] = {{5005, 1024, 1024, true, true},    {5005, 1024, 2048, true, true},    {5005, 2048, 1024, true, true},
                          {7000, 768, 2048, true, true},     {10000, 1024, 1024, true, true},   {13000, 4096, 1024, true, true},
                          {16384, 768, 768, true, true},     {8192, 1024, 2048, true, true},    {30304, 2048, 256, true, true},
                          {22226, 640, 4096, true, true},    {3000, 1024, 4096, false, false},  {2000, 1280, 4096, false, false},
                          {1552, 1536, 1024, false, true},   {1670, 1280, 1024, false, true},   {5984, 512, 4096, false, false},
                          {19504, 640, 4096, false, true},   {33416, 640, 2048, false, true},   {28856, 2048, 2048, false, true},
                          {30304, 4096, 768, false, true},   {16384, 1024, 1024, false, false}, {2000, 2048, 1024, false, false}};
    for (const auto& call : measured)
        for (const int added : {0, 1, 2}) {
            GemmArgs g = contraction(added == 1 ? Kind::input_gradient : Kind::forward, call.m, call.n, call.k, CGPTX_BF16);
            if (added == 2) g.bias = address();
            const int tile = make_plan(g).tile;
            expect((tile > 256) == (added == 2 ? call.gains_with_bias : call.gains), name_of(g) + (added == 2 ? " + bias" : "") + ": tiles of " + std::to_string(tile));
        }
    // Both gradients of a projection: one round of workgroups, C of either in whole aligned chunks.
    int pairs_taken = 0;
    for (std::size_t rows = 500; rows <= 20000; rows += rows / 9)
        for (const std::size_t in : {640, 768, 1000, 1024, 2048})
            for (const std::size_t out : {256, 1024, 2048, 4096})
                for (const int extra : {0, 1, 2, 3, 4}) {
                    GemmArgs calls[2] = {contraction(Kind::input_gradient, rows, in, out, CGPTX_BF16), contraction(Kind::weight_gradient, out, in, rows, CGPTX_BF16)};
                    if (extra == 1) calls[0].accumulate = true;
                    if (extra == 2) calls[1].accumulate = true, calls[1].a_sums = address();
                    if (extra == 3) calls[0].c = address(8);
                    if (extra == 4) calls[1].c = address(8);
                    const GemmGroup plan = plan_group(calls, 2, true);
                    if (!plan.pair || plan.tile[0] <= 256) continue;
                    ++pairs_taken;
                    const long items = Plan::tiles_of(calls[0], plan.tile[0]) + tiles_of_size(calls[1], kPairWeightRows, kPairWeightColumns) * plan.slices;
                    expect(extra < 3 && items <= compute_units(), name_of(calls[0]) + ": " + std::to_string(items) + " workgroups for a pair");
                }
    expect(pairs_taken > 20, std::to_string(pairs_taken) + " pairs on oblong tiles");
    // One on every XCD: either call's tiles are dealt out by themselves.
    for (std::size_t rows = 500; rows <= 20000; rows += rows / 23)
        for (const std::size_t in : {576, 640, 768, 1000, 1024, 1152, 1408, 2048, 2304})
            for (const std::size_t out : {256, 1024, 1792, 2048, 2304, 2560, 3584, 4096}) {
                const GemmArgs calls[2] = {contraction(Kind::input_gradient, rows, in, out, CGPTX_BF16), contraction(Kind::weight_gradient, out, in, rows, CGPTX_BF16)};
                const GemmGroup plan = plan_group(calls, 2, true);
                if (!plan.pair || plan.tile[0] <= 256) continue;
                const long input = Plan::tiles_of(calls[0], plan.tile[0]), weight = tiles_of_size(calls[1], kPairWeightRows, kPairWeightColumns) * plan.slices;
                expect(((input + 7) / 8 + (weight + 7) / 8) * 8 <= compute_units(),
                       name_of(calls[0]) + ": " + std::to_string(input) + " and " + std::to_string(weight) + " workgroups for a pair");
            }
    // Columns in segments are whole tiles of 256; an input gradient's segments along K take nothing added.
    GemmArgs g = contraction(Kind::input_gradient, 5005, 1024, 1536, CGPTX_BF16);
    g.a_segments.count = 3;
    expect(make_plan(g).tile > 256, "segments along K");
    g.accumulate = true;
    expect(make_plan(g).tile <= 256, "segments along K, added to C");
}

// The tiles that tests of values are there for: tests/test_gpu_linear.py's products (forward, with a bias, as an input gradient, added to C) and
// gemm_group_test.cpp's (an operand or a result in three buffers, a residual).
void check_oblong_shapes() {
    struct Shape {
        std::size_t rows, k, n;
        int tile;
    };
    auto expect_tile = [](const GemmArgs& g, int tile, const char* what) {
        const int taken = make_plan(g).tile;
        expect(taken == tile, name_of(g) + ", " + what + ": tiles of " + std::to_string(taken));
    };
    for (const int dtype : {CGPTX_BF16, CGPTX_F16}) {
        for (const Shape& s : {Shape{5005, 1024, 1024, 160128}, {4833, 992, 1000, 160128}, {7000, 2048, 768, 192128}, {8999, 1728, 640, 192128}, {8161, 4096, 1024, 256128},
                               {5005, 1024, 2048, 160256}, {10000, 1024, 1016, 160256}, {11900, 1024, 1024, 192256}, {11871, 992, 1016, 192256}, {12500, 1024, 1024, 224256},
                               {13001, 1024, 4096, 224256}}) {
            GemmArgs g = contraction(Kind::forward, s.rows, s.n, s.k, dtype);
            expect_tile(g, s.tile, "forward");
            g.bias = address();
            expect_tile(g, s.tile, "bias");
            g = contraction(Kind::input_gradient, s.rows, s.n, s.k, dtype);
            expect_tile(g, s.tile, "input gradient");
            g.accumulate = true;
            expect_tile(g, s.tile, "added");
        }
        for (const Shape& s : {Shape{5003, 1024, 1024, 160128}, {6999, 2048, 768, 192128}, {8161, 4096, 1024, 256128}, {9999, 1024, 1024, 160256}, {11871, 1024, 1024, 192256},
                               {12470, 1024, 1024, 224256}}) {
            GemmArgs g = contraction(Kind::input_gradient, s.rows, s.n - 8, s.k, dtype);
            g.a = nullptr;
            g.a_segments.count = 3;
            for (int i = 0; i < 3; ++i) {
                g.a_segments.ptr[i] = address();
                g.a_segments.ld[i] = g.a_segments.cols[i] = i == 0 ? s.k / 2 : s.k / 4;
            }
            expect_tile(g, s.tile, "three operands");
            g = contraction(Kind::forward, s.rows, s.n, s.k - 32, dtype);
            g.c_segments.count = 3;
            for (int i = 0; i < 3; ++i) {
                g.c_segments.ptr[i] = address();
                g.c_segments.ld[i] = g.c_segments.cols[i] = i == 0 ? s.n - 512 : 256;
            }
            expect_tile(g, s.tile, "three results");
            g = contraction(Kind::forward, s.rows, s.n - 8, s.k - 32, dtype);
            g.residual = address();
            g.ldr = s.n - 8;
            expect_tile(g, s.tile, "residual");
        }
    }
}

// Both gradients of a projection (rows, in, out), measured in one launch: each tile and slice count of the pairs on oblong tiles at ragged shapes, those
// that gain by them, and those that do not and keep 128 x 128 tiles.
void check_oblong_pairs() {
    struct {
        std::size_t rows, in, out;
        int tile, slices;
    } const ragged[] = {{732, 1368, 2208, 160128, 1},  {2419, 656, 3104, 160128, 2},  {3691, 400, 2208, 160128, 3}, {779, 3960, 1184, 160256, 1},
                        {3336, 1040, 1824, 160256, 2}, {2957, 720, 1184, 160256, 3},  {2323, 648, 3104, 192128, 1}, {3226, 600, 1632, 192128, 3},
                        {1080, 3624, 1056, 192256, 1}, {3963, 1040, 1632, 192256, 2}, {5180, 968, 1504, 192256, 3}, {1196, 3616, 1056, 224256, 1},
                        {3965, 1160, 1440, 224256, 2}, {4010, 1192, 1248, 224256, 3}, {2732, 776, 3232, 256128, 1}, {3004, 792, 1184, 256128, 3}};
    auto plan_of = [](std::size_t rows, std::size_t in, std::size_t out, int dtype, bool accumulate, bool bias) {
        GemmArgs calls[2] = {contraction(Kind::input_gradient, rows, in, out, dtype), contraction(Kind::weight_gradient, out, in, rows, dtype)};
        calls[0].accumulate = calls[1].accumulate = accumulate;
        if (bias) calls[1].a_sums = address();
        return plan_group(calls, 2, true);
    };
    auto named = [](std::size_t rows, std::size_t in, std::size_t out, const GemmGroup& plan) {
        return std::to_string(rows) + " x " + std::to_string(in) + " x " + std::to_string(out) + (plan.pair ? ": pair of tile " : plan.joined ? ": group of tile " : ": apart, ") +
               std::to_string(plan.tile[0]) + " in " + std::to_string(plan.slices);
    };
    for (const auto& shape : ragged)
        for (const int dtype : {CGPTX_BF16, CGPTX_F16})
            for (const bool accumulate : {false, true}) {
                const GemmGroup plan = plan_of(shape.rows, shape.in, shape.out, dtype, accumulate, true);
                expect(plan.pair && plan.tile[0] == shape.tile && plan.slices == shape.slices, named(shape.rows, shape.in, shape.out, plan));
            }
    struct {
        std::size_t rows, in, out;
        bool gains;
    } const measured[] = {{5005, 1024, 2048, true},  {6000, 1024, 2048, true},  {6983, 760, 2048, true},   {7000, 768, 2048, true},   {3425, 1536, 3072, true},
                          {5862, 896, 3840, true},   {5005, 1024, 1024, false}, {4096, 768, 2048, false},  {2816, 896, 2944, false},  {1615, 1792, 1472, false},
                          {3357, 1024, 2688, false}, {6546, 384, 2944, false},  {1508, 1408, 1792, false}, {17175, 256, 640, false},
                          {26156, 768, 1920, false}, {4978, 256, 3840, false}};
    for (const auto& shape : measured) {
        const GemmGroup plan = plan_of(shape.rows, shape.in, shape.out, CGPTX_BF16, false, false);
        expect(plan.pair && (plan.tile[0] > 256) == shape.gains, named(shape.rows, shape.in, shape.out, plan));
    }
}

// A step holds memory for its tokens by id where they are grouped beside their lookup: up to 8192 tokens.
void check_token_groups() {
    for (const std::size_t vocab : {std::size_t{1}, std::size_t{517}, std::size_t{50257}, std::size_t{1} << 20})
        for (const std::size_t tokens : {1, 300, 4096, 8191, 8192, 8193, 32768, 1 << 20}) {
            const std::size_t bytes = embedding_groups_ahead_bytes(tokens, vocab), all = (vocab + 1 + tokens) * sizeof(unsigned int);
            expect(tokens <= 8192 ? bytes == 0 || (bytes >= all && bytes < all + 256) : bytes == 0,
                   std::to_string(tokens) + " tokens of " + std::to_string(vocab) + " ids: " + std::to_string(bytes) + " bytes");
            expect(tokens > 4096 || vocab > 50257 || bytes != 0, std::to_string(tokens) + " tokens of " + std::to_string(vocab) + " ids are not grouped ahead");
        }
    expect(embedding_groups_ahead_bytes(0, 100) == 0 && embedding_groups_ahead_bytes(100, 0) == 0 && embedding_groups_ahead_bytes(100, std::size_t{1} << 31) == 0, "no such step");
}

// q's, k's and v's gradients over `rows` tokens as one group: their input gradients as one call in segments, then the weight gradients.
struct Gradients {
    GemmArgs calls[4], input[3];
    Gradients(std::size_t rows, std::size_t hidden, std::size_t q, std::size_t k, int dtype) {
        const std::size_t width[3] = {q, k, k};
        calls[0] = contraction(Kind::input_gradient, rows, hidden, q + 2 * k, dtype);
        calls[0].a = nullptr;
        calls[0].a_segments.count = 3;
        for (int i = 0; i < 3; ++i) {
            calls[0].a_segments.ptr[i] = address();
            calls[0].a_segments.ld[i] = calls[0].a_segments.cols[i] = width[i];
            calls[1 + i] = contraction(Kind::weight_gradient, width[i], hidden, rows, dtype);
            input[i] = contraction(Kind::input_gradient, rows, hidden, width[i], dtype);
        }
    }
};
// Additions that follow each other in a sum of a call by itself: four wavefronts share a small tile's K range.
double chain(const GemmArgs& g) {
    const Plan plan = make_plan(g);
    return static_cast<double>(g.k) / (plan.slices * (plan.tile <= 64 ? 4 : 1));
}

// fp32: a group gives no sum a longer chain of additions than the calls that it stands for have, each with its weight gradient.
void check_chains() {
    int joined = 0, refused = 0;
    for (const std::size_t head_dim : {32, 64, 128})
        for (const std::size_t kv : {1, 2, 4})
            for (const std::size_t group : {1, 2, 4})
                for (std::size_t rows = 32; rows <= 2048; rows += rows / 8) {
                    const std::size_t q = head_dim * kv * group, k = head_dim * kv;
                    const Gradients of(rows, q, q, k, CGPTX_F32);
                    const bool together = gemm_segments_add_as_joined(of.calls, nullptr) && gemm_joins(of.calls, 4).joined;
                    (together ? joined : refused) += 1;
                    if (!together) continue;
                    for (int i = 0; i < 3; ++i) {
                        const GemmArgs pair[2] = {of.input[i], of.calls[1 + i]};
                        if (gemm_joins(pair, 2).joined) continue;
                        for (const GemmArgs& g : pair)
                            expect(static_cast<double>(g.k) / 4 <= 1.01 * chain(g), name_of(g) + ": a chain of " + std::to_string(g.k / 4) + " for " + std::to_string(chain(g)));
                    }
                }
    expect(joined > 100 && refused > 10, std::to_string(joined) + " groups joined, " + std::to_string(refused) + " not");
}

// The prediction of a pair stops short where it cannot be below what the caller has already; it never says otherwise than the whole one.
void check_predictions() {
    std::mt19937 rng(4);
    int stopped = 0;
    for (int i = 0; i < 3000; ++i) {
        const long tiles_x = 1 + static_cast<long>(rng() % 4000), tiles_w = 1 + static_cast<long>(rng() % 1000), steps_x = 2 + static_cast<long>(rng() % 128);
        const long steps_w = 2 + static_cast<long>(rng() % 1024), slices = 1 + static_cast<long>(rng() % 12);
        auto predicted = [&](double worth) { return predicted_pair_us(tiles_x, steps_x, tiles_w, steps_w, slices, 256, worth); };
        const double whole = predicted(std::numeric_limits<double>::infinity());
        for (const double worth : {0.5 * whole, 0.97 * whole, 1.03 * whole}) {
            const double short_of = predicted(worth);
            stopped += short_of != whole;
            expect((short_of < worth) == (whole < worth) && (short_of >= worth || short_of == whole),
                   std::to_string(whole) + " predicted as " + std::to_string(short_of) + " for " + std::to_string(worth));
        }
    }
    expect(stopped > 100, "nothing was stopped short");
}

// The counters of tiles in K slices: the last workgroup of a launch, and only it, finds zero; launches that meet on a counter, whose
// workgroups come in any order, may mistake each other's for the last one, but leave zero for the next.
void check_counters() {
    std::mt19937 rng(3);
    unsigned int counter = 0;
    auto launch = [&](std::vector<int> slice_counts) {  // how often somebody found zero
        std::vector<unsigned int> shares;
        for (const int slices : slice_counts)
            for (int s = 0; s < slices; ++s) shares.push_back(fold_share(s, slices));
        std::shuffle(shares.begin(), shares.end(), rng);
        int last = 0;
        for (std::size_t i = 0; i < shares.size(); ++i) {
            counter += shares[i];
            if (counter == 0) {
                ++last;
                if (slice_counts.size() == 1) expect(i + 1 == shares.size(), "an early last workgroup of " + std::to_string(slice_counts[0]));
            }
        }
        return last;
    };
    for (int slices = 2; slices <= 16; ++slices)
        for (int other = 2; other <= 16; ++other) {
            const std::string name = std::to_string(slices) + " and " + std::to_string(other) + " slices";
            launch({slices, other});
            expect(counter == 0, name + ": the counter is left at " + std::to_string(counter));
            launch({other, slices, other});
            expect(counter == 0, name + ": the counter is left at " + std::to_string(counter) + " by three");
            for (const int alone : {slices, other}) expect(launch({alone}) == 1, name + ": not one last workgroup afterwards");
        }
}

// The rows in which a step's dense loss leaves its gradient never take its row pass from whole vectors to elements, and are whole chunks
// wherever that costs nothing.
void check_loss_rows() {
    int streamed = 0;
    for (const int dtype : {CGPTX_F32, CGPTX_F16, CGPTX_BF16}) {
        const std::size_t vec = 16 / dtype_size(dtype), held = kMostHeldVectors * vec;
        for (const std::size_t vocab : {std::size_t{203}, std::size_t{50257}, held - 1, held, held + 1, held + vec - 1, held + vec, held + vec + 1, held + 3 * vec + 2, 2 * held - 1})
            for (const std::size_t rows : {1, 33, 512}) {
                const std::size_t pitch = cross_entropy_gradient_pitch(rows, 128, vocab, dtype);
                const std::string name = std::to_string(rows) + " rows of " + std::to_string(vocab) + " logits of type " + std::to_string(dtype);
                expect(cross_entropy_in_vectors(vocab, vocab, pitch, dtype), name + ": by elements, gradient in rows of " + std::to_string(pitch));
                if (vocab / vec > kMostHeldVectors) ++streamed;
                else expect(pitch == linear_backward_pitch(rows, 128, vocab, dtype), name + ": gradient in rows of " + std::to_string(pitch));
            }
    }
    expect(streamed >= 30, std::to_string(streamed) + " streamed shapes");
}

}  // namespace

int main(int argc, char** argv) {
    if (argc > 1 && std::strcmp(argv[1], "pinned") == 0) check_pinned();
    if (argc > 1 && std::strcmp(argv[1], "chains") == 0) check_chains();
    if (argc > 1 && std::strcmp(argv[1], "narrow") == 0) check_narrow();
    if (argc > 1 && std::strcmp(argv[1], "oblong") == 0) check_oblong();
    if (argc > 1 && std::strcmp(argv[1], "oblong_pairs") == 0) check_oblong_pairs();
    if (argc > 1 && std::strcmp(argv[1], "counters") == 0) check_counters();
    if (argc > 1 && std::strcmp(argv[1], "predictions") == 0) check_predictions();
    if (argc > 1 && std::strcmp(argv[1], "oblong_shapes") == 0) check_oblong_shapes();
    if (argc > 1 && std::strcmp(argv[1], "token_groups") == 0) check_token_groups();
    if (argc > 1 && std::strcmp(argv[1], "loss_rows") == 0) check_loss_rows();
    std::printf("%d failure(s)\n", failures);
    return failures == 0 ? 0 : 1;
}
