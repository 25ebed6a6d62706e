// How contractions are cut and which of them share a launch: the rules of cgpt_amd/csrc/gemm.hip, read where they stand. Host code
// only, no GPU needed. Built by `python -m cgpt_amd.build`; run by tests/test_cpp_interface.py.
#include <cstdio>
#include <cstring>
#include <random>
#include <string>

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

}  // namespace

int main(int argc, char** argv) {
    if (argc > 1 && std::strcmp(argv[1], "pinned") == 0) check_pinned();
    std::printf("%d failure(s)\n", failures);
    return failures == 0 ? 0 : 1;
}
