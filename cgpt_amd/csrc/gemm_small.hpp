// Host interface of the small-contraction kernel (gemm_small_kernel.hpp), one translation unit per storage type.
#pragma once

#include "gemm.hpp"

namespace cgptx {

struct SmallSegments {
    const void* ptr[3];
    long ld[3];
    int cols[3];
    int count;
};

// Everything a plain call reads comes first: a workgroup's start waits for as few scalar loads as possible.
struct SmallArgs {
    const void* a;
    const void* b;
    void* c;  // T*, float* when c_f32, float partial tiles when split
    long lda, ldb, ldc;  // ldc: row length of a partial tile matrix when split
    int m, n, k;
    int a_extent, b_extent, b_k;  // see GemmArgs
    int k_tiles, k_tiles_per_slice;
    // the general epilogue
    const void* bias;
    const void* residual;
    const float* addend;
    long ldr, ld_addend;
    int accumulate, c_f32, ragged;
    // grouped weight gradients: sums of A's columns, T*, or null
    void* a_sums;
    int a_sums_accumulate;
    // segmented operands
    SmallSegments a_seg, c_seg;
};

enum class SmallEpilogue { plain, general, split };

struct SmallCall {
    SmallArgs args;
    bool a_k_contiguous, b_k_contiguous;
    int tile;   // 32 or 64
    bool deep;  // twice the LDS stages, one workgroup per CU instead of two
    SmallEpilogue epilogue;
    int slices;
};

// Several calls in one launch: call i takes the workgroups from first_block[i] on, tile rows first.
enum class SmallLayout { forward, input_gradient, weight_gradient, segmented_input_gradient };
// The launch's arguments hold as many calls as its kernel is made for.
template <int CALLS>
struct SmallGroup {
    SmallArgs call[CALLS];
    int first_block[CALLS];
    int tiles_m[CALLS];
    int tile[CALLS];  // 32 or 64
    SmallLayout layout[CALLS];
    int count;
};

int gemm_small_bf16(const SmallCall& call, hipStream_t stream);
int gemm_small_f16(const SmallCall& call, hipStream_t stream);
int gemm_small_f32(const SmallCall& call, hipStream_t stream);
int gemm_small_bf16(const SmallGroup<kFewCalls>& group, int blocks, bool deep, hipStream_t stream);
int gemm_small_bf16(const SmallGroup<kGroupCalls>& group, int blocks, bool deep, hipStream_t stream);
int gemm_small_f16(const SmallGroup<kFewCalls>& group, int blocks, bool deep, hipStream_t stream);
int gemm_small_f16(const SmallGroup<kGroupCalls>& group, int blocks, bool deep, hipStream_t stream);
int gemm_small_f32(const SmallGroup<kFewCalls>& group, int blocks, bool deep, hipStream_t stream);
int gemm_small_f32(const SmallGroup<kGroupCalls>& group, int blocks, bool deep, hipStream_t stream);

}  // namespace cgptx
