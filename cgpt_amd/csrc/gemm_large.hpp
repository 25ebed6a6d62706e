// Host interface of the persistent contraction kernels (gemm_large_kernel.hpp), one translation unit per storage type.
#pragma once

#include "gemm.hpp"

namespace cgptx {

constexpr int kLdsBytes = 160 * 1024;  // of a CU

struct KernelSegments {
    const void* ptr[3];
    long ld[3];
    int cols[3];
    int count;
};

struct KernelArgs {
    const void* a;
    const void* b;
    void* c;            // T* (or float* when c_f32), or float partials when split
    const void* bias;
    const void* residual;  // T*, row stride ldr, or null
    const float* addend;   // fp32 [M, N], row stride ld_addend, added before anything else, or null
    long ld_addend;
    int m, n, k;
    // What the operands hold: rows or columns of A and of B (A's may exceed m, B's n: whole 16-byte chunks of padded
    // rows), K positions of B (below k when A's padding reaches further: past them B reads as zeros).
    int a_extent, b_extent, b_k;
    int k_tiles;            // K tiles of kBK, the last one possibly short
    int ragged;             // C (or an addend) has rows that are not whole 16-byte chunks: stored element by element
    long ld_partial;        // SPLIT kernels: row length of a partial tile matrix
    long lda, ldb, ldc, ldr;
    int tiles_m, tiles_n;
    int k_tiles_per_slice;  // K tiles handled by one work item
    int slices;             // K slices per output tile
    int accumulate;
    int c_f32;
    KernelSegments a_seg, c_seg;  // column segments of A (as stored) and of C; count 0 = one buffer
    // ceil(2^32 / (group rows * tiles_n)) when multiplying by it divides every item index of the
    // launch exactly, else 0 (the kernel then divides).
    unsigned int group_reciprocal;
    int group_rows_log2;  // tile-rows per L2 locality group: 1 << group_rows_log2
    void* act;      // SWIGLU kernels: [M, inter] = silu(gate) * up, T*
    long ld_act;
    const void* saved;  // GRAD kernels: the forward's [M, 2 * inter] = [gate | up], T*
    long ld_saved;
    int inter;      // SWIGLU kernels: columns of gate (= of up); n = 2 * inter
    // Stacked products (weight-gradient layout only): rows of C per product (0 = one product) and what a and b (or
    // A's segments) move by from one product to the next, in elements.
    int batch_rows;
    long a_batch_stride, b_batch_stride;
    long a_seg_batch_stride[3];
    // Calls of a pair: partial tiles of K slices and a ticket per tile (slices > 1); weight gradients: sums of A's columns, T*, or null.
    unsigned char* fold_partial;
    unsigned int* fold_tickets;
    void* a_sums;
    int a_sums_accumulate;
};

// The input and the weight gradient of a projection in one launch; each call's tiles_m, tiles_n, slices and
// k_tiles_per_slice are set.
constexpr int fold_tile_bytes(int rows, int columns) { return rows * columns * 4 + rows * 4; }  // of a tile's slice: accumulators, and sums of A's columns
constexpr int kPairWeightRows = 256, kPairWeightColumns = 128;  // the weight gradient's tile beside an oblong one of the input gradient
struct PairArgs {
    KernelArgs input, weight;
    int input_tile;  // 128: both on 128 x 128 tiles
    int first_blocks, weight_first;  // set by the launch: the workgroups of the call that starts first
};

// Tiles by a number: the edge of a square one, 192 for 256 rows of 192 columns, and these for oblong ones (16-bit storage).
constexpr int oblong_tile(int rows, int columns) { return rows * 1000 + columns; }
constexpr int tile_rows(int tile) { return tile > 256 ? tile / 1000 : tile == 192 ? 256 : tile; }
constexpr int tile_columns(int tile) { return tile > 256 ? tile % 1000 : tile; }

struct LargeCall {
    KernelArgs args;
    bool a_k_contiguous, b_k_contiguous;
    int tile;    // 128 or, in 16-bit storage, 256, 192 or an oblong one
    bool split;  // fp32 partial tiles of K slices
    int slices;
};

int gemm_large_bf16(const LargeCall& call, hipStream_t stream);
int gemm_large_f16(const LargeCall& call, hipStream_t stream);
int gemm_large_f32(const LargeCall& call, hipStream_t stream);
int gemm_oblong_bf16(const LargeCall& call, hipStream_t stream);
int gemm_oblong_f16(const LargeCall& call, hipStream_t stream);
int gemm_pair_bf16(const PairArgs& pair, hipStream_t stream);
int gemm_pair_f16(const PairArgs& pair, hipStream_t stream);
int gemm_oblong_pair_bf16(const PairArgs& pair, hipStream_t stream);
int gemm_oblong_pair_f16(const PairArgs& pair, hipStream_t stream);

}  // namespace cgptx
