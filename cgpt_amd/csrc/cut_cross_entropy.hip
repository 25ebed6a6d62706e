// Cut cross-entropy: loss and both gradients of a linear classifier without ever
// holding the [rows, vocabulary] logits.
//
// Semantics: include/ops/cut_cross_entropy.h:25-33 (src/ops/cut_cross_entropy.cu:97-221):
//   z = X·Cᵀ, loss = mean_r(logsumexp z_r − z_{r,y_r}),
//   dX = (softmax(z) − onehot)·C / rows, dC = (softmax(z) − onehot)ᵀ·X / rows.
// The reference recomputes full dot products per thread (O(rows·hidden²·vocab)), which
// cannot run at training size. Here rows are processed in chunks of at most 1 GiB of logits: one
// MFMA contraction produces the chunk's logits into scratch, the softmax kernel turns them into
// the scaled logit gradient in place, and two more contractions consume that gradient (dX for the
// chunk's rows; dC accumulated in fp32 across chunks — the last chunk's contraction adds the
// accumulator in its epilogue — so the classifier gradient is rounded once; a single chunk writes
// it straight out of its contraction, which rounds the same sum in another order of additions).
// Scratch is chunk·vocab logits + vocab·hidden fp32, independent of the number of rows, and three
// vocabulary-sized contractions are done instead of four because the chunk's logits stay resident
// between loss and gradient.
//
// Extensions over the reference: any storage dtype, a gradient scale (loss scaling),
// and accumulate_classifier for tied embeddings.
#include "cross_entropy.hpp"
#include "gemm.hpp"

#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <limits>

namespace cgptx {
namespace {

// row_losses: null, or where the rows' losses are left, in place of their mean in `loss`.
int run(float* loss, float* row_losses, void* input_gradient, void* classifier_gradient, const void* input, const void* classifier,
        const std::uint32_t* targets, std::size_t rows, std::size_t hidden, std::size_t vocab, float gradient_scale,
        int accumulate_classifier, int dtype, hipStream_t stream) {
    const char* name = "cut_cross_entropy";
    if (!valid_dtype(dtype)) return fail(CGPTX_INVALID_ARGUMENT, std::string(name) + ": unsupported dtype");
    if ((loss == nullptr && row_losses == nullptr) || input_gradient == nullptr || classifier_gradient == nullptr || input == nullptr ||
        classifier == nullptr || targets == nullptr || rows == 0 || hidden == 0 || vocab == 0)
        return fail(CGPTX_INVALID_ARGUMENT,
                    std::string(name) + ": input and classifier must be non-empty matrices with gradients and targets");
    if (!std::isfinite(gradient_scale) || gradient_scale <= 0.0f)
        return fail(CGPTX_INVALID_ARGUMENT, std::string(name) + ": gradient scale must be finite and positive");
    constexpr std::size_t i32max = std::numeric_limits<int>::max();
    if (rows > i32max || hidden > i32max || vocab > i32max)
        return fail(CGPTX_OVERFLOW, std::string(name) + ": dimension exceeds int range");
    const std::size_t elem = dtype_size(dtype);
    // Rows are processed in chunks so that the logits scratch stays within 1 GiB whatever the number of rows
    // (CGPTX_CUT_CE_LOGITS_BYTES, read per call, sets another bound, up to 2 GiB - 1 MiB: the streamed contraction
    // kernels address an operand with 32-bit byte offsets below that). The rows are split evenly over the chunks.
    // At V = 32000 in 16-bit storage the bound gives chunks of 16384 rows, which still fill the chip: 64 x 4 tiles
    // of a chunk's input gradient, one per compute unit. Measured at [32768, 1024] x [32000, 1024]: 1 GiB costs
    // nothing against one 2 GiB chunk (6.04 - 6.12 against 6.03 - 6.05 ms), 512 MiB 3.5 % (the input gradient of an
    // 8192-row chunk has to be split along K), 256 MiB 8 %.
    constexpr std::size_t kMaxLogitsBytes = (std::size_t{1} << 31) - (std::size_t{1} << 20);
    std::size_t logits_bytes = std::size_t{1} << 30;
    if (const char* text = std::getenv("CGPTX_CUT_CE_LOGITS_BYTES")) {
        const unsigned long long asked = std::strtoull(text, nullptr, 0);
        if (asked > 0) logits_bytes = std::min<std::size_t>(static_cast<std::size_t>(asked), kMaxLogitsBytes);
    }
    // Rows of logits are padded to whole cache lines (128 bytes, a K tile of the input gradient's contraction): an odd
    // vocabulary then streams like any other (bf16 2048 x 768 x 50257: 552 us with rows of whole 64 bytes, 545 so). The
    // padding holds zeros: columns of Z the classifier has no rows for, and cleared by the softmax pass.
    std::size_t pitch = 0, chunk = 0, loss_bytes = 0, acc_bytes = 0, logit_bytes = 0;
    bool single = true;
    auto lay_out = [&](std::size_t row_length) {
        pitch = row_length;
        std::size_t limit = logits_bytes / (pitch * elem);
        limit = std::max<std::size_t>(256, limit / 256 * 256);
        const std::size_t pieces = (rows + limit - 1) / limit;
        chunk = ((rows + pieces - 1) / pieces + 255) / 256 * 256;
        chunk = std::min(chunk, rows);
        single = chunk >= rows;
        loss_bytes = (rows * sizeof(float) + 255) & ~std::size_t{255};
        acc_bytes = single ? 0 : (vocab * hidden * sizeof(float) + 255) & ~std::size_t{255};
        logit_bytes = (chunk * pitch * elem + 255) & ~std::size_t{255};
    };
    lay_out((vocab + 128 / elem - 1) / (128 / elem) * (128 / elem));
    // The gradients' contractions may be split along K (a chunk's input gradient has few output tiles and the vocabulary
    // as its K, a small vocabulary's gradient few tiles and the rows); their partial tiles get room of their own.
    auto input_gradient_call = [&](std::size_t r0, std::size_t r) {  // dX[r, H] = dZ[r, V]·C[V, H]
        GemmArgs dx;
        dx.b = classifier;
        dx.c = static_cast<char*>(input_gradient) + r0 * hidden * elem;
        dx.m = r;
        dx.n = hidden;
        dx.k = pitch;
        dx.b_k = vocab;
        dx.lda = pitch;
        dx.ldb = hidden;
        dx.ldc = hidden;
        dx.b_k_contiguous = false;
        dx.dtype = dtype;
        return dx;
    };
    auto classifier_gradient_call = [&](std::size_t r0, std::size_t r) {  // dC[V, H] = dZᵀ[V, r]·X[r, H]
        GemmArgs dc;
        dc.b = static_cast<const char*>(input) + r0 * hidden * elem;
        dc.m = vocab;
        dc.a_extent = pitch;
        dc.n = hidden;
        dc.k = r;
        dc.lda = pitch;
        dc.ldb = hidden;
        dc.ldc = hidden;
        dc.a_k_contiguous = false;
        dc.b_k_contiguous = false;
        dc.dtype = dtype;
        return dc;
    };
    std::size_t split_bytes = 0;
    for (const std::size_t r : {chunk, (rows - 1) % chunk + 1})
        split_bytes = std::max({split_bytes, gemm_split_bytes(input_gradient_call(0, r)), gemm_split_bytes(classifier_gradient_call(0, r))});
    split_bytes = (split_bytes + 255) & ~std::size_t{255};
    void* mem = nullptr;
    std::size_t held = 0;
    // Arena layout: [row_loss | acc | split-K partials | logits]. The contractions below run with no_split: they
    // never ask the arena for scratch of their own, and split only into the room given to them here. An arena that
    // cannot grow is used as it is: less room to split into, and logits without padding before none at all.
    auto needed = [&] { return loss_bytes + acc_bytes + logit_bytes; };
    if (int s = scratch_up_to(stream, needed() + split_bytes, &mem, &held)) return s;
    if (held < needed()) {
        if (int s = scratch_up_to(stream, needed(), &mem, &held)) return s;
    }
    if (held < needed()) {
        lay_out(vocab);
        if (int s = scratch(stream, needed(), &mem)) return s;
        held = std::max(held, needed());
    }
    split_bytes = std::min(split_bytes, (held - needed()) & ~std::size_t{255});
    auto* base = static_cast<char*>(mem);
    auto* row_loss = row_losses != nullptr ? row_losses : reinterpret_cast<float*>(base);
    auto* acc = reinterpret_cast<float*>(base + loss_bytes);
    void* split_room = split_bytes != 0 ? base + loss_bytes + acc_bytes : nullptr;
    void* logits = base + loss_bytes + acc_bytes + split_bytes;
    const float factor = gradient_scale / static_cast<float>(rows);
    bool mean_taken = false;
    for (std::size_t r0 = 0; r0 < rows; r0 += chunk) {
        const std::size_t r = std::min(chunk, rows - r0);
        const void* x = static_cast<const char*>(input) + r0 * hidden * elem;
        GemmArgs z;  // logits[r, V] = X[r, H]·C[V, H]ᵀ
        z.a = x;
        z.b = classifier;
        z.c = logits;
        z.m = r;
        z.n = pitch;
        z.b_extent = vocab;
        z.k = hidden;
        z.lda = hidden;
        z.ldb = hidden;
        z.ldc = pitch;
        z.dtype = dtype;
        z.no_split = true;
        if (int s = gemm(z, stream)) return s;
        if (int s = cross_entropy_rows(row_loss + r0, logits, pitch, logits, pitch, targets + r0, r, vocab, factor, dtype, stream,
                                       single ? loss : nullptr, &mean_taken))
            return s;
        GemmArgs dx = input_gradient_call(r0, r);
        dx.a = logits;
        dx.no_split = true;
        dx.split_workspace = split_room;
        dx.split_workspace_bytes = split_bytes;
        if (int s = gemm(dx, stream)) return s;
        // dC = Σ_chunks dZᵀ[V, r]·X[r, H]: all chunks but the last add their product to acc (fp32; the first one
        // starts it), the last one adds acc to its own and writes the gradient, rounded once. A single chunk
        // writes the gradient itself.
        const bool last = r0 + chunk >= rows;
        GemmArgs dc = classifier_gradient_call(r0, r);
        dc.a = logits;
        dc.c = last ? classifier_gradient : static_cast<void*>(acc);
        dc.accumulate = last ? accumulate_classifier != 0 : r0 != 0;
        dc.c_is_f32 = !last;
        if (last && !single) {
            dc.addend_f32 = acc;
            dc.ld_addend = hidden;
        }
        dc.no_split = true;
        dc.split_workspace = split_room;
        dc.split_workspace_bytes = split_bytes;
        if (int s = gemm(dc, stream)) return s;
    }
    return mean_taken || row_losses != nullptr ? CGPTX_OK : mean_reduce(loss, row_loss, rows, stream);
}

}  // namespace

int cut_cross_entropy(float* row_losses, void* input_gradient, void* classifier_gradient, const void* input, const void* classifier,
                      const std::uint32_t* targets, std::size_t rows, std::size_t hidden, std::size_t vocab, float gradient_scale,
                      int dtype, hipStream_t stream) {
    return run(nullptr, row_losses, input_gradient, classifier_gradient, input, classifier, targets, rows, hidden, vocab, gradient_scale,
               0, dtype, stream);
}

}  // namespace cgptx

extern "C" int cgptx_cut_cross_entropy_forward_backward(float* loss, void* input_gradient, void* classifier_gradient,
                                                        const void* input, const void* classifier,
                                                        const uint32_t* targets, size_t rows, size_t hidden,
                                                        size_t vocab, float gradient_scale,
                                                        int accumulate_classifier, int dtype, cgptx_stream stream) {
    return cgptx::run(loss, nullptr, input_gradient, classifier_gradient, input, classifier, targets, rows, hidden, vocab,
                      gradient_scale, accumulate_classifier, dtype, static_cast<hipStream_t>(stream));
}
