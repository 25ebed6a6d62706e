// fp32 attention on the fp32 matrix cores (attention_f32.hip): the calls of attention.hip whose storage is fp32.
#pragma once

#include "common.hpp"

namespace cgptx {

struct AttentionF32Args {
    const float *q, *k, *v;
    float* out;          // forward: O
    float* lse_out;      // forward, may be null
    const float *dout, *o, *lse;  // backward
    float* delta;        // backward: [batch, query, head], written by the dQ pass and read by the dK/dV pass
    float *dq, *dk, *dv;
    int batch, qs, ks, hq, hkv, d;
    float scale;
    int causal, offset, accumulate;
    int parts;       // dK/dV: workgroups that share a key tile; more than one leave their sums in `partial`,
    float* partial;  // [part][dK | dV][key, kv head, d], for the caller to add up
};

// Whether these kernels take the call: head dimensions in multiples of 4 and 16-byte aligned tensors.
bool attention_f32_takes(std::size_t head_dim, bool aligned);
int attention_f32_forward(const AttentionF32Args& args, hipStream_t stream);
int attention_f32_backward(const AttentionF32Args& args, hipStream_t stream);

}  // namespace cgptx
