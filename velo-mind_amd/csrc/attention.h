// Attention of several query rows per head on the matrix cores
// (attention_mfma.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace vmhip {

// q [batch, heads, rows, head_dim]; k, v [batch, kv_heads, keys, head_dim];
// query head h reads kv head h / (heads / kv_heads).  Output row r of head h
// of batch b starts at o + r * out_row + (b * heads + h) * out_head.
// With `pos` the keys are a cache of `keys` rows whose positions *pos ..
// *pos + rows - 1 are the queries' (keys past them are not read); without,
// the queries are the last `rows` of `keys` positions.  causal: a query sees
// the keys up to its own position.
struct AttentionCall {
    const float* q;
    const float* k;
    const float* v;
    float* o;
    const int32_t* pos = nullptr;
    int rows, batch, heads, kv_heads, head_dim, keys;
    int64_t out_row, out_head;
    float scale;
    bool causal;
};

// Whether attention_mfma() takes a call: head_dim 64 or 128, 16-byte aligned
// operands, a grid within 32 bits.
bool attention_mfma_takes(const AttentionCall& c);
int attention_mfma(const AttentionCall& c, const char* op, hipStream_t stream);

}  // namespace vmhip
