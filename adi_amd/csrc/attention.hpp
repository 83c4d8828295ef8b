// attention.hpp -- the decoder layer for the model-level entry points, and
// the attention of a chunk of tokens (attention_chunk.hip) for the layer.
#pragma once

#include "context.hpp"

namespace adi_hip {

// The full-attention heads, and the rows that parts of a history leave for
// k_attention_combine: acc[256], maximum, denominator.
constexpr uint32_t kQueryHeads = 16;
constexpr uint32_t kKvHeads = 2;
constexpr uint32_t kHeadSize = 256;
constexpr uint32_t kMaxSplits = 64;
constexpr uint32_t kPartialStride = kHeadSize + 2;

// The attention of `count` tokens at position .. position + count - 1 over
// the caches (entries of [2][256], the chunk's own included) on the matrix
// cores: query_gate [count][16][256 query, 256 gate], normalized and rotated.
// With 1 split the gated result goes to attended[count][16][256], else each
// split's part goes to partial[count][16][splits][kPartialStride].
// attention_chunk_takes says for which attentions it is the faster kernel;
// attention_chunk_splits gives the splits that fill the chip with partial
// rows of at most free_bytes.
bool attention_chunk_takes(uint32_t position, uint32_t count);
uint32_t attention_chunk_splits(uint32_t position, uint32_t count, size_t free_bytes);
void launch_attention_chunk(adi_hip_context *ctx, const float *query_gate, const float *keys, const float *values,
                            uint32_t position, uint32_t count, uint32_t splits, float *partial, float *attended);

// One decode token of each of `rows` sequences through one decoder layer on
// hidden[rows][moe.hidden]: row r is at positions[r] of the sequence whose
// state for this layer is states[r] (decode_batch's layer step,
// src/executor.cpp:1620-1811). The kernels read the positions from
// device_positions (the same values); the launches cover positions below
// `span` (0: the largest positions[r] + 1), so a captured step replays
// correctly at any positions below it. `pending` (nullable) holds the
// previous layer's MoE rows, added to hidden first; this layer's MoE rows go
// to moe_out (may be `pending`), left for the next layer's first norm or the
// final norm to add.
void decoder_rows(adi_hip_context *ctx, const adi_hip_decoder_layer *L, uint32_t rows,
                  float *hidden, const float *pending, float *moe_out,
                  const adi_hip_layer_state *const *states, const uint32_t *positions,
                  const uint32_t *device_positions, uint32_t span);

// `count` consecutive tokens of one sequence at positions position ..
// position + count - 1 through one decoder layer (the layer step of prefill,
// src/executor.cpp:1869-2058) on hidden[count][moe.hidden], pending and
// moe_out as decoder_rows'.
void prefill_chunk(adi_hip_context *ctx, const adi_hip_decoder_layer *L, uint32_t position,
                   uint32_t count, float *hidden, const float *pending, float *moe_out,
                   const adi_hip_layer_state *state);

// ---- device helpers of the attention kernels -------------------------------

__device__ __forceinline__ float wave_sum(float v) {
    v += lane_xor<1>(v);
    v += lane_xor<2>(v);
    v += lane_xor<4>(v);
    v += lane_xor<8>(v);
    v += lane_xor<16>(v);
    v += lane_xor<32>(v);
    return v;
}

__device__ __forceinline__ float sigmoid_of(float v) { return 1.0f / (1.0f + expf(-v)); }

// update_online_softmax (src/attention.cpp:15-35) on a lane's four values.
__device__ __forceinline__ void online_step(float score, float4 value, float &maximum,
                                            float &denominator, float4 &acc) {
#pragma clang fp contract(off)
    if (score <= maximum) {
        const float weight = expf(score - maximum);
        denominator += weight;
        acc.x += value.x * weight;
        acc.y += value.y * weight;
        acc.z += value.z * weight;
        acc.w += value.w * weight;
        return;
    }
    const float previous = expf(maximum - score);
    denominator = denominator * previous + 1.0f;
    acc.x = acc.x * previous + value.x;
    acc.y = acc.y * previous + value.y;
    acc.z = acc.z * previous + value.z;
    acc.w = acc.w * previous + value.w;
    maximum = score;
}

}  // namespace adi_hip
