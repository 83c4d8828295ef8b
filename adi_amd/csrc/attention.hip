// attention.hip -- the attention half of a decoder layer on the device, for a
// chunk of consecutive tokens of one sequence (one token when decoding):
//   full_attention_forward   (src/executor.cpp:332-418, src/attention.cpp)
//   linear_attention_forward (src/executor.cpp:420-557, Gated DeltaNet)
// A chunk gives what decoding its tokens one after another gives (token b sees
// the cache up to its own position; the recurrence runs over the chunk in
// order); its projections and MoE run batched.
//
// Full attention, after the q/k/v projections:
//   norm_rope   one block per head: RMS norm with (1 + w), then RoPE on the
//               first 64 dimensions from a cos/sin table the host computes
//               with the same libm calls as the reference (prepare_rope):
//               a kernel argument for one token, a cached device table of
//               every position for a chunk; the key lands in its cache slot,
//               the value is projected there
//   partial     flash-decoding: block (head, split) runs the online softmax
//               over its share of the history, one wave per token stream,
//               and merges its four waves
//   combine     per head: merge the splits, times sigmoid(gate)
//   A long chunk's partial runs on the matrix cores (attention_chunk.hip).
// Linear attention, after the projections:
//   conv        per 128-channel group: the width-4 causal convolution, SiLU,
//               one token's state shift, and the L2 norm of the query and key
//               heads
//   delta       block (value head, 16 rows): the gated delta update of each
//               state row, state read and written once
//   norm_gate   per value head: RMS norm (weight offset 0) times SiLU(gate);
//               after a chunk also the convolution's state shift
// The sums run in a different order from the CPU's (wave and block
// reductions); results agree to float rounding.
#include "attention.hpp"
#include "dense.hpp"
#include "projection.hpp"

#include <algorithm>
#include <cmath>
#include <type_traits>

namespace adi_hip {
namespace {

constexpr uint32_t kQueryStride = 2 * kHeadSize;  // query then gate, per head
constexpr uint32_t kRopeHalf = 32;

constexpr uint32_t kKeyHeads = 16;
constexpr uint32_t kValueHeads = 32;
constexpr uint32_t kLinearHead = 128;
constexpr uint32_t kQkSize = kKeyHeads * kLinearHead;      // 2048
constexpr uint32_t kValueSize = kValueHeads * kLinearHead; // 4096
constexpr uint32_t kChannels = 2 * kQkSize + kValueSize;   // 8192
constexpr uint32_t kDeltaRows = 16;                        // state rows per block

constexpr float kEpsilon = 1.0e-6f;

// Sequences per launch of the per-sequence kernels of a decode step over
// many sequences; their state pointers travel as kernel arguments, their
// positions in a device array (so a captured step replays at new positions).
constexpr uint32_t kRowGroup = 32;

struct FullRows {
    float *keys[kRowGroup];
    float *values[kRowGroup];
};

// The parts of a row's history in a decode step over sequences: a part is a
// block's four waves taking tiles of kTile entries in turn. A row's parts
// follow from its own position and the step's cap alone, so its result does not
// depend on the launch's grid (any grid with at least this many parts gives the
// same bits) or on the other rows. A short history takes one tile a wave, the
// shortest chain; past kShortHistory entries two tiles a wave, which halves the
// parts to write and merge (one row at 600 entries: 15.9 us with one tile, 18.0
// with two; at 4096 26.5 and 23.1; 16 rows at up to 4096 64 and 60).
constexpr uint32_t kTile = 16;
constexpr uint32_t kShortHistory = 1024;
constexpr uint32_t kRowPartials = 1024, kLeastPartials = 64;  // parts of all rows
__host__ __device__ __forceinline__ uint32_t history_parts(uint32_t tokens) {
    const uint32_t entries = tokens <= kShortHistory ? 4u * kTile : 8u * kTile;
    return (tokens + entries - 1u) / entries;
}
struct RowParts {
    uint32_t splits, chunk;  // live parts, entries a part (a multiple of kTile)
};
__host__ __device__ __forceinline__ RowParts row_parts(uint32_t tokens, uint32_t cap) {
    const uint32_t most = history_parts(tokens);
    const uint32_t splits = most > cap ? cap : most;
    const uint32_t chunk = ((tokens + splits - 1u) / splits + kTile - 1u) / kTile * kTile;
    return {(tokens + chunk - 1u) / chunk, chunk};
}
// The most parts of a history of 1 .. last entries.
inline uint32_t most_parts(uint32_t last, uint32_t cap) {
    return std::min(cap, std::max(history_parts(last), history_parts(std::min(last, kShortHistory))));
}

// Blocks of k_attention_partial (block b runs on XCD b % 8).
// Under kPairSplits splits block b is query head b % 16 of split b / 16: all
// splits of a head on one XCD, whose L2 then still holds them for the
// combine. From kPairSplits splits the history is long and the eight query
// heads of a KV head, which read the same cache entries, are dealt to one
// XCD instead, so the entries pass through that XCD's L2 once rather than
// once per XCD: block b (k = b / 8) takes pair g = 8 (k / 8) + b % 8,
// g = kKvHeads split + kv, and query head 8 kv + k % 8; the grid of
// partial_blocks(splits) covers every pair, and blocks of pairs past the
// last split return at once.
static_assert(kQueryHeads == 8 * kKvHeads, "eight query heads to a KV head");
constexpr uint32_t kPairSplits = 32;
__host__ __device__ __forceinline__ uint32_t partial_blocks(uint32_t splits) {
    return splits < kPairSplits ? kQueryHeads * splits : (kKvHeads * splits + 7u) / 8u * 64u;
}
struct PartialBlock {
    uint32_t head, split;
    bool live;
};
__device__ __forceinline__ PartialBlock partial_block(uint32_t b, uint32_t splits) {
    if (splits < kPairSplits) {
        return {b % kQueryHeads, b / kQueryHeads, true};
    }
    const uint32_t k = b >> 3;
    const uint32_t g = ((k >> 3) << 3) | (b & 7u);
    const uint32_t kv = g % kKvHeads;
    return {kv * 8u + (k & 7u), g / kKvHeads, g < kKvHeads * splits};
}

struct LinearRows {
    float *convolution[kRowGroup];
    float *recurrent[kRowGroup];
};

struct RopeTable {
    float cosine[kRopeHalf];
    float sine[kRopeHalf];
};

// MachModel's RoPE divisors (src/model.cpp:606-615), computed on the host.
struct RopeDivisors {
    float divisor[kRopeHalf];
};

// Sum over the block (blockDim.x a multiple of 64, at most 1024); every
// thread receives it. `partial` holds 16 floats.
__device__ __forceinline__ float block_sum(float v, float *partial) {
    v = wave_sum(v);
    const uint32_t waves = blockDim.x >> 6;
    if ((threadIdx.x & 63u) == 0) {
        partial[threadIdx.x >> 6] = v;
    }
    __syncthreads();
    float total = 0.0f;
    for (uint32_t w = 0; w < waves; ++w) {
        total += partial[w];
    }
    __syncthreads();
    return total;
}

__device__ __forceinline__ float silu_of(float v) { return v / (1.0f + expf(-v)); }

// normalize_head then apply_rope (src/executor.cpp:25-41, 60-72, 376-390)
// of one 256-value head by a block of kHeadSize threads: RMS norm with
// (1 + w), then thread t < 32 rotates the pair (t, t + 32) by its cosine and
// sine. src and dst may be the same.
__device__ __forceinline__ void norm_rope_head(const float *src, float *dst, const uint16_t *w,
                                               float cosine, float sine, float *partial,
                                               float *head) {
#pragma clang fp contract(off)
    const uint32_t t = threadIdx.x;
    float x = src[t];
    const float squares = block_sum(x * x, partial);
    const float scale = 1.0f / sqrtf(squares / static_cast<float>(kHeadSize) + kEpsilon);
    x *= scale * (1.0f + bf16_bits_to_float(w[t]));
    head[t] = x;
    __syncthreads();
    if (t < kRopeHalf) {
        const float first = head[t], second = head[t + kRopeHalf];
        dst[t] = first * cosine - second * sine;
        dst[t + kRopeHalf] = second * cosine + first * sine;
    } else if (t >= 2 * kRopeHalf) {
        dst[t] = x;
    }
}

// Block (h, b) of token b of a chunk: h 0-15 the query heads (stride 512),
// 16-17 the new key heads, in place. One token takes the host's table `rope`;
// in a chunk, token b reads the host-computed table of position + b from
// `rope_rows` ([position][32 cosines, 32 sines]), so every token of a chunk
// rotates exactly as it would alone (the reference builds its prefill table
// on the host too, src/executor.cpp:1853-1866).
__global__ __launch_bounds__(kHeadSize) void k_norm_rope(float *query_gate, float *key,
                                                         const uint16_t *query_norm,
                                                         const uint16_t *key_norm, RopeTable rope,
                                                         const float *rope_rows, uint32_t position) {
    __shared__ float partial[16];
    __shared__ float head[kHeadSize];
    const uint32_t h = blockIdx.x, b = blockIdx.y, t = threadIdx.x;
    query_gate += static_cast<size_t>(b) * kQueryHeads * kQueryStride;
    key += static_cast<size_t>(b) * kKvHeads * kHeadSize;
    float *v = h < kQueryHeads ? query_gate + static_cast<size_t>(h) * kQueryStride
                               : key + static_cast<size_t>(h - kQueryHeads) * kHeadSize;
    float cosine = 0.0f, sine = 0.0f;
    if (t < kRopeHalf) {
        cosine = rope.cosine[t];
        sine = rope.sine[t];
        if (rope_rows != nullptr) {
            const float *row = rope_rows + static_cast<size_t>(position + b) * (2 * kRopeHalf);
            cosine = row[t];
            sine = row[kRopeHalf + t];
        }
    }
    norm_rope_head(v, v, h < kQueryHeads ? query_norm : key_norm, cosine, sine, partial, head);
}

// The same for one decode token of each of up to kRowGroup sequences: block
// (h, r), h 0-15 the query heads of row r (in place), 16-17 its key heads,
// normalized and rotated into the sequence's cache entry positions[r], and
// 18-19 its value heads, copied into that entry. The RoPE table row is the
// row's position.
__global__ __launch_bounds__(kHeadSize) void k_norm_rope_rows(float *query_gate, const float *key,
                                                              const float *value,
                                                              const uint16_t *query_norm,
                                                              const uint16_t *key_norm,
                                                              const float *rope_rows, FullRows rows,
                                                              const uint32_t *positions) {
    __shared__ float partial[16];
    __shared__ float head[kHeadSize];
    const uint32_t h = blockIdx.x, r = blockIdx.y, t = threadIdx.x;
    const uint32_t position = positions[r];
    const size_t entry = static_cast<size_t>(position) * kKvHeads * kHeadSize;
    if (h >= kQueryHeads + kKvHeads) {  // uniform over the block
        const uint32_t kv = h - kQueryHeads - kKvHeads;
        rows.values[r][entry + kv * kHeadSize + t] =
            value[(static_cast<size_t>(r) * kKvHeads + kv) * kHeadSize + t];
        return;
    }
    float cosine = 0.0f, sine = 0.0f;
    if (t < kRopeHalf) {
        const float *row = rope_rows + static_cast<size_t>(position) * (2 * kRopeHalf);
        cosine = row[t];
        sine = row[kRopeHalf + t];
    }
    if (h < kQueryHeads) {
        float *q = query_gate + static_cast<size_t>(r) * kQueryHeads * kQueryStride +
                   static_cast<size_t>(h) * kQueryStride;
        norm_rope_head(q, q, query_norm, cosine, sine, partial, head);
    } else {
        const uint32_t kv = h - kQueryHeads;
        norm_rope_head(key + (static_cast<size_t>(r) * kKvHeads + kv) * kHeadSize,
                       rows.keys[r] + entry + kv * kHeadSize, key_norm, cosine, sine, partial,
                       head);
    }
}

// Block (query head, split) of one token's query row: cache entries
// [split * chunk, ...) below `tokens` of the head's KV stream, wave w taking
// every fourth. Lane l holds dimensions 4l..4l+3. Writes the split's
// accumulator, maximum and denominator to the token's partial rows
// (maximum -inf and denominator 0 when the split lies past the token).
// With COHERENT the partial row is written through to memory (a later block
// of the same launch reads it). The query head is at `query` (global or LDS).
template <bool COHERENT = false>
__device__ __forceinline__ void attention_partial_span(const float *query, const float *keys,
                                                       const float *values, uint32_t tokens,
                                                       uint32_t chunk, float *partial, uint32_t h,
                                                       uint32_t split, uint32_t splits) {
#pragma clang fp contract(off)
    __shared__ __align__(16) float wave_acc[4][kHeadSize];
    __shared__ float wave_max[4], wave_den[4];
    const uint32_t kv = h / (kQueryHeads / kKvHeads);
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    const float4 q = reinterpret_cast<const float4 *>(query)[lane];
    const float score_scale = 1.0f / 16.0f;  // 1 / sqrt(256)
    const uint32_t begin = split * chunk;
    const uint32_t end = begin + chunk < tokens ? begin + chunk : tokens;
    float maximum = -__builtin_huge_valf(), denominator = 0.0f;
    float4 acc = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    // the wave's tokens t0, t0 + 4, ... in batches of eight: the batch's
    // entries are loaded together (a token past the span reloads t0, unused),
    // its dot products reduced together, then the online updates in order
    constexpr uint32_t kBatch = 8;
    for (uint32_t t0 = begin + wave; t0 < end; t0 += 4u * kBatch) {
        // no branch around a load, so that the batch's loads are counted and
        // waited for once
        float4 k[kBatch], v[kBatch];
#pragma unroll
        for (uint32_t j = 0; j < kBatch; ++j) {
            const uint32_t t = t0 + 4u * j < end ? t0 + 4u * j : t0;
            const size_t at = (static_cast<size_t>(t) * kKvHeads + kv) * kHeadSize;
            k[j] = reinterpret_cast<const float4 *>(keys + at)[lane];
            v[j] = reinterpret_cast<const float4 *>(values + at)[lane];
        }
        float dot[kBatch];
#pragma unroll
        for (uint32_t j = 0; j < kBatch; ++j) {
            dot[j] = wave_sum(((q.x * k[j].x + q.y * k[j].y) + q.z * k[j].z) + q.w * k[j].w);
        }
#pragma unroll
        for (uint32_t j = 0; j < kBatch; ++j) {
            if (t0 + 4u * j < end) {
                online_step(dot[j] * score_scale, v[j], maximum, denominator, acc);
            }
        }
    }
    reinterpret_cast<float4 *>(wave_acc[wave])[lane] = acc;
    if (lane == 0) {
        wave_max[wave] = maximum;
        wave_den[wave] = denominator;
    }
    __syncthreads();
    float m = wave_max[0];
    for (uint32_t w = 1; w < 4; ++w) {
        m = fmaxf(m, wave_max[w]);
    }
    float a = 0.0f, d = 0.0f;
    if (m != -__builtin_huge_valf()) {  // else no token in this split
        for (uint32_t w = 0; w < 4; ++w) {
            const float f = expf(wave_max[w] - m);  // 0 for a wave without tokens
            a += wave_acc[w][threadIdx.x] * f;
            d += wave_den[w] * f;
        }
    }
    float *out = partial + (static_cast<size_t>(h) * splits + split) * kPartialStride;
    if constexpr (COHERENT) {
        coherent_store(out + threadIdx.x, a);
        if (threadIdx.x == 0) {
            coherent_store(out + kHeadSize, m);
            coherent_store(out + kHeadSize + 1, d);
        }
    } else {
        out[threadIdx.x] = a;
        if (threadIdx.x == 0) {
            out[kHeadSize] = m;
            out[kHeadSize + 1] = d;
        }
    }
}

// Token b of a chunk at `position` sees entries 0 .. position + b.
__global__ __launch_bounds__(256) void k_attention_partial(const float *query_gate,
                                                           const float *keys, const float *values,
                                                           uint32_t position, uint32_t chunk,
                                                           uint32_t splits, float *partial) {
    const PartialBlock pb = partial_block(blockIdx.x, splits);
    if (!pb.live) {
        return;
    }
    const uint32_t b = blockIdx.z;
    attention_partial_span(query_gate + static_cast<size_t>(b) * kQueryHeads * kQueryStride +
                               static_cast<size_t>(pb.head) * kQueryStride,
                           keys,
                           values, position + b + 1, chunk,
                           partial + static_cast<size_t>(b) * kQueryHeads * splits * kPartialStride, pb.head,
                           pb.split, splits);
}

typedef float f32x4 __attribute__((ext_vector_type(4)));
constexpr uint32_t kHeadsPerKv = kQueryHeads / kKvHeads;  // 8
constexpr uint32_t kQueryPad = kHeadSize + 16;  // LDS rows whose 16-byte pieces fall on different banks
constexpr uint32_t kMergePad = kHeadSize + 4;

struct RowsLds {
    __align__(16) float query[kHeadsPerKv][kQueryPad];
    __align__(16) float acc[4][kHeadsPerKv][kMergePad];
    float maximum[4][kHeadsPerKv], denominator[4][kHeadsPerKv];
    float factor[kHeadsPerKv][4], top[kHeadsPerKv];
    uint32_t odd;
};

// Entries [split * chunk, ...) below `tokens` of KV head `kv` for its eight
// query heads (lds.query) by a block of four waves, wave w taking every fourth
// tile of kTile entries, and the split's part of each head to partial (written
// through to memory with COHERENT: a later block of the same launch reads it).
// With `attended` (a row of one part) each head's output, times its sigmoid
// gate at query_gate, goes there instead, unless a score is infinite.
// Returns whether it went to partial.
//
// A tile is two chains of v_mfma_f32_16x16x4_f32 in which a lane's registers
// are loaded as the matrix core reads them, straight from the cache: the
// scores are keys (16 entries a column of A, dimensions 16 j + 4 g + i at step
// (j, i) of lane group g) times queries (B, the eight heads twice), and their
// result, entry 4 g + r of head l % 16 in register r, is B of the second
// chain's step r as it stands; its A is the values transposed (dimension
// 64 m + 4 (l % 16) + i of entry 4 g + r). So a head's maximum, factors and
// weights live in the lanes of its column, one exponential serves one score,
// and an entry is read once for the eight heads.
//
// Bound by the entries' bytes where rows and histories are many, by a part's
// chain of norm, tile and merge where they are few. One head's wave at a time
// over float registers (a wave sum and an exponential a head and entry, each
// entry read eight times) took 201 us for 32 rows at up to 2,000 entries, this
// 62 (131 MB: 2.1 TB/s); one row at 40, 200, 400 and 2,000 entries 10.8, 11.5,
// 13.6, 27.6 and 10.1, 14.4, 14.4, 19.7 (a row of one part without the round
// trip through memory, 12.8 with it; every thread taking the waves' factors of
// every head itself cost 1.7 more).
template <bool COHERENT>
__device__ __forceinline__ bool attention_rows_span(RowsLds &lds, const float *keys, const float *values,
                                                    uint32_t tokens, uint32_t chunk, float *partial, uint32_t kv,
                                                    uint32_t split, uint32_t splits, const float *query_gate = nullptr,
                                                    float *attended = nullptr) {
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    const uint32_t c = lane & 15u, g = lane >> 4;
    const uint32_t begin = split * chunk;
    const uint32_t end = begin + chunk < tokens ? begin + chunk : tokens;
    const float *key_head = keys + static_cast<size_t>(kv) * kHeadSize;
    const float *value_head = values + static_cast<size_t>(kv) * kHeadSize;
    constexpr size_t kEntry = kKvHeads * kHeadSize;
    const float *query = lds.query[c & 7u] + 4u * g;
    f32x4 k[16], v[16], o[16];
    // entries past the part read its last one; their scores are masked
    const auto load_keys = [&](uint32_t t0) {
        const uint32_t t = t0 + c < end ? t0 + c : end - 1u;
        const float *at = key_head + t * kEntry + 4u * g;
#pragma unroll
        for (uint32_t j = 0; j < 16; ++j) {
            k[j] = *reinterpret_cast<const f32x4 *>(at + 16u * j);
        }
    };
    const auto load_values = [&](uint32_t t0) {
#pragma unroll
        for (uint32_t r = 0; r < 4; ++r) {
            const uint32_t e = t0 + 4u * g + r;
            const float *at = value_head + (e < end ? e : end - 1u) * kEntry + 4u * c;
#pragma unroll
            for (uint32_t m = 0; m < 4; ++m) {
                v[4u * r + m] = *reinterpret_cast<const f32x4 *>(at + 64u * m);
            }
        }
    };
#pragma unroll
    for (uint32_t i = 0; i < 16; ++i) {
        o[i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    }
    float maximum = -__builtin_huge_valf(), denominator = 0.0f;
    bool odd = false;
    uint32_t t0 = begin + wave * kTile;
    if (t0 < end) {
        load_keys(t0);
        load_values(t0);
    }
    for (; t0 < end; t0 += 4u * kTile) {
        const bool ragged = t0 + kTile >= tokens;  // the row's last tile
        f32x4 s[4];
#pragma unroll
        for (uint32_t i = 0; i < 4; ++i) {
            s[i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        }
#pragma unroll
        for (uint32_t j = 0; j < 16; ++j) {
            const f32x4 q = *reinterpret_cast<const f32x4 *>(query + 16u * j);
#pragma unroll
            for (uint32_t i = 0; i < 4; ++i) {
                s[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(k[j][i], q[i], s[i], 0, 0, 0);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        if (t0 + 4u * kTile < end) {
            load_keys(t0 + 4u * kTile);
        }
        f32x4 p = ((s[0] + s[1]) + (s[2] + s[3])) * (1.0f / 16.0f);  // 1 / sqrt(256)
#pragma unroll
        for (uint32_t r = 0; r < 4; ++r) {
            odd |= fabsf(p[r]) == __builtin_huge_valf();
        }
        if (ragged) {
#pragma unroll
            for (uint32_t r = 0; r < 4; ++r) {
                const uint32_t e = t0 + 4u * g + r;
                p[r] = e < tokens ? p[r] : -__builtin_huge_valf();
#pragma unroll
                for (uint32_t m = 0; m < 4; ++m) {
                    v[4u * r + m] = e < tokens ? v[4u * r + m] : f32x4{0.0f, 0.0f, 0.0f, 0.0f};
                }
            }
        }
        float top = fmaxf(fmaxf(p[0], p[1]), fmaxf(p[2], p[3]));
        top = fmaxf(top, lane_xor<16>(top));
        top = fmaxf(top, lane_xor<32>(top));
        if (__any(top > maximum)) {
            const float next = fmaxf(top, maximum);
            const float factor = expf(maximum - next);
            maximum = next;
            denominator *= factor;
#pragma unroll
            for (uint32_t i = 0; i < 16; ++i) {
                o[i] *= factor;
            }
        }
#pragma unroll
        for (uint32_t r = 0; r < 4; ++r) {
            p[r] = expf(p[r] - maximum);
        }
        denominator += (p[0] + p[1]) + (p[2] + p[3]);
#pragma unroll
        for (uint32_t r = 0; r < 4; ++r) {
#pragma unroll
            for (uint32_t m = 0; m < 4; ++m) {
#pragma unroll
                for (uint32_t i = 0; i < 4; ++i) {
                    o[4u * m + i] =
                        __builtin_amdgcn_mfma_f32_16x16x4f32(v[4u * r + m][i], p[r], o[4u * m + i], 0, 0, 0);
                }
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        if (t0 + 4u * kTile < end) {
            load_values(t0 + 4u * kTile);
        }
    }
    denominator += lane_xor<16>(denominator);
    denominator += lane_xor<32>(denominator);
    if (threadIdx.x == 0) {
        lds.odd = 0u;
    }
    __syncthreads();
    if (__any(odd) && lane == 0) {
        lds.odd = 1u;
    }
    if (c < kHeadsPerKv) {
#pragma unroll
        for (uint32_t m = 0; m < 4; ++m) {
#pragma unroll
            for (uint32_t r = 0; r < 4; ++r) {
                *reinterpret_cast<f32x4 *>(&lds.acc[wave][c][64u * m + 16u * g + 4u * r]) =
                    f32x4{o[4u * m][r], o[4u * m + 1u][r], o[4u * m + 2u][r], o[4u * m + 3u][r]};
            }
        }
        if (g == 0u) {
            lds.maximum[wave][c] = maximum;
            lds.denominator[wave][c] = denominator;
        }
    }
    __syncthreads();
    // uniform: an infinite score, whose row goes entry by entry, head by head.
    // (One that is a NaN stays: it leaves NaNs in its head's denominator and
    // accumulator whatever the factors are, as it does entry by entry.)
    if (lds.odd != 0u) {
        for (uint32_t h = 0; h < kHeadsPerKv; ++h) {
            attention_partial_span<COHERENT>(lds.query[h], keys, values, tokens, chunk, partial,
                                             kv * kHeadsPerKv + h, split, splits);
            __syncthreads();
        }
        return true;
    }
    // each wave's factor of each head by one thread, not by all
    if (threadIdx.x < 4u * kHeadsPerKv) {
        const uint32_t h = threadIdx.x % kHeadsPerKv, w = threadIdx.x / kHeadsPerKv;
        const float m = fmaxf(fmaxf(lds.maximum[0][h], lds.maximum[1][h]), fmaxf(lds.maximum[2][h], lds.maximum[3][h]));
        // 0 for a wave without tokens, and where no wave has any
        lds.factor[h][w] = m != -__builtin_huge_valf() ? expf(lds.maximum[w][h] - m) : 0.0f;
        lds.top[h] = m;
    }
    __syncthreads();
    const auto merged = [&](uint32_t h, float &a, float &d) {
        a = 0.0f;
        d = 0.0f;
#pragma unroll
        for (uint32_t w = 0; w < 4; ++w) {
            a += lds.acc[w][h][threadIdx.x] * lds.factor[h][w];
            d += lds.denominator[w][h] * lds.factor[h][w];
        }
    };
    if (attended != nullptr) {  // uniform; the combine of one part
        float gate[kHeadsPerKv];
#pragma unroll
        for (uint32_t h = 0; h < kHeadsPerKv; ++h) {
            gate[h] = query_gate[h * kQueryStride + kHeadSize + threadIdx.x];
        }
#pragma unroll
        for (uint32_t h = 0; h < kHeadsPerKv; ++h) {
            float a, d;
            merged(h, a, d);
            attended[h * kHeadSize + threadIdx.x] = a * (1.0f / d) * sigmoid_of(gate[h]);
        }
        return false;
    }
#pragma unroll
    for (uint32_t h = 0; h < kHeadsPerKv; ++h) {
        const float m = lds.top[h];
        float a, d;
        merged(h, a, d);
        float *out = partial + (static_cast<size_t>(kv * kHeadsPerKv + h) * splits + split) * kPartialStride;
        if constexpr (COHERENT) {
            coherent_store(out + threadIdx.x, a);
            if (threadIdx.x == 0) {
                coherent_store(out + kHeadSize, m);
                coherent_store(out + kHeadSize + 1, d);
            }
        } else {
            out[threadIdx.x] = a;
            if (threadIdx.x == 0) {
                out[kHeadSize] = m;
                out[kHeadSize + 1] = d;
            }
        }
    }
    return true;
}

// Row r of a decode step over sequences sees its own cache's entries
// 0 .. positions[r] in row_parts' parts: block (KV head, split, r). The grid's
// further splits lie past the row's tokens and come out empty (skipped by the
// combine).
__global__ __launch_bounds__(256, 2) void k_attention_partial_rows(const float *query_gate, FullRows rows,
                                                                   const uint32_t *positions, uint32_t cap,
                                                                   uint32_t grid_splits, float *partial) {
    __shared__ RowsLds lds;
    const uint32_t kv = blockIdx.x % kKvHeads, split = blockIdx.x / kKvHeads, r = blockIdx.z;
    const uint32_t tokens = positions[r] + 1;
    const RowParts parts = row_parts(tokens, cap);
    for (uint32_t h = 0; h < kHeadsPerKv; ++h) {
        lds.query[h][threadIdx.x] =
            query_gate[(static_cast<size_t>(r) * kQueryHeads + kv * kHeadsPerKv + h) * kQueryStride + threadIdx.x];
    }
    __syncthreads();
    attention_rows_span<false>(lds, rows.keys[r], rows.values[r], tokens, parts.chunk,
                               partial + static_cast<size_t>(r) * kQueryHeads * grid_splits * kPartialStride, kv,
                               split, grid_splits);
}
// The splits of one query head merged (splits <= N): every split's
// accumulator, then the splits' maxima and denominators (through LDS),
// loaded in one round, then the accumulators added in split order.
template <uint32_t N>
__device__ __forceinline__ void combine_splits(const float *p, uint32_t splits, uint32_t t, float *split_max,
                                               float *split_den, float *split_factor, float &a, float &d) {
#pragma clang fp contract(off)
    float acc[N];
#pragma unroll
    for (uint32_t s = 0; s < N; ++s) {
        acc[s] = s < splits ? p[s * kPartialStride + t] : 0.0f;
    }
    static_assert(N <= kHeadSize, "a thread's split");
    // both words of the thread's split loaded before either is stored (one
    // round trip with the accumulators')
    if (t < splits) {
        const float mx = p[t * kPartialStride + kHeadSize];
        const float dn = p[t * kPartialStride + kHeadSize + 1];
        split_max[t] = mx;
        split_den[t] = dn;
    }
    __syncthreads();
    // split 0 always holds token 0, so the maximum is finite
    float m = split_max[0];
    for (uint32_t s = 1; s < splits; ++s) {
        m = fmaxf(m, split_max[s]);
    }
    for (uint32_t s = t; s < splits; s += kHeadSize) {
        split_factor[s] = expf(split_max[s] - m);
    }
    __syncthreads();
    a = 0.0f;
    d = 0.0f;
#pragma unroll
    for (uint32_t s = 0; s < N; ++s) {
        const float den = s < splits ? split_den[s] : 0.0f;
        if (den == 0.0f) {
            continue;  // a split past the token (or past the splits)
        }
        const float f = split_factor[s];
        a += acc[s] * f;
        d += den * f;
    }
}

// Per query head: the splits merged, divided by the denominator, times the
// head's sigmoid gate (src/executor.cpp:403-411).
__global__ __launch_bounds__(kHeadSize) void k_attention_combine(const float *partial,
                                                                 uint32_t splits,
                                                                 const float *query_gate,
                                                                 float *attended) {
#pragma clang fp contract(off)
    const uint32_t h = blockIdx.x, t = threadIdx.x, b = blockIdx.y;
    query_gate += static_cast<size_t>(b) * kQueryHeads * kQueryStride;
    attended += static_cast<size_t>(b) * kQueryHeads * kHeadSize;
    __shared__ float split_max[kMaxSplits], split_den[kMaxSplits], split_factor[kMaxSplits];
    const float *p = partial + (static_cast<size_t>(b) * kQueryHeads + h) * splits * kPartialStride;
    const float gate = query_gate[static_cast<size_t>(h) * kQueryStride + kHeadSize + t];
    float a, d;
    if (splits <= 16u) {
        combine_splits<16>(p, splits, t, split_max, split_den, split_factor, a, d);
    } else {
        combine_splits<kMaxSplits>(p, splits, t, split_max, split_den, split_factor, a, d);
    }
    attended[static_cast<size_t>(h) * kHeadSize + t] = a * (1.0f / d) * sigmoid_of(gate);
}

// norm_rope_head by one wave, the same sums: lane l holds dimensions l, l + 64,
// l + 128, l + 192; row holds the position's 32 cosines and 32 sines.
__device__ __forceinline__ void norm_rope_wave(const float *src, float *dst, const uint16_t *w, const float *row) {
#pragma clang fp contract(off)
    const uint32_t lane = threadIdx.x & 63u;
    float x[4], weight[4];
#pragma unroll
    for (uint32_t i = 0; i < 4; ++i) {
        x[i] = src[64u * i + lane];
        weight[i] = bf16_bits_to_float(w[64u * i + lane]);
    }
    const float cosine = row[lane & 31u], sine = row[kRopeHalf + (lane & 31u)];
    float squares = 0.0f;
#pragma unroll
    for (uint32_t i = 0; i < 4; ++i) {
        squares += wave_sum(x[i] * x[i]);
    }
    const float scale = 1.0f / sqrtf(squares / static_cast<float>(kHeadSize) + kEpsilon);
#pragma unroll
    for (uint32_t i = 0; i < 4; ++i) {
        x[i] *= scale * (1.0f + weight[i]);
    }
    const float other = lane_xor<32>(x[0]);
    x[0] = lane < kRopeHalf ? x[0] * cosine - other * sine : x[0] * cosine + other * sine;
#pragma unroll
    for (uint32_t i = 0; i < 4; ++i) {
        dst[64u * i + lane] = x[i];
    }
}

// One decode token of each of up to kRowGroup sequences through full
// attention's core in one launch, with the arithmetic of k_norm_rope_rows,
// k_attention_partial_rows and k_attention_combine. Block (KV head, split,
// sequence r):
// - normalizes and rotates its eight query heads into LDS itself (every split
//   does);
// - the split holding the row's new entry (position) normalizes and rotates its
//   key and writes it and the value into the cache: no other block reads that
//   entry;
// - writes its split's partial rows through to memory; the last block of the
//   row's live splits through the KV head's ticket merges the eight heads and
//   applies the sigmoid gates.
// Blocks of splits past the row's history leave at once. `tickets` holds
// kQueryHeads words a sequence (one a KV head used), zero between calls.
__global__ __launch_bounds__(256, 2) void k_attention_rows_one(const float *query_gate, const float *key,
                                                               const float *value, const uint16_t *query_norm,
                                                               const uint16_t *key_norm, const float *rope_rows,
                                                               FullRows rows, const uint32_t *positions, uint32_t cap,
                                                               uint32_t grid_splits, float *partial, float *attended, uint32_t *tickets) {
#pragma clang fp contract(off)
    __shared__ RowsLds lds;
    __shared__ uint32_t last;
    const uint32_t kv = blockIdx.x % kKvHeads, split = blockIdx.x / kKvHeads, r = blockIdx.z;
    const uint32_t t = threadIdx.x, lane = t & 63u, wave = t >> 6;
    const uint32_t position = positions[r];
    const uint32_t tokens = position + 1u;
    const RowParts parts = row_parts(tokens, cap);
    if (split >= parts.splits) {  // uniform over the block
        return;
    }
    const float *rope = rope_rows + static_cast<size_t>(position) * (2 * kRopeHalf);
    const size_t head = static_cast<size_t>(r) * kQueryHeads + kv * kHeadsPerKv;
#pragma unroll
    for (uint32_t i = 0; i < 2; ++i) {
        const uint32_t h = 2u * wave + i;
        norm_rope_wave(query_gate + (head + h) * kQueryStride, lds.query[h], query_norm, rope);
    }
    if (split == parts.splits - 1u) {  // uniform over the block
        // (ahead of the queries, which its way to memory then overlaps)
        const size_t src = (static_cast<size_t>(r) * kKvHeads + kv) * kHeadSize;
        const size_t entry = (static_cast<size_t>(position) * kKvHeads + kv) * kHeadSize;
        rows.values[r][entry + t] = value[src + t];
        if (wave == 0u) {
            norm_rope_wave(key + src, rows.keys[r] + entry, key_norm, rope);
        }
    }
    __syncthreads();  // the block reads back its own entry
    float *p = partial + static_cast<size_t>(r) * kQueryHeads * grid_splits * kPartialStride;
    const bool one = parts.splits == 1u;
    if (!attention_rows_span<true>(lds, rows.keys[r], rows.values[r], tokens, parts.chunk, p, kv, split, grid_splits,
                                   query_gate + head * kQueryStride, one ? attended + head * kHeadSize : nullptr)) {
        return;
    }
    wait_stores();
    __syncthreads();
    uint32_t *ticket = tickets + static_cast<size_t>(r) * kQueryHeads + kv;
    if (t == 0) {
        last = coherent_add(ticket, 1u) + 1u == parts.splits ? 1u : 0u;
    }
    __syncthreads();
    if (last == 0u) {
        return;
    }
    // k_attention_combine's sums, two heads a wave: lane s holds split s's
    // maximum and denominator, lane l dimensions l + 64 i
    static_assert(kMaxSplits <= 64, "a lane a split");
#pragma unroll
    for (uint32_t i = 0; i < 2; ++i) {
        const uint32_t h = 2u * wave + i;
        const float *ph = p + static_cast<size_t>(kv * kHeadsPerKv + h) * grid_splits * kPartialStride;
        float mx = -__builtin_huge_valf(), den = 0.0f;
        if (lane < parts.splits) {
            mx = coherent_load(ph + lane * kPartialStride + kHeadSize);
            den = coherent_load(ph + lane * kPartialStride + kHeadSize + 1);
        }
        float gate[4];
#pragma unroll
        for (uint32_t j = 0; j < 4; ++j) {
            gate[j] = query_gate[(head + h) * kQueryStride + kHeadSize + 64u * j + lane];
        }
        float m = mx;
        m = fmaxf(m, lane_xor<1>(m));
        m = fmaxf(m, lane_xor<2>(m));
        m = fmaxf(m, lane_xor<4>(m));
        m = fmaxf(m, lane_xor<8>(m));
        m = fmaxf(m, lane_xor<16>(m));
        m = fmaxf(m, lane_xor<32>(m));
        const float factor = expf(mx - m);
        float a[4] = {0.0f, 0.0f, 0.0f, 0.0f}, d = 0.0f;
        constexpr uint32_t kBatch = 8;
        for (uint32_t s0 = 0; s0 < parts.splits; s0 += kBatch) {
            float acc[kBatch][4];
#pragma unroll
            for (uint32_t s = 0; s < kBatch; ++s) {
                const uint32_t at = s0 + s < parts.splits ? s0 + s : parts.splits - 1u;
#pragma unroll
                for (uint32_t j = 0; j < 4; ++j) {
                    acc[s][j] = coherent_load(ph + at * kPartialStride + 64u * j + lane);
                }
            }
#pragma unroll
            for (uint32_t s = 0; s < kBatch; ++s) {
                const int at = static_cast<int>(s0 + s);
                const float ds = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(den), at & 63));
                const float fs = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(factor), at & 63));
                if (s0 + s < parts.splits && ds != 0.0f) {  // uniform
#pragma unroll
                    for (uint32_t j = 0; j < 4; ++j) {
                        a[j] += acc[s][j] * fs;
                    }
                    d += ds * fs;
                }
            }
        }
#pragma unroll
        for (uint32_t j = 0; j < 4; ++j) {
            attended[(head + h) * kHeadSize + 64u * j + lane] = a[j] * (1.0f / d) * sigmoid_of(gate[j]);
        }
    }
    if (t == 0) {
        coherent_store(ticket, 0u);
    }
}

// The causal convolution of 128 channels for token b of a chunk
// (src/executor.cpp:480-496) and, for the query and key groups (blocks
// 0-31), their L2 norm (497-505). The three inputs before token b are the
// chunk's earlier qkv rows or, before the chunk, the state. With `shift` (one
// token) the state shifts here; for a chunk k_linear_norm_gate
// does it, after every token has read it.
__device__ __forceinline__ void linear_conv_token(const float *qkv, const uint16_t *weights,
                                                  float *state, float *convolved, uint32_t b,
                                                  bool shift) {
#pragma clang fp contract(off)
    __shared__ float partial[16];
    const uint32_t c = blockIdx.x * kLinearHead + threadIdx.x;
    float *history = state + static_cast<size_t>(c) * 3u;
    const uint2 packed = *reinterpret_cast<const uint2 *>(weights + static_cast<size_t>(c) * 4u);
    const float w0 = bf16_bits_to_float(packed.x & 0xFFFFu), w1 = bf16_bits_to_float(packed.x >> 16);
    const float w2 = bf16_bits_to_float(packed.y & 0xFFFFu), w3 = bf16_bits_to_float(packed.y >> 16);
    // input at relative time b - 3 + i: row b - 3 + i, or state slot b + i
    float earlier[3];
#pragma unroll
    for (uint32_t i = 0; i < 3; ++i) {
        earlier[i] = b + i >= 3 ? qkv[static_cast<size_t>(b + i - 3) * kChannels + c] : history[b + i];
    }
    const float h0 = earlier[0], h1 = earlier[1], h2 = earlier[2];
    const float x = qkv[static_cast<size_t>(b) * kChannels + c];
    float v = 0.0f;
    v += h0 * w0;
    v += h1 * w1;
    v += h2 * w2;
    v += x * w3;
    float y = silu_of(v);
    if (shift) {
        history[0] = h1;
        history[1] = h2;
        history[2] = x;
    }
    if (blockIdx.x < 2u * kKeyHeads) {  // uniform over the block
        const float squares = block_sum(y * y, partial);
        y *= 1.0f / sqrtf(squares + kEpsilon);
    }
    convolved[static_cast<size_t>(b) * kChannels + c] = y;
}

__global__ __launch_bounds__(kLinearHead) void k_linear_conv(const float *qkv,
                                                             const uint16_t *weights,
                                                             float *state, float *convolved) {
    linear_conv_token(qkv, weights, state, convolved, blockIdx.y, gridDim.y == 1);
}

// One decode token of each of up to kRowGroup sequences: row r convolves
// with its own state, which shifts.
__global__ __launch_bounds__(kLinearHead) void k_linear_conv_rows(const float *qkv,
                                                                  const uint16_t *weights,
                                                                  LinearRows rows,
                                                                  float *convolved) {
    const uint32_t r = blockIdx.y;
    linear_conv_token(qkv + static_cast<size_t>(r) * kChannels, weights, rows.convolution[r],
                      convolved + static_cast<size_t>(r) * kChannels, 0, true);
}

// The convolution state of channel c after a chunk of `count` tokens: the last
// three of (state, qkv rows).
__device__ __forceinline__ void shift_history(const float *qkv, uint32_t count, float *state, uint32_t c) {
    float *history = state + static_cast<size_t>(c) * 3u;
    float next[3];
#pragma unroll
    for (uint32_t i = 0; i < 3; ++i) {
        // slot i holds relative time count - 3 + i
        next[i] = count + i >= 3 ? qkv[static_cast<size_t>(count + i - 3) * kChannels + c]
                                 : history[count + i];
    }
#pragma unroll
    for (uint32_t i = 0; i < 3; ++i) {
        history[i] = next[i];
    }
}

constexpr uint32_t kDeltaTokens = 1024;  // tokens of one k_gated_delta_chunk launch, at most

// Sums of a and b over each 16-lane row of the wave, the two rotations of a
// step side by side (each fills the other's wait); every lane of the row gets
// the same bits (a rotation adds the same two partial sums in either order).
__device__ __forceinline__ void row16_sums(float &a, float &b) {
    const auto step = [&](auto control) {
        const auto rotated = [](float x) {
            return __uint_as_float(static_cast<uint32_t>(__builtin_amdgcn_mov_dpp(
                static_cast<int>(__float_as_uint(x)), decltype(control)::value, 0xF, 0xF, true)));
        };
        a += rotated(a);
        b += rotated(b);
    };
    step(std::integral_constant<int, 0x128>{});  // row_ror:8
    step(std::integral_constant<int, 0x124>{});  // row_ror:4
    step(std::integral_constant<int, 0x122>{});  // row_ror:2
    step(std::integral_constant<int, 0x121>{});  // row_ror:1
}

// gated_delta_head over a chunk of tokens in order: block (value head, 16
// state rows), wave w its rows 4 w .. 4 w + 3, sixteen lanes a row, lane j of
// them columns 4 j .. 4 j + 3 and 64 + 4 j .. 64 + 4 j + 3. What bounds it is
// the chain from one token's state to the next (dot, reduction, update), so
// the chip's 4096 rows are spread to one wave a SIMD, with a reduction of four
// row rotations over eight values a lane: 60 vector instructions a token for
// four rows. One wave a row (two values a lane, six cross-lane steps, two of
// them row swaps, four waves a SIMD) took 230 us for 512 tokens, this takes
// 80. The block's query, key and value entries of sixteen tokens are loaded
// while the sixteen before run, and pass through LDS (one barrier per
// sixteen), from where each token's are read while the one before runs (read
// at their use: 101 us). Lane j keeps token j's attended value, so sixteen
// tokens go out in one store.
__global__ __launch_bounds__(256, 1) void k_gated_delta_chunk(const float *convolved, const float *alpha,
                                                              const float *beta, const uint16_t *alpha_bias,
                                                              const uint16_t *a_log, uint32_t count,
                                                              float *recurrent, float *output) {
    constexpr uint32_t kStep = 16;  // tokens a stage
    __shared__ float2 token_gates[kDeltaTokens];  // decay, beta
    __shared__ __align__(16) float4 qk_lds[2][kStep][2 * kLinearHead / 4];  // query, then key
    __shared__ float v_lds[2][kStep][kDeltaRows];
    const uint32_t h = blockIdx.x;
    const uint32_t kh = h / (kValueHeads / kKeyHeads);
    const uint32_t t = threadIdx.x, lane = t & 63u, wave = t >> 6;
    const uint32_t j = lane & 15u, local_row = wave * 4u + (lane >> 4);
    const uint32_t row = blockIdx.y * kDeltaRows + local_row;
    // (the state's alignment is 8 bytes)
    float2 *state = reinterpret_cast<float2 *>(recurrent + (static_cast<size_t>(h) * kLinearHead + row) * kLinearHead);
    const float2 a = state[2u * j], b = state[2u * j + 1u], c = state[32u + 2u * j], d = state[33u + 2u * j];
    float4 s0 = make_float4(a.x, a.y, b.x, b.y), s1 = make_float4(c.x, c.y, d.x, d.y);
    // thread t stages float4 t % 64 (query 0-31, key 32-63) of tokens
    // t / 64 + 4 i, and the value entry of token t / 16, row t % 16; a token
    // past the chunk reloads the last one
    const float4 *qk_from = reinterpret_cast<const float4 *>(
        convolved + ((t & 63u) < 32u ? static_cast<size_t>(kh) * kLinearHead
                                     : kQkSize + static_cast<size_t>(kh) * kLinearHead));
    const float *v_from = convolved + 2u * kQkSize + static_cast<size_t>(h) * kLinearHead +
                          blockIdx.y * kDeltaRows + (t & 15u);
    struct Stage {
        float4 qk0, qk1, qk2, qk3;
        float v;
    };
    const auto load_stage = [&](uint32_t b0) {
        const auto qk = [&](uint32_t i) {
            const uint32_t at = min(b0 + (t >> 6) + 4u * i, count - 1u);
            return qk_from[static_cast<size_t>(at) * (kChannels / 4u) + (t & 31u)];
        };
        return Stage{qk(0), qk(1), qk(2), qk(3),
                     v_from[static_cast<size_t>(min(b0 + (t >> 4), count - 1u)) * kChannels]};
    };
    const auto store_stage = [&](uint32_t slot, const Stage &in) {
        qk_lds[slot][t >> 6][t & 63u] = in.qk0;
        qk_lds[slot][(t >> 6) + 4u][t & 63u] = in.qk1;
        qk_lds[slot][(t >> 6) + 8u][t & 63u] = in.qk2;
        qk_lds[slot][(t >> 6) + 12u][t & 63u] = in.qk3;
        v_lds[slot][t >> 4][t & 15u] = in.v;
    };
    const Stage first = load_stage(0);
    const float bias = bf16_bits_to_float(alpha_bias[h]);
    const float rate = expf(bf16_bits_to_float(a_log[h]));
    for (uint32_t at = t; at < count; at += 256u) {
        const float biased = alpha[static_cast<size_t>(at) * kValueHeads + h] + bias;
        const float softplus = biased > 20.0f ? biased : log1pf(expf(biased));
        token_gates[at] = make_float2(expf(-rate * softplus),
                                      sigmoid_of(beta[static_cast<size_t>(at) * kValueHeads + h]));
    }
    const float output_scale = 1.0f / sqrtf(static_cast<float>(kLinearHead));
    store_stage(0, first);
    uint32_t slot = 0;
    for (uint32_t b0 = 0; b0 < count; b0 += kStep, slot ^= 1u) {
        // the barrier also frees the other slot: its tokens ran before it
        __syncthreads();
        const Stage ahead = load_stage(b0 + kStep);
        float kept = 0.0f;
        const uint32_t tokens = min(kStep, count - b0);
        struct TokenIn {
            float4 q0, q1, k0, k1;
            float2 gates;
            float v;
        };
        const auto read = [&](uint32_t u) {
            return TokenIn{qk_lds[slot][u][j], qk_lds[slot][u][16u + j], qk_lds[slot][u][32u + j],
                           qk_lds[slot][u][48u + j], token_gates[b0 + u], v_lds[slot][u][local_row]};
        };
        const auto dot = [&](const float4 &x, const float4 &y) {
            return fmaf(s0.w, x.w, fmaf(s0.z, x.z, fmaf(s0.y, x.y, s0.x * x.x))) +
                   fmaf(s1.w, y.w, fmaf(s1.z, y.z, fmaf(s1.y, y.y, s1.x * y.x)));
        };
        // token u's attended value is summed beside token u + 1's prediction
        float attended = 0.0f;
        const auto update = [&](uint32_t u, const TokenIn &in) {
            float prediction = dot(in.k0, in.k1);
            row16_sums(prediction, attended);
            kept = j + 1u == u ? attended : kept;
            const float decay = in.gates.x;
            const float delta = (in.v - prediction * decay) * in.gates.y;
            s0.x = fmaf(s0.x, decay, in.k0.x * delta);
            s0.y = fmaf(s0.y, decay, in.k0.y * delta);
            s0.z = fmaf(s0.z, decay, in.k0.z * delta);
            s0.w = fmaf(s0.w, decay, in.k0.w * delta);
            s1.x = fmaf(s1.x, decay, in.k1.x * delta);
            s1.y = fmaf(s1.y, decay, in.k1.y * delta);
            s1.z = fmaf(s1.z, decay, in.k1.z * delta);
            s1.w = fmaf(s1.w, decay, in.k1.w * delta);
            attended = dot(in.q0, in.q1);
        };
        // each token's entries are read from LDS while the one before runs
        TokenIn in = read(0);
        if (tokens == kStep) {
#pragma unroll
            for (uint32_t u = 0; u < kStep; ++u) {
                const TokenIn next = read(u + 1u < kStep ? u + 1u : u);
                __builtin_amdgcn_sched_barrier(0);
                update(u, in);
                in = next;
            }
        } else {
            for (uint32_t u = 0; u < tokens; ++u) {
                update(u, read(u));
            }
        }
        float unused = 0.0f;
        row16_sums(attended, unused);
        kept = j + 1u == tokens ? attended : kept;
        kept *= output_scale;
        if (j < tokens) {
            output[static_cast<size_t>(b0 + j) * kValueSize + static_cast<size_t>(h) * kLinearHead + row] = kept;
        }
        store_stage(slot ^ 1u, ahead);
    }
    state[2u * j] = make_float2(s0.x, s0.y);
    state[2u * j + 1u] = make_float2(s0.z, s0.w);
    state[32u + 2u * j] = make_float2(s1.x, s1.y);
    state[33u + 2u * j] = make_float2(s1.z, s1.w);
}

// gated_delta_head (src/executor.cpp:121-155) for one token of sequence r:
// block (value head, row block, r), a wave four of the block's 16 state rows,
// a lane two of a row's 128 values (src/simd.cpp:108-127).
__global__ __launch_bounds__(256) void k_gated_delta_rows(const float *convolved,
                                                          const float *alpha, const float *beta,
                                                          const uint16_t *alpha_bias,
                                                          const uint16_t *a_log, LinearRows rows,
                                                          float *output) {
#pragma clang fp contract(off)
    constexpr uint32_t kRows = kDeltaRows / 4u;  // rows of a wave
    const uint32_t h = blockIdx.x, r = blockIdx.z;
    const uint32_t kh = h / (kValueHeads / kKeyHeads);
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    const uint32_t row0 = blockIdx.y * kDeltaRows + wave * kRows;
    const float *token = convolved + static_cast<size_t>(r) * kChannels;
    float2 *state = reinterpret_cast<float2 *>(rows.recurrent[r] +
                                               (static_cast<size_t>(h) * kLinearHead + row0) * kLinearHead);
    const float2 q = reinterpret_cast<const float2 *>(token + static_cast<size_t>(kh) * kLinearHead)[lane];
    const float2 k = reinterpret_cast<const float2 *>(token + kQkSize + static_cast<size_t>(kh) * kLinearHead)[lane];
    const float4 v = *reinterpret_cast<const float4 *>(token + 2u * kQkSize + static_cast<size_t>(h) * kLinearHead + row0);
    const float value[kRows] = {v.x, v.y, v.z, v.w};
    const float beta_value = sigmoid_of(beta[static_cast<size_t>(r) * kValueHeads + h]);
    const float biased = alpha[static_cast<size_t>(r) * kValueHeads + h] + bf16_bits_to_float(alpha_bias[h]);
    const float softplus = biased > 20.0f ? biased : log1pf(expf(biased));
    const float decay = expf(-expf(bf16_bits_to_float(a_log[h])) * softplus);
    const float output_scale = 1.0f / sqrtf(static_cast<float>(kLinearHead));
    float attended[kRows];
#pragma unroll
    for (uint32_t j = 0; j < kRows; ++j) {
        float2 s = state[j * (kLinearHead / 2u) + lane];
        s.x *= decay;
        s.y *= decay;
        const float prediction = wave_sum(s.x * k.x + s.y * k.y);
        const float delta = (value[j] - prediction) * beta_value;
        s.x += k.x * delta;
        s.y += k.y * delta;
        attended[j] = wave_sum(s.x * q.x + s.y * q.y) * output_scale;
        state[j * (kLinearHead / 2u) + lane] = s;
    }
    if (lane == 0) {
        *reinterpret_cast<float4 *>(output + static_cast<size_t>(r) * kValueSize + static_cast<size_t>(h) * kLinearHead +
                                    row0) = make_float4(attended[0], attended[1], attended[2], attended[3]);
    }
}

// The causal convolution and SiLU of channel c for one token whose three
// earlier inputs are in `history` (src/executor.cpp:480-496): the output and
// the channel's shifted state (h1, h2, x).
struct ConvChannel {
    float y, h1, h2, x;
};
__device__ __forceinline__ ConvChannel conv_channel(const float *qkv_row, const uint16_t *weights,
                                                    const float *history, uint32_t c) {
#pragma clang fp contract(off)
    const uint2 packed = *reinterpret_cast<const uint2 *>(weights + static_cast<size_t>(c) * 4u);
    const float w0 = bf16_bits_to_float(packed.x & 0xFFFFu), w1 = bf16_bits_to_float(packed.x >> 16);
    const float w2 = bf16_bits_to_float(packed.y & 0xFFFFu), w3 = bf16_bits_to_float(packed.y >> 16);
    const float h0 = history[0], h1 = history[1], h2 = history[2];
    const float x = qkv_row[c];
    float v = 0.0f;
    v += h0 * w0;
    v += h1 * w1;
    v += h2 * w2;
    v += x * w3;
    return {silu_of(v), h1, h2, x};
}

// One decode token of each of up to kRowGroup sequences through the Gated
// DeltaNet core in one launch: the convolution with the query and key L2
// norms, the delta rule and the gated RMS norm (src/executor.cpp:480-550),
// with the arithmetic of k_linear_conv_rows, k_gated_delta_rows and
// k_linear_norm_gate. Block (value head h, row block y, sequence r):
// - convolves the 128 query and 128 key channels of h's key head itself (every
//   block of a key head does, each sum in the 128-thread block's order) and its
//   own ROWS value channels, whose state only it shifts;
// - updates its ROWS state rows and writes their outputs through to memory;
// - the last of the head's blocks through the head's ticket reads the 128
//   outputs back and writes the head's gated norm; the last of the key head's
//   blocks through its ticket shifts the query and key channels' state (every
//   one of them has read it by then).
// `tickets` holds 48 words a sequence (32 value heads, 16 key heads), zero
// between calls: the last block through each ticket clears it.
// With LANES 8 or 16 the block also computes its head's alpha and beta
// (the bf16 matmuls of the normalized row `x`, in the CPU's LANES-lane order
// as k_bf16_lds does): the row and the two weight rows staged in LDS, one
// wave's lanes 0 .. 2 LANES - 1 running the chains. With LANES 0 they come
// precomputed in alpha and beta.
//
// ROWS state rows a block: every block of a head repeats the head's
// convolution, decay chains and their loads, so more rows a block cost less in
// all, and fewer blocks leave the chip idle for few sequences. us a launch with
// 16, 32, 64, 128 rows: 1 sequence 11.0, 9.9, 11.1, 13.0; 4 15.4, 13.0, 13.0,
// 14.3; 8 20.4, 17.1, 16.8, 17.3; 16 32.9, 26.7, 23.3, 23.3; 32 (134 MB of
// states) 54.3, 40.8, 40.3, 42.6.
constexpr uint32_t kCoreRows = 32;       // below kCoreManyRows sequences, then 64
constexpr uint32_t kCoreManyRows = 8;
constexpr uint32_t kDecayColumns = 2048;  // the widest row staged for alpha and beta
template <int LANES, uint32_t ROWS>
__global__ __launch_bounds__(256) void k_linear_core_rows(const float *qkv, const uint16_t *weights,
                                                          LinearRows rows, const float *x,
                                                          const uint16_t *alpha_w, const uint16_t *beta_w,
                                                          uint32_t columns, const float *alpha,
                                                          const float *beta, const uint16_t *alpha_bias,
                                                          const uint16_t *a_log, const uint16_t *norm,
                                                          const float *gate, float *recurrent_output,
                                                          float *normalized, uint32_t *tickets) {
#pragma clang fp contract(off)
    constexpr uint32_t kRows = ROWS / 4u;
    constexpr uint32_t kHeadBlocks = kLinearHead / ROWS;
    constexpr uint32_t kStaged = LANES > 0 ? kDecayColumns : 4u;
    __shared__ float qk[2][kLinearHead];
    __shared__ float vv[ROWS];
    __shared__ float part[4];
    __shared__ float decay_in[2];
    __shared__ __align__(16) float x_lds[kStaged];
    __shared__ __align__(16) uint16_t w_lds[2][kStaged];
    __shared__ uint32_t last;
    const uint32_t h = blockIdx.x, y = blockIdx.y, r = blockIdx.z;
    const uint32_t kh = h / (kValueHeads / kKeyHeads);
    const uint32_t t = threadIdx.x, lane = t & 63u, wave = t >> 6;
    const float *row = qkv + static_cast<size_t>(r) * kChannels;
    float *history = rows.convolution[r];
    const uint32_t row0 = y * ROWS + wave * kRows;
    // the state rows first, so that their loads overlap the convolution
    float2 *state = reinterpret_cast<float2 *>(rows.recurrent[r] +
                                               (static_cast<size_t>(h) * kLinearHead + row0) * kLinearHead);
    float2 s[kRows];
#pragma unroll
    for (uint32_t j = 0; j < kRows; ++j) {
        s[j] = state[j * (kLinearHead / 2u) + lane];
    }
    // the row and the head's alpha and beta weight rows (columns <= 2048, a
    // multiple of 256) into LDS: every load issued first (indexes past the
    // row clamped), then the stores
    constexpr uint32_t kX4 = LANES > 0 ? kDecayColumns / 4u / 256u : 1u;
    constexpr uint32_t kW8 = LANES > 0 ? kDecayColumns / 8u / 256u : 1u;
    float4 xv[kX4];
    uint4 av[kW8], bv[kW8];
    if constexpr (LANES > 0) {
        const float4 *xs = reinterpret_cast<const float4 *>(x + static_cast<size_t>(r) * columns);
#pragma unroll
        for (uint32_t k = 0; k < kX4; ++k) {
            xv[k] = xs[min(t + 256u * k, columns / 4u - 1u)];
        }
        const uint4 *wa = reinterpret_cast<const uint4 *>(alpha_w + static_cast<size_t>(h) * columns);
        const uint4 *wb = reinterpret_cast<const uint4 *>(beta_w + static_cast<size_t>(h) * columns);
#pragma unroll
        for (uint32_t k = 0; k < kW8; ++k) {
            av[k] = wa[min(t + 256u * k, columns / 8u - 1u)];
            bv[k] = wb[min(t + 256u * k, columns / 8u - 1u)];
        }
    }
    if constexpr (LANES > 0) {
#pragma unroll
        for (uint32_t k = 0; k < kX4; ++k) {
            if (t + 256u * k < columns / 4u) {
                reinterpret_cast<float4 *>(x_lds)[t + 256u * k] = xv[k];
            }
        }
#pragma unroll
        for (uint32_t k = 0; k < kW8; ++k) {
            if (t + 256u * k < columns / 8u) {
                reinterpret_cast<uint4 *>(w_lds[0])[t + 256u * k] = av[k];
                reinterpret_cast<uint4 *>(w_lds[1])[t + 256u * k] = bv[k];
            }
        }
    }
    // threads 0-127 the query channels, 128-255 the key channels; each L2
    // norm sums as a 128-thread block does: (0 + wave 0) + wave 1
    const uint32_t half = t >> 7;
    const uint32_t c = half * kQkSize + kh * kLinearHead + (t & (kLinearHead - 1u));
    const ConvChannel cc = conv_channel(row, weights, history + static_cast<size_t>(c) * 3u, c);
    const float sq = wave_sum(cc.y * cc.y);
    if (lane == 0) {
        part[wave] = sq;
    }
    if (t < ROWS) {
        const uint32_t cv = 2u * kQkSize + h * kLinearHead + y * ROWS + t;
        float *hv = history + static_cast<size_t>(cv) * 3u;
        const ConvChannel v = conv_channel(row, weights, hv, cv);
        vv[t] = v.y;
        hv[0] = v.h1;
        hv[1] = v.h2;
        hv[2] = v.x;
    }
    __syncthreads();
    float squares = 0.0f;
    squares += part[2u * half];
    squares += part[2u * half + 1u];
    qk[half][t & (kLinearHead - 1u)] = cc.y * (1.0f / sqrtf(squares + kEpsilon));
    if constexpr (LANES > 0) {
        if (wave == 3u) {
            // lanes 0 .. LANES - 1 alpha's chains, LANES .. 2 LANES - 1 beta's
            // (the lanes past them repeat those)
            const uint32_t g = (lane / LANES) & 1u;
            const float acc = router_chain<LANES>(w_lds[g], x_lds, columns, lane % LANES);
            const float a = router_lane_sum<LANES>(acc, 0u);
            const float b = router_lane_sum<LANES>(acc, 1u);
            if (lane == 0) {
                decay_in[0] = a;
                decay_in[1] = b;
            }
        }
    }
    __syncthreads();
    // the delta rule on the block's rows (gated_delta_rows_of_head, one token)
    {
        const float2 q = make_float2(qk[0][2u * lane], qk[0][2u * lane + 1u]);
        const float2 k = make_float2(qk[1][2u * lane], qk[1][2u * lane + 1u]);
        const float bias = bf16_bits_to_float(alpha_bias[h]);
        const float rate = expf(bf16_bits_to_float(a_log[h]));
        const float output_scale = 1.0f / sqrtf(static_cast<float>(kLinearHead));
        const float alpha_in = LANES > 0 ? decay_in[0] : alpha[static_cast<size_t>(r) * kValueHeads + h];
        const float beta_in = LANES > 0 ? decay_in[1] : beta[static_cast<size_t>(r) * kValueHeads + h];
        const float beta_value = sigmoid_of(beta_in);
        const float biased = alpha_in + bias;
        const float softplus = biased > 20.0f ? biased : log1pf(expf(biased));
        const float decay = expf(-rate * softplus);
        float *out = recurrent_output + static_cast<size_t>(r) * kValueSize + static_cast<size_t>(h) * kLinearHead;
        float attended = 0.0f;  // lane j the output of row j
#pragma unroll
        for (uint32_t j = 0; j < kRows; ++j) {
            s[j].x *= decay;
            s[j].y *= decay;
            const float prediction = wave_sum(s[j].x * k.x + s[j].y * k.y);
            const float delta = (vv[wave * kRows + j] - prediction) * beta_value;
            s[j].x += k.x * delta;
            s[j].y += k.y * delta;
            const float output = wave_sum(s[j].x * q.x + s[j].y * q.y) * output_scale;
            attended = lane == j ? output : attended;
        }
        if (lane < kRows) {
            coherent_store(out + row0 + lane, attended);
        }
#pragma unroll
        for (uint32_t j = 0; j < kRows; ++j) {
            state[j * (kLinearHead / 2u) + lane] = s[j];
        }
    }
    uint32_t *ticket = tickets + static_cast<size_t>(r) * (kValueHeads + kKeyHeads);
    wait_stores();
    __syncthreads();
    if (t == 0) {
        last = coherent_add(ticket + h, 1u) + 1u == kHeadBlocks ? 1u : 0u;
    }
    __syncthreads();
    if (last != 0u) {
        // the head's gated RMS norm (k_linear_norm_gate's arithmetic on
        // threads 0-127)
        const size_t i = static_cast<size_t>(r) * kValueSize + static_cast<size_t>(h) * kLinearHead + t;
        const float x = t < kLinearHead ? coherent_load(recurrent_output + i) : 0.0f;
        const float sx = wave_sum(x * x);
        if (lane == 0) {
            part[wave] = sx;
        }
        __syncthreads();
        if (t < kLinearHead) {
            float total = 0.0f;
            total += part[0];
            total += part[1];
            const float scale = 1.0f / sqrtf(total / static_cast<float>(kLinearHead) + kEpsilon);
            normalized[i] = x * scale * (0.0f + bf16_bits_to_float(norm[t])) * silu_of(gate[i]);
        }
        if (t == 0) {
            coherent_store(ticket + h, 0u);
        }
    }
    __syncthreads();
    if (t == 0) {
        last = coherent_add(ticket + kValueHeads + kh, 1u) + 1u == 2u * kHeadBlocks ? 1u : 0u;
    }
    __syncthreads();
    if (last != 0u) {
        float *hc = history + static_cast<size_t>(c) * 3u;
        hc[0] = cc.h1;
        hc[1] = cc.h2;
        hc[2] = cc.x;
        if (t == 0) {
            coherent_store(ticket + kValueHeads + kh, 0u);
        }
    }
}

// rms_norm (weight offset 0, src/kernels.cpp:1052-1073) of each value head,
// times SiLU of the gate (src/executor.cpp:538-550).
__global__ __launch_bounds__(kLinearHead) void k_linear_norm_gate(const float *recurrent_output,
                                                                  const uint16_t *norm,
                                                                  const float *gate,
                                                                  float *normalized, const float *qkv,
                                                                  float *convolution) {
#pragma clang fp contract(off)
    if (blockIdx.x >= kValueHeads) {  // the grid's last columns, after a chunk: the convolution state
        const uint32_t block = (blockIdx.x - kValueHeads) * gridDim.y + blockIdx.y;
        const uint32_t blocks = (gridDim.x - kValueHeads) * gridDim.y;
        for (uint32_t c = block * kLinearHead + threadIdx.x; c < kChannels; c += blocks * kLinearHead) {
            shift_history(qkv, gridDim.y, convolution, c);
        }
        return;
    }
    __shared__ float partial[16];
    const size_t i = static_cast<size_t>(blockIdx.y) * kValueSize +
                     static_cast<size_t>(blockIdx.x) * kLinearHead + threadIdx.x;
    const float x = recurrent_output[i];
    const float squares = block_sum(x * x, partial);
    const float scale = 1.0f / sqrtf(squares / static_cast<float>(kLinearHead) + kEpsilon);
    normalized[i] = x * scale * (0.0f + bf16_bits_to_float(norm[threadIdx.x])) * silu_of(gate[i]);
}

// hidden += branch (the residual adds of decode_layer).
__global__ __launch_bounds__(256) void k_residual_add(float *hidden, const float *branch,
                                                      uint32_t count) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < count) {
        hidden[i] = hidden[i] + branch[i];
    }
}

// prepare_rope (src/executor.cpp:43-58) with MachModel's divisors
// (src/model.cpp:606-615), on the host with the reference's float libm calls.
RopeDivisors rope_divisors() {
    RopeDivisors d{};
    for (uint32_t i = 0; i < kRopeHalf; ++i) {
        d.divisor[i] = std::pow(10000000.0F, 2.0F * static_cast<float>(i) / 64.0F);
    }
    return d;
}

RopeTable rope_table(uint32_t position) {
    const RopeDivisors d = rope_divisors();
    RopeTable t{};
    for (uint32_t i = 0; i < kRopeHalf; ++i) {
        const float theta = static_cast<float>(position) / d.divisor[i];
        t.cosine[i] = std::cos(theta);
        t.sine[i] = std::sin(theta);
    }
    return t;
}

// The context's device table of rope_table(p) for p < end, grown on demand
// (the whole table is rebuilt on the host and copied when it grows).
const float *rope_rows(adi_hip_context *ctx, uint32_t end) {
    if (end > ctx->rope_positions) {
        uint32_t positions = ctx->rope_positions * 2 > 1024 ? ctx->rope_positions * 2 : 1024u;
        positions = positions > end ? positions : end;
        std::vector<float> host(size_t(positions) * 2 * kRopeHalf);
        for (uint32_t p = 0; p < positions; ++p) {
            const RopeTable t = rope_table(p);
            std::copy(t.cosine, t.cosine + kRopeHalf, host.begin() + size_t(p) * 2 * kRopeHalf);
            std::copy(t.sine, t.sine + kRopeHalf,
                      host.begin() + size_t(p) * 2 * kRopeHalf + kRopeHalf);
        }
        ctx->rope_positions = 0;
        ctx->rope_cache.ensure(host.size() * sizeof(float));  // waits for the device before a free
        check_hip(hipStreamSynchronize(ctx->stream), "rope table synchronize");
        check_hip(hipMemcpy(ctx->rope_cache.base, host.data(), host.size() * sizeof(float),
                            hipMemcpyHostToDevice),
                  "rope table upload");
        ctx->rope_positions = positions;
    }
    return static_cast<const float *>(ctx->rope_cache.base);
}

// A nested entry's status becomes this call's failure.
void forward(adi_hip_context *ctx, int status) {
    if (status != ADI_HIP_OK) {
        fail(status, ctx->last_error());
    }
}

// The query (with its gate), key and value projections of the same rows
// (three backend.ne_matmul calls, src/executor.cpp:596-613) in one NE launch
// where it takes the shapes.
void project_qkv(adi_hip_context *ctx, const adi_hip_full_attention *L, const float *inputs,
                 uint32_t count, float *query_gate, float *key, float *value, const NeNormIn *norm_in) {
    const adi_hip_ne_matrix *m[3] = {&L->query, &L->key, &L->value};
    float *out[3] = {query_gate, key, value};
    ne_matmul_group(ctx, m, 3, inputs, count, out, norm_in);
}

// The Gated DeltaNet's qkv and gate projections of the same rows (two
// backend.ne_matmul calls, src/executor.cpp:764-775) in one NE launch where
// it takes the shapes.
void project_qkv_gate(adi_hip_context *ctx, const adi_hip_linear_attention *L, const float *inputs,
                      uint32_t count, float *qkv, float *gate, const NeNormIn *norm_in) {
    const adi_hip_ne_matrix *m[2] = {&L->qkv, &L->gate};
    float *out[2] = {qkv, gate};
    ne_matmul_group(ctx, m, 2, inputs, count, out, norm_in);
}

// The decay inputs alpha and beta of the same rows (two dense bf16 matmuls,
// src/executor.cpp:776-787) in one launch where the small-batch kernel
// takes them (with the one-launch decode paths on).
void project_decay(adi_hip_context *ctx, const adi_hip_linear_attention *L, const float *x, uint32_t count,
                   float *alpha, float *beta) {
    if (!ctx->fused_moe) {
        forward(ctx, adi_hip_bf16_matmul(ctx, &L->alpha, x, count, alpha));
        forward(ctx, adi_hip_bf16_matmul(ctx, &L->beta, x, count, beta));
        return;
    }
    launch_bf16_pair(ctx, L->alpha.values, L->alpha.rows, L->beta.values, L->beta.rows, L->alpha.columns, x,
                     count, alpha, beta, ctx->isa_lanes);
}

// The output projection, then (with `tail`) the residual add and the next
// RMS norm folded into it where the one-launch NE projection takes it.
void project_output(adi_hip_context *ctx, const adi_hip_ne_matrix *m, const float *inputs, uint32_t count,
                    float *outputs, const NeNormTail *tail) {
    if (tail == nullptr) {
        forward(ctx, adi_hip_ne_matmul(ctx, m, inputs, count, outputs));
        return;
    }
    ne_matmul_group(ctx, &m, 1, inputs, count, &outputs, nullptr, tail);
}

bool ne_shaped(const adi_hip_ne_matrix &m, uint32_t rows, uint32_t columns) {
    return m.rows == rows && m.columns == columns && m.trellis != nullptr;
}

// full_attention_forward for tokens position .. position + count - 1.
void full_attention_chunk(adi_hip_context *ctx, const adi_hip_full_attention *L,
                          uint32_t position, uint32_t count, const float *inputs, float *outputs,
                          float *keys, float *values, uint32_t capacity,
                          const NeNormIn *norm_in = nullptr, const NeNormTail *norm_tail = nullptr) {
    require(L != nullptr && inputs != nullptr && outputs != nullptr && keys != nullptr &&
                values != nullptr && count > 0,
            "full attention state or input shape mismatch");
    const uint32_t hidden = L->query.columns;
    require(ne_shaped(L->query, kQueryHeads * kQueryStride, hidden) &&
                ne_shaped(L->key, kKvHeads * kHeadSize, hidden) &&
                ne_shaped(L->value, kKvHeads * kHeadSize, hidden) &&
                ne_shaped(L->output, hidden, kQueryHeads * kHeadSize) &&
                L->query_norm != nullptr && L->key_norm != nullptr && position < capacity &&
                count <= capacity - position,
            "full attention state or input shape mismatch");
    require(aligned_to(keys, 16) && aligned_to(values, 16),
            "attention caches must be 16-byte aligned");
    auto &ws = ctx->layer_workspace;
    ws.used = 0;
    const size_t fixed = Workspace::round(size_t(count) * kQueryHeads * kQueryStride * 4) +
                         Workspace::round(size_t(count) * kQueryHeads * kHeadSize * 4);
    const bool matrix = attention_chunk_takes(position, count);
    // splits of the history for the chunk's last token; a chunk's many tokens
    // already give blocks enough, so they split less
    const uint32_t last = position + count;
    const uint32_t cap = kMaxSplits / count > 0 ? kMaxSplits / count : 1u;
    uint32_t splits = ceil_div(last, 32);
    splits = splits < 1 ? 1 : (splits > cap ? cap : splits);
    uint32_t chunk = ceil_div(last, splits);
    splits = ceil_div(last, chunk);
    if (matrix) {
        splits = attention_chunk_splits(position, count, ws.limit > fixed ? ws.limit - fixed : 0);
    }
    const size_t partials = matrix && splits == 1 ? 0 : size_t(count) * kQueryHeads * splits * kPartialStride;
    ws.ensure(fixed + Workspace::round(partials * 4));
    float *query_gate = ws.take<float>(size_t(count) * kQueryHeads * kQueryStride);
    float *attended = ws.take<float>(size_t(count) * kQueryHeads * kHeadSize);
    float *partial = ws.take<float>(partials);
    float *key = keys + static_cast<size_t>(position) * kKvHeads * kHeadSize;
    float *value = values + static_cast<size_t>(position) * kKvHeads * kHeadSize;
    project_qkv(ctx, L, inputs, count, query_gate, key, value, norm_in);
    launch(ctx, "attention_norm_rope", k_norm_rope, dim3(kQueryHeads + kKvHeads, count),
           dim3(kHeadSize), 0, query_gate, key, L->query_norm, L->key_norm,
           count == 1 ? rope_table(position) : RopeTable{},
           count == 1 ? nullptr : rope_rows(ctx, position + count), position);
    if (matrix) {
        launch_attention_chunk(ctx, query_gate, keys, values, position, count, splits, partial, attended);
    } else {
        launch(ctx, "attention_partial", k_attention_partial, dim3(partial_blocks(splits), 1, count),
               dim3(256), 0, static_cast<const float *>(query_gate), static_cast<const float *>(keys),
               static_cast<const float *>(values), position, chunk, splits, partial);
    }
    if (!matrix || splits > 1) {
        launch(ctx, "attention_combine", k_attention_combine, dim3(kQueryHeads, count),
               dim3(kHeadSize), 0, static_cast<const float *>(partial), splits,
               static_cast<const float *>(query_gate), attended);
    }
    project_output(ctx, &L->output, attended, count, outputs, norm_tail);
}

// Whether the Gated DeltaNet core launch computes alpha and beta itself from
// the normalized rows x (8- or 16-lane order, rows of at most 2048 columns,
// a multiple of 256, 16-byte aligned).
bool core_takes_decay(const adi_hip_context *ctx, const adi_hip_linear_attention *L, const float *x) {
    const uint32_t columns = L->alpha.columns;
    return (ctx->isa_lanes == 8 || ctx->isa_lanes == 16) && columns <= kDecayColumns && columns % 256u == 0 &&
           aligned_to(x, 16) && aligned_to(L->alpha.values, 16) && aligned_to(L->beta.values, 16);
}

// The Gated DeltaNet core of one token of each of `count` (<= kRowGroup)
// sequences in one launch (k_linear_core_rows): alpha and beta from the
// normalized rows x when core_takes_decay holds, else from alpha and beta.
void launch_linear_core(adi_hip_context *ctx, const adi_hip_linear_attention *L, const float *qkv,
                        const LinearRows &table, uint32_t count, const float *x, const float *alpha,
                        const float *beta, const float *gate, float *recurrent_output, float *normalized) {
    static_assert(kRowGroup * (kValueHeads + kKeyHeads) <= kMoeSyncWords - kMoeSyncLinear,
                  "the DeltaNet tickets fit their sync lines");
    using Kernel = void (*)(const float *, const uint16_t *, LinearRows, const float *, const uint16_t *,
                            const uint16_t *, uint32_t, const float *, const float *, const uint16_t *,
                            const uint16_t *, const uint16_t *, const float *, float *, float *, uint32_t *);
    const uint32_t lanes = core_takes_decay(ctx, L, x) ? ctx->isa_lanes : 0u;
    const auto pick = [&](auto rows) -> Kernel {
        constexpr uint32_t kBlockRows = decltype(rows)::value;
        return lanes == 16u  ? k_linear_core_rows<16, kBlockRows>
               : lanes == 8u ? k_linear_core_rows<8, kBlockRows>
                             : k_linear_core_rows<0, kBlockRows>;
    };
    const uint32_t block_rows = count < kCoreManyRows ? kCoreRows : 2u * kCoreRows;
    const Kernel kernel = count < kCoreManyRows ? pick(std::integral_constant<uint32_t, kCoreRows>{})
                                                : pick(std::integral_constant<uint32_t, 2u * kCoreRows>{});
    launch(ctx, "linear_core", kernel, dim3(kValueHeads, kLinearHead / block_rows, count), dim3(256), 0, qkv,
           L->convolution, table, x, L->alpha.values, L->beta.values, L->alpha.columns, alpha, beta,
           L->alpha_bias, L->a_log, L->norm, gate, recurrent_output, normalized, ctx->moe_sync + kMoeSyncLinear);
}

// linear_attention_forward for `count` consecutive tokens.
void linear_attention_chunk(adi_hip_context *ctx, const adi_hip_linear_attention *L,
                            uint32_t count, const float *inputs, float *outputs,
                            float *convolution_state, float *recurrent_state,
                            const NeNormIn *norm_in = nullptr, const NeNormTail *norm_tail = nullptr) {
    require(L != nullptr && inputs != nullptr && outputs != nullptr &&
                convolution_state != nullptr && recurrent_state != nullptr && count > 0,
            "linear attention input shape mismatch");
    const uint32_t hidden = L->qkv.columns;
    require(ne_shaped(L->qkv, kChannels, hidden) && ne_shaped(L->gate, kValueSize, hidden) &&
                ne_shaped(L->output, hidden, kValueSize),
            "linear attention input shape mismatch");
    require(L->alpha.rows == kValueHeads && L->alpha.columns == hidden &&
                L->beta.rows == kValueHeads && L->beta.columns == hidden &&
                L->alpha.values != nullptr && L->beta.values != nullptr &&
                L->alpha_bias != nullptr && L->a_log != nullptr,
            "linear attention decay shape mismatch");
    require(L->convolution != nullptr && aligned_to(L->convolution, 8),
            "linear attention convolution shape mismatch");
    require(L->norm != nullptr, "linear attention input shape mismatch");
    require(aligned_to(recurrent_state, 8), "linear attention state must be 8-byte aligned");
    auto &ws = ctx->layer_workspace;
    ws.used = 0;
    const size_t n = count;
    ws.ensure(Workspace::round(n * kChannels * 4) * 2 + Workspace::round(n * kValueSize * 4) * 3 +
              Workspace::round(n * kValueHeads * 4) * 2);
    float *qkv = ws.take<float>(n * kChannels);
    float *convolved = ws.take<float>(n * kChannels);
    float *gate = ws.take<float>(n * kValueSize);
    float *recurrent_output = ws.take<float>(n * kValueSize);
    float *normalized = ws.take<float>(n * kValueSize);
    float *alpha = ws.take<float>(n * kValueHeads);
    float *beta = ws.take<float>(n * kValueHeads);
    project_qkv_gate(ctx, L, inputs, count, qkv, gate, norm_in);
    const float *x = norm_in != nullptr ? norm_in->out : inputs;  // the normalized rows
    if (count == 1 && ctx->fused_moe) {
        if (!core_takes_decay(ctx, L, x)) {
            project_decay(ctx, L, x, count, alpha, beta);
        }
        LinearRows table{};
        table.convolution[0] = convolution_state;
        table.recurrent[0] = recurrent_state;
        launch_linear_core(ctx, L, qkv, table, 1, x, alpha, beta, gate, recurrent_output, normalized);
        project_output(ctx, &L->output, normalized, count, outputs, norm_tail);
        return;
    }
    project_decay(ctx, L, x, count, alpha, beta);
    launch(ctx, "linear_conv", k_linear_conv, dim3(kChannels / kLinearHead, count),
           dim3(kLinearHead), 0, static_cast<const float *>(qkv), L->convolution,
           convolution_state, convolved);
    const dim3 delta_grid(kValueHeads, kLinearHead / kDeltaRows);
    if (count == 1) {  // the decode step's bits
        LinearRows table{};
        table.recurrent[0] = recurrent_state;
        launch(ctx, "gated_delta", k_gated_delta_rows, delta_grid, dim3(256), 0, static_cast<const float *>(convolved),
               static_cast<const float *>(alpha), static_cast<const float *>(beta), L->alpha_bias, L->a_log, table,
               recurrent_output);
    }
    // at most kDeltaTokens tokens a launch; the state carries over in order
    for (uint32_t b0 = 0; count > 1 && b0 < count; b0 += kDeltaTokens) {
        const uint32_t n = count - b0 < kDeltaTokens ? count - b0 : kDeltaTokens;
        launch(ctx, "gated_delta", k_gated_delta_chunk, delta_grid, dim3(256), 0,
               static_cast<const float *>(convolved + static_cast<size_t>(b0) * kChannels),
               static_cast<const float *>(alpha + static_cast<size_t>(b0) * kValueHeads),
               static_cast<const float *>(beta + static_cast<size_t>(b0) * kValueHeads), L->alpha_bias, L->a_log,
               n, recurrent_state, recurrent_output + static_cast<size_t>(b0) * kValueSize);
    }
    // a chunk's state shifts here, where every token has read it, in blocks of
    // its own (a launch for it alone took 4.7 us): one for each 128 channels, or
    // as many as there are tokens (two blocks for all channels of two tokens
    // took longer than the launch: 52.5 us a layer, 48.7 before)
    const uint32_t shifts = count > 1 ? ceil_div(kChannels / kLinearHead, count) : 0u;
    launch(ctx, "linear_norm_gate", k_linear_norm_gate, dim3(kValueHeads + shifts, count),
           dim3(kLinearHead), 0, static_cast<const float *>(recurrent_output), L->norm,
           static_cast<const float *>(gate), normalized, static_cast<const float *>(qkv), convolution_state);
    project_output(ctx, &L->output, normalized, count, outputs, norm_tail);
}

// decode_layer for `count` consecutive tokens of rows `hidden`.
// The decoder layer on rows hidden[count][moe.hidden] (decode_layer,
// src/executor.cpp:1473-1529) up to its MoE block: hidden (+= pending, the
// previous layer's MoE rows, when given) is normalized, the attention's rows
// are added to it and normalized again, each add fused into its norm; the MoE
// rows go to moe_out (may be `pending`: that is read first), not yet added.
template <typename Attention>
void layer_body(adi_hip_context *ctx, const adi_hip_decoder_layer *L, uint32_t count,
                float *hidden, const float *pending, float *moe_out, Attention &&attention) {
    require(L != nullptr && hidden != nullptr && moe_out != nullptr && L->input_norm != nullptr &&
                L->post_attention_norm != nullptr && count > 0,
            "decoder layer input is null");
    const uint32_t n = L->moe.hidden;
    require(n > 0 && aligned_to(hidden, 16), "decoder hidden row must be 16-byte aligned");
    auto &ws = ctx->decoder_workspace;
    ws.used = 0;
    const size_t rows = size_t(count) * n;
    ws.ensure(Workspace::round(rows * 4) * 2);
    float *normalized = ws.take<float>(rows);
    float *branch = ws.take<float>(rows);
    // the input norm (with the residual add of the previous layer's MoE rows)
    // and the post-attention norm run inside the attention's first and last
    // projections where they can, else as norm launches around them
    const NeNormIn norm_in{hidden, pending, L->input_norm, normalized};
    const NeNormTail norm_tail{hidden, L->post_attention_norm, normalized};
    attention(static_cast<const float *>(normalized), branch, &norm_in, &norm_tail);
    forward(ctx, adi_hip_moe_forward(ctx, &L->moe, normalized, count, nullptr, moe_out, nullptr,
                                     nullptr));
}

// `count` consecutive tokens of one sequence at position .. position + count
// - 1 (pending and moe_out as layer_body's).
void decoder_chunk_body(adi_hip_context *ctx, const adi_hip_decoder_layer *L, uint32_t position,
                        uint32_t count, float *hidden, const float *pending, float *moe_out,
                        const adi_hip_layer_state *state) {
    require(state != nullptr, "decoder layer input is null");
    layer_body(ctx, L, count, hidden, pending, moe_out,
               [&](const float *in, float *out, const NeNormIn *norm_in, const NeNormTail *norm_tail) {
        if (L->full_attention != 0) {
            full_attention_chunk(ctx, &L->full, position, count, in, out, state->keys,
                                 state->values, state->capacity, norm_in, norm_tail);
        } else {
            linear_attention_chunk(ctx, &L->linear, count, in, out, state->convolution,
                                   state->recurrent, norm_in, norm_tail);
        }
    });
}

// The whole layer in place (the public layer entries): the MoE rows are
// added to hidden at the end.
void decoder_chunk(adi_hip_context *ctx, const adi_hip_decoder_layer *L, uint32_t position,
                   uint32_t count, float *hidden, const adi_hip_layer_state *state) {
    require(L != nullptr && hidden != nullptr && count > 0, "decoder layer input is null");
    auto &ws = ctx->layer_output;
    ws.used = 0;
    const size_t rows = size_t(count) * L->moe.hidden;
    ws.ensure(Workspace::round(rows * 4));
    float *moe_out = ws.take<float>(rows);
    decoder_chunk_body(ctx, L, position, count, hidden, nullptr, moe_out, state);
    launch(ctx, "residual_add", k_residual_add, dim3(ceil_div(rows, 256)), dim3(256), 0, hidden,
           static_cast<const float *>(moe_out), static_cast<uint32_t>(rows));
}

// full_attention_forward_batch (src/executor.cpp:561-731) for one decode
// token of each of `rows` sequences: row r is at positions[r] of the
// sequence whose cache is states[r]; the kernels read the positions from
// device_positions. The launches cover positions below `span` (the RoPE
// table and the grid's splits; at least every positions[r] + 1). The
// projections run batched over the rows; normalization, RoPE, the cache
// append and the attention run per sequence, kRowGroup sequences per launch.
void full_attention_rows(adi_hip_context *ctx, const adi_hip_full_attention *L, uint32_t rows,
                         const float *inputs, float *outputs,
                         const adi_hip_layer_state *const *states, const uint32_t *positions,
                         const uint32_t *device_positions, uint32_t span,
                         const NeNormIn *norm_in, const NeNormTail *norm_tail) {
    require(L != nullptr && inputs != nullptr && outputs != nullptr && states != nullptr &&
                positions != nullptr && device_positions != nullptr && rows > 0,
            "full attention batch shape mismatch");
    const uint32_t hidden = L->query.columns;
    require(ne_shaped(L->query, kQueryHeads * kQueryStride, hidden) &&
                ne_shaped(L->key, kKvHeads * kHeadSize, hidden) &&
                ne_shaped(L->value, kKvHeads * kHeadSize, hidden) &&
                ne_shaped(L->output, hidden, kQueryHeads * kHeadSize) &&
                L->query_norm != nullptr && L->key_norm != nullptr,
            "full attention batch shape mismatch");
    uint32_t last = 0;
    for (uint32_t r = 0; r < rows; ++r) {
        const adi_hip_layer_state *st = states[r];
        require(st != nullptr && st->keys != nullptr && st->values != nullptr &&
                    positions[r] < st->capacity,
                "full attention batch state mismatch");
        require(aligned_to(st->keys, 16) && aligned_to(st->values, 16),
                "attention caches must be 16-byte aligned");
        last = positions[r] + 1 > last ? positions[r] + 1 : last;
    }
    last = span > last ? span : last;
    auto &ws = ctx->layer_workspace;
    ws.used = 0;
    const size_t n = rows;
    const size_t fixed = Workspace::round(n * kQueryHeads * kQueryStride * 4) +
                         Workspace::round(n * kKvHeads * kHeadSize * 4) * 2 +
                         Workspace::round(n * kQueryHeads * kHeadSize * 4);
    // partial rows of at most kRowPartials parts, and within a workspace limit
    // (kLeastPartials parts are asked for in any case)
    const size_t part = n * kQueryHeads * kPartialStride * 4;
    const size_t fit = ws.limit > fixed + 256 ? (ws.limit - fixed - 256) / part : 0;
    uint32_t cap = std::min<uint32_t>(kMaxSplits, kRowPartials / rows);
    cap = std::max<uint32_t>(std::min<size_t>(cap, fit), std::max<uint32_t>(kLeastPartials / rows, 1u));
    const uint32_t splits = most_parts(last, cap);
    ws.ensure(fixed + Workspace::round(part * splits));
    float *query_gate = ws.take<float>(n * kQueryHeads * kQueryStride);
    float *key = ws.take<float>(n * kKvHeads * kHeadSize);
    float *value = ws.take<float>(n * kKvHeads * kHeadSize);
    float *attended = ws.take<float>(n * kQueryHeads * kHeadSize);
    float *partial = ws.take<float>(n * kQueryHeads * splits * kPartialStride);
    project_qkv(ctx, L, inputs, rows, query_gate, key, value, norm_in);
    const float *rope = rope_rows(ctx, last);
    for (uint32_t first = 0; first < rows; first += kRowGroup) {
        const uint32_t count = rows - first < kRowGroup ? rows - first : kRowGroup;
        FullRows table{};
        for (uint32_t i = 0; i < count; ++i) {
            table.keys[i] = states[first + i]->keys;
            table.values[i] = states[first + i]->values;
        }
        const uint32_t *row_positions = device_positions + first;
        float *qg = query_gate + static_cast<size_t>(first) * kQueryHeads * kQueryStride;
        if (ctx->fused_moe) {
            static_assert(kRowGroup * kQueryHeads <= kMoeSyncWords - kMoeSyncAttention,
                          "the attention tickets fit their sync line");
            launch(ctx, "attention_rows_one", k_attention_rows_one, dim3(kKvHeads * splits, 1, count),
                   dim3(256), 0, static_cast<const float *>(qg),
                   static_cast<const float *>(key + static_cast<size_t>(first) * kKvHeads * kHeadSize),
                   static_cast<const float *>(value + static_cast<size_t>(first) * kKvHeads * kHeadSize),
                   L->query_norm, L->key_norm, rope, table, row_positions, cap, splits,
                   partial + static_cast<size_t>(first) * kQueryHeads * splits * kPartialStride,
                   attended + static_cast<size_t>(first) * kQueryHeads * kHeadSize,
                   ctx->moe_sync + kMoeSyncAttention);
            continue;
        }
        launch(ctx, "attention_norm_rope_rows", k_norm_rope_rows,
               dim3(kQueryHeads + 2 * kKvHeads, count), dim3(kHeadSize), 0, qg,
               static_cast<const float *>(key + static_cast<size_t>(first) * kKvHeads * kHeadSize),
               static_cast<const float *>(value + static_cast<size_t>(first) * kKvHeads * kHeadSize),
               L->query_norm, L->key_norm, rope, table, row_positions);
        launch(ctx, "attention_partial_rows", k_attention_partial_rows,
               dim3(kKvHeads * splits, 1, count), dim3(256), 0, static_cast<const float *>(qg), table,
               row_positions, cap, splits,
               partial + static_cast<size_t>(first) * kQueryHeads * splits * kPartialStride);
        launch(ctx, "attention_combine", k_attention_combine, dim3(kQueryHeads, count), dim3(kHeadSize), 0,
               static_cast<const float *>(partial + static_cast<size_t>(first) * kQueryHeads * splits * kPartialStride),
               splits, static_cast<const float *>(qg), attended + static_cast<size_t>(first) * kQueryHeads * kHeadSize);
    }
    project_output(ctx, &L->output, attended, rows, outputs, norm_tail);
}

// linear_attention_forward_batch (src/executor.cpp:733-966) for one decode
// token of each of `rows` sequences with the states states[r]: projections
// batched, convolution and recurrence per sequence.
void linear_attention_rows(adi_hip_context *ctx, const adi_hip_linear_attention *L, uint32_t rows,
                           const float *inputs, float *outputs,
                           const adi_hip_layer_state *const *states,
                           const NeNormIn *norm_in, const NeNormTail *norm_tail) {
    require(L != nullptr && inputs != nullptr && outputs != nullptr && states != nullptr &&
                rows > 0,
            "linear attention batch shape mismatch");
    const uint32_t hidden = L->qkv.columns;
    require(ne_shaped(L->qkv, kChannels, hidden) && ne_shaped(L->gate, kValueSize, hidden) &&
                ne_shaped(L->output, hidden, kValueSize),
            "linear attention batch shape mismatch");
    require(L->alpha.rows == kValueHeads && L->alpha.columns == hidden &&
                L->beta.rows == kValueHeads && L->beta.columns == hidden &&
                L->alpha.values != nullptr && L->beta.values != nullptr &&
                L->alpha_bias != nullptr && L->a_log != nullptr,
            "linear attention decay shape mismatch");
    require(L->convolution != nullptr && aligned_to(L->convolution, 8),
            "linear attention convolution shape mismatch");
    require(L->norm != nullptr, "linear attention batch shape mismatch");
    for (uint32_t r = 0; r < rows; ++r) {
        const adi_hip_layer_state *st = states[r];
        require(st != nullptr && st->convolution != nullptr && st->recurrent != nullptr,
                "linear attention recurrent state mismatch");
        require(aligned_to(st->recurrent, 8), "linear attention state must be 8-byte aligned");
    }
    auto &ws = ctx->layer_workspace;
    ws.used = 0;
    const size_t n = rows;
    ws.ensure(Workspace::round(n * kChannels * 4) * 2 + Workspace::round(n * kValueSize * 4) * 3 +
              Workspace::round(n * kValueHeads * 4) * 2);
    float *qkv = ws.take<float>(n * kChannels);
    float *convolved = ws.take<float>(n * kChannels);
    float *gate = ws.take<float>(n * kValueSize);
    float *recurrent_output = ws.take<float>(n * kValueSize);
    float *normalized = ws.take<float>(n * kValueSize);
    float *alpha = ws.take<float>(n * kValueHeads);
    float *beta = ws.take<float>(n * kValueHeads);
    project_qkv_gate(ctx, L, inputs, rows, qkv, gate, norm_in);
    const float *x = norm_in != nullptr ? norm_in->out : inputs;  // the normalized rows
    if (!ctx->fused_moe || !core_takes_decay(ctx, L, x)) {
        project_decay(ctx, L, x, rows, alpha, beta);
    }
    for (uint32_t first = 0; first < rows; first += kRowGroup) {
        const uint32_t count = rows - first < kRowGroup ? rows - first : kRowGroup;
        LinearRows table{};
        for (uint32_t i = 0; i < count; ++i) {
            table.convolution[i] = states[first + i]->convolution;
            table.recurrent[i] = states[first + i]->recurrent;
        }
        const size_t at = static_cast<size_t>(first);
        if (ctx->fused_moe) {
            launch_linear_core(ctx, L, qkv + at * kChannels, table, count, x + at * L->alpha.columns,
                               alpha + at * kValueHeads, beta + at * kValueHeads, gate + at * kValueSize,
                               recurrent_output + at * kValueSize, normalized + at * kValueSize);
            continue;
        }
        launch(ctx, "linear_conv_rows", k_linear_conv_rows, dim3(kChannels / kLinearHead, count),
               dim3(kLinearHead), 0, static_cast<const float *>(qkv + at * kChannels),
               L->convolution, table, convolved + at * kChannels);
        launch(ctx, "gated_delta_rows", k_gated_delta_rows,
               dim3(kValueHeads, kLinearHead / kDeltaRows, count), dim3(256), 0,
               static_cast<const float *>(convolved + at * kChannels),
               static_cast<const float *>(alpha + at * kValueHeads),
               static_cast<const float *>(beta + at * kValueHeads), L->alpha_bias, L->a_log, table,
               recurrent_output + at * kValueSize);
        launch(ctx, "linear_norm_gate", k_linear_norm_gate, dim3(kValueHeads, count), dim3(kLinearHead),
               0, static_cast<const float *>(recurrent_output + at * kValueSize), L->norm,
               static_cast<const float *>(gate + at * kValueSize), normalized + at * kValueSize,
               static_cast<const float *>(nullptr), static_cast<float *>(nullptr));
    }
    project_output(ctx, &L->output, normalized, rows, outputs, norm_tail);
}

}  // namespace

void decoder_rows(adi_hip_context *ctx, const adi_hip_decoder_layer *L, uint32_t rows,
                  float *hidden, const float *pending, float *moe_out,
                  const adi_hip_layer_state *const *states, const uint32_t *positions,
                  const uint32_t *device_positions, uint32_t span) {
    require(states != nullptr && positions != nullptr, "decoder batch shape mismatch");
    layer_body(ctx, L, rows, hidden, pending, moe_out,
               [&](const float *in, float *out, const NeNormIn *norm_in, const NeNormTail *norm_tail) {
        if (L->full_attention != 0) {
            full_attention_rows(ctx, &L->full, rows, in, out, states, positions, device_positions,
                                span, norm_in, norm_tail);
        } else {
            linear_attention_rows(ctx, &L->linear, rows, in, out, states, norm_in, norm_tail);
        }
    });
}

void prefill_chunk(adi_hip_context *ctx, const adi_hip_decoder_layer *L, uint32_t position,
                   uint32_t count, float *hidden, const float *pending, float *moe_out,
                   const adi_hip_layer_state *state) {
    decoder_chunk_body(ctx, L, position, count, hidden, pending, moe_out, state);
}

}  // namespace adi_hip

using namespace adi_hip;

extern "C" {

int adi_hip_full_attention_forward(adi_hip_context *ctx, const adi_hip_full_attention *L,
                                   uint32_t position, const float *input, float *output,
                                   float *keys, float *values, uint32_t capacity) {
    return guarded(ctx, [&] {
        full_attention_chunk(ctx, L, position, 1, input, output, keys, values, capacity);
    });
}

int adi_hip_full_attention_prefill(adi_hip_context *ctx, const adi_hip_full_attention *L,
                                   uint32_t position, uint32_t count, const float *inputs,
                                   float *outputs, float *keys, float *values, uint32_t capacity) {
    return guarded(ctx, [&] {
        full_attention_chunk(ctx, L, position, count, inputs, outputs, keys, values, capacity);
    });
}

int adi_hip_linear_attention_forward(adi_hip_context *ctx, const adi_hip_linear_attention *L,
                                     const float *input, float *output, float *convolution_state,
                                     float *recurrent_state) {
    return guarded(ctx, [&] {
        linear_attention_chunk(ctx, L, 1, input, output, convolution_state, recurrent_state);
    });
}

int adi_hip_linear_attention_prefill(adi_hip_context *ctx, const adi_hip_linear_attention *L,
                                     uint32_t count, const float *inputs, float *outputs,
                                     float *convolution_state, float *recurrent_state) {
    return guarded(ctx, [&] {
        linear_attention_chunk(ctx, L, count, inputs, outputs, convolution_state, recurrent_state);
    });
}

int adi_hip_decode_layer(adi_hip_context *ctx, const adi_hip_decoder_layer *L, uint32_t position,
                         float *hidden, const adi_hip_layer_state *state) {
    return guarded(ctx, [&] { decoder_chunk(ctx, L, position, 1, hidden, state); });
}

int adi_hip_prefill_layer(adi_hip_context *ctx, const adi_hip_decoder_layer *L, uint32_t position,
                          uint32_t count, float *hidden, const adi_hip_layer_state *state) {
    return guarded(ctx, [&] { decoder_chunk(ctx, L, position, count, hidden, state); });
}

}  // extern "C"
