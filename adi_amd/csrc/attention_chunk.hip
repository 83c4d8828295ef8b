// attention_chunk.hip -- causal grouped attention of a chunk of tokens over
// the key and value caches on the matrix cores (the attention of
// full_attention_forward's prefill, src/executor.cpp:561-731,
// src/attention.cpp), for attentions long enough (attention_chunk_takes).
//
// A block takes 128 query rows of one KV head, 16 tokens times the 8 query
// heads that share it, so every cache entry it stages serves 128 rows; each of
// its 8 waves holds 16 of them (2 tokens) with their 256-wide output in
// registers. Per tile of 32 keys a wave computes S^T = K Q^T (32 keys x 16
// rows), the online softmax of its rows (four lanes hold 8 keys of a row each)
// and O^T += V^T P^T. S^T's register layout is P^T's operand layout but for
// the order of the keys, and the values are staged in that order, so the
// probabilities never leave their lane.
//
// Precision: operands are split so that the matrix cores' 16-bit products add
// up to a float product's accuracy, in float accumulators. Queries and keys
// take two f16 pieces (round to nearest: 22 significant bits and a sign) and
// the three products without lo lo, which is below 2^-22 of a product. f16's
// range is small, so they are scaled first, by an exact power of two for a
// query row and for each four keys (a wave's), to a largest value of 2^14 to
// 2^15, and the scores scaled back: the low pieces' absolute floor of 2^-25 is
// then 2^-39 of the largest. (The scales cost 6 us of 177; unscaled, queries of
// 2^13 over keys of 2^-13 came out 1e-4 off.) Probabilities and values take
// three bf16 pieces that sum to them exactly, at any scale, and the six products
// down to 2^-16; what is left out is below 2^-25 of a product. Against 64 bits
// the layer's output is as far off as with the vector kernel: 1.231e-6 and
// 1.233e-6 for 512 tokens at position 3584, 7.35e-7 and 7.47e-7 for 64 at 1000,
// 8.24e-7 and 8.19e-7 for 128 at 0 (relative, the projections' part included);
// with queries and keys of 2^-30 to 2^30, 64 at 1000 and 256 hidden values, 4.8
// to 6.2e-7 and 4.8 to 6.1e-7.
//
// What bounds it: the matrix cores are busy 45% of the time, the LDS (every
// wave reads every staged entry) 30%, vector issue (the splits, the softmax)
// 45%, in phases between barriers. 512 tokens at position 3584: 177 us, the
// vector kernel 3048 (each query head of each token read the history again).
// Four waves of 32 rows with v_mfma_f32_32x32x16, one a SIMD: 200 us.
//
// A tile with a value the pieces cannot stand for (an infinity, a NaN, 2^60 and
// more in a key or query, whose scores could overflow) runs in plain floats,
// entry by entry, on the same running state: a row skips the entries behind its
// position, which a matrix product multiplies by zero. A query row with a NaN
// is NaN either way and stays on the matrix cores.
#include "attention.hpp"

#include <type_traits>

namespace adi_hip {
namespace {

constexpr uint32_t kHeads = kQueryHeads / kKvHeads;      // query heads of a KV head
constexpr uint32_t kRowTokens = 16;                      // tokens of a block
constexpr uint32_t kThreads = 512;
constexpr uint32_t kWaveTokens = kRowTokens / (kThreads / 64u);
constexpr uint32_t kKeys = 32;                           // keys of a tile
static_assert(kWaveTokens * kHeads == 16, "a wave holds the 16 columns of an MFMA tile");
constexpr uint32_t kKeyPieces = 2;                       // f16
constexpr uint32_t kPieces = 3;                          // bf16
// LDS rows: a key's 256 dimensions and a dimension's 32 keys in bf16 or f16.
// A row's 16-byte pieces are permuted (key_place, value_place) so that the
// lanes of a 16-byte read's phase, 0-3, 12-15 and 20-27 and their like, fall
// on different banks; rows 16 bytes further apart instead left half of the
// LDS's active cycles to conflicts (179 us for 512 tokens at position 3584).
constexpr uint32_t kKeyPitch = kHeadSize * 2;
constexpr uint32_t kValuePitch = kKeys * 2;
constexpr uint32_t kKeyPiece = kKeys * kKeyPitch;
constexpr uint32_t kValuePiece = kHeadSize * kValuePitch;
__device__ __forceinline__ uint32_t key_place(uint32_t row, uint32_t piece) {
    return row * kKeyPitch + ((piece ^ (row & 15u)) << 4);
}
__device__ __forceinline__ uint32_t value_place(uint32_t row, uint32_t piece) {
    return row * kValuePitch + ((piece ^ ((0x78u >> ((row >> 1) & 6u)) & 3u)) << 4);
}
constexpr uint32_t kStaged = kKeyPieces * kKeyPiece + kPieces * kValuePiece;
constexpr uint32_t kChunkLds = kStaged + 16 + kThreads / 64u * 4u;
// the smallest float bits that round to an infinity in bf16, those of 2^60, and
// of infinity
constexpr uint32_t kBf16Overflow = 0x7F7F8000u;
constexpr uint32_t kScoreLimit = (127u + 60u) << 23;
constexpr uint32_t kInfinity = 0x7F800000u;
constexpr uint32_t kNoTile = 0xFFFFFFFFu;

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// Two floats as three packed bf16 pairs whose sums are the floats, exactly.
struct Pieces {
    uint32_t p[kPieces];
};
__device__ __forceinline__ Pieces split_pair(float x, float y) {
    Pieces out;
#pragma unroll
    for (uint32_t i = 0; i < kPieces; ++i) {
        const f32x2 v = {x, y};
        out.p[i] = __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
        x -= __uint_as_float(out.p[i] << 16);
        y -= __uint_as_float(out.p[i] & 0xFFFF0000u);
    }
    return out;
}

// Two floats as two packed f16 pairs.
struct HalfPieces {
    uint32_t hi, lo;
};
__device__ __forceinline__ HalfPieces split_pair_f16(float x, float y) {
    const f32x2 v = {x, y};
    const f16x2 hi = __builtin_convertvector(v, f16x2);
    const f32x2 rest = {x - static_cast<float>(hi.x), y - static_cast<float>(hi.y)};
    return {__builtin_bit_cast(uint32_t, hi), __builtin_bit_cast(uint32_t, __builtin_convertvector(rest, f16x2))};
}

__device__ __forceinline__ f32x4 mfma_f16(u32x4 a, u32x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0,
                                                  0);
}

__device__ __forceinline__ f32x4 mfma(u32x4 a, u32x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c,
                                                   0, 0, 0);
}

// The six piece products of a K = 32 step, smallest first.
__device__ __forceinline__ f32x4 product(const u32x4 (&a)[kPieces], const u32x4 (&b)[kPieces], f32x4 c) {
    c = mfma(a[2], b[0], c);
    c = mfma(a[0], b[2], c);
    c = mfma(a[1], b[1], c);
    c = mfma(a[1], b[0], c);
    c = mfma(a[0], b[1], c);
    return mfma(a[0], b[0], c);
}

struct ChunkArgs {
    const float *query_gate;  // [count][16 heads][256 query, 256 gate], normalized and rotated
    const float *keys, *values;
    uint32_t position, count;
    uint32_t splits;    // of a block's key tiles
    float *partial;     // [count][16][splits][kPartialStride] (splits > 1)
    float *attended;    // [count][16][256] (splits 1)
};

// exp(d) for d <= 0 (or NaN), to about one rounding of the exponential unit:
// 2^(d log2 e) with the product's rounding and the constant's tail put back.
// Results below 2^-126 of the row's largest weight are 0.
__device__ __forceinline__ float weight_of(float d) {
    constexpr float kLog2e = 1.44269502f, kLog2eTail = 1.92596299e-8f, kLn2 = 0.693147182f;
    d = d < -200.0f ? -200.0f : d;
    const float e = d * kLog2e;
    const float tail = fmaf(d, kLog2eTail, fmaf(d, kLog2e, -e));
    const float y = __builtin_amdgcn_exp2f(e);
    return fmaf(y * tail, kLn2, y);
}

// The power of two that brings values of a largest magnitude of these float
// bits (below infinity) to 2^14 .. 2^15, and its inverse; 2^126 at most.
__device__ __forceinline__ uint32_t scale_exponent(uint32_t largest) { return min(268u - (largest >> 23), 253u); }
__device__ __forceinline__ float scale_of(uint32_t exponent) { return __uint_as_float(exponent << 23); }
__device__ __forceinline__ float unscale_of(uint32_t exponent) { return __uint_as_float((254u - exponent) << 23); }

// The largest of the wave's values, a scalar.
__device__ __forceinline__ uint32_t wave_max(uint32_t v) {
    const auto rotated = [](uint32_t x, auto control) {
        return static_cast<uint32_t>(
            __builtin_amdgcn_mov_dpp(static_cast<int>(x), decltype(control)::value, 0xF, 0xF, true));
    };
    v = max(v, rotated(v, std::integral_constant<int, 0x128>{}));  // row_ror:8
    v = max(v, rotated(v, std::integral_constant<int, 0x124>{}));  // row_ror:4
    v = max(v, rotated(v, std::integral_constant<int, 0x122>{}));  // row_ror:2
    v = max(v, rotated(v, std::integral_constant<int, 0x121>{}));  // row_ror:1
    const auto row = [&](int lane) {
        return static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(v), lane));
    };
    return max(max(row(0), row(16)), max(row(32), row(48)));
}

__global__ __launch_bounds__(kThreads, 2) void k_attention_chunk(ChunkArgs args) {
    extern __shared__ __align__(16) unsigned char lds[];
    unsigned char *const key_lds = lds;
    unsigned char *const value_lds = lds + kKeyPieces * kKeyPiece;
    // the last tile with an unsplittable key, and value, and whether a query is
    volatile uint32_t *const odd = reinterpret_cast<volatile uint32_t *>(lds + kStaged);
    // what takes the scores of keys 4 w .. 4 w + 3 back from their scale
    volatile float *const key_unscale = reinterpret_cast<volatile float *>(lds + kStaged + 16);
    // blocks of one (KV head, split) read the same entries: with 8 or more
    // such pairs each stays on one XCD (block b runs on XCD b % 8)
    const uint32_t pairs = kKvHeads * args.splits;
    const uint32_t pair = blockIdx.x % pairs, row_block = blockIdx.x / pairs;
    const uint32_t kv = pair % kKvHeads, split = pair / kKvHeads;
    const auto uniform = [](uint32_t v) {
        return static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(v)));
    };
    // the wave scalar, so that cache rows are addressed by scalar registers
    const uint32_t t = threadIdx.x, lane = t & 63u, wave = uniform(t >> 6);
    const uint32_t quarter = lane >> 4, column = lane & 15u;
    const uint32_t first_token = row_block * kRowTokens;
    const uint32_t wave_token = first_token + wave * kWaveTokens;
    const uint32_t token = min(wave_token + column / kHeads, args.count - 1u);
    const uint32_t head = kv * kHeads + column % kHeads;
    const uint32_t seen = args.position + token;  // the row's last key
    const uint32_t total = args.position + args.count;
    const uint32_t block_keys = args.position + min(first_token + kRowTokens, args.count);
    const uint32_t tiles = (block_keys + kKeys - 1u) / kKeys;
    const uint32_t per_split = (tiles + args.splits - 1u) / args.splits;
    const uint32_t tile0 = min(split * per_split, tiles), tile_end = min(tile0 + per_split, tiles);
    const float *const query = args.query_gate + (static_cast<size_t>(token) * kQueryHeads + head) * 2u * kHeadSize;
    const float *const keys = args.keys + kv * kHeadSize;
    const float *const values = args.values + kv * kHeadSize;
    const auto largest = [](uint32_t m, const float4 &v) {
        const uint32_t a = max(__float_as_uint(v.x) & 0x7FFFFFFFu, __float_as_uint(v.y) & 0x7FFFFFFFu);
        const uint32_t b = max(__float_as_uint(v.z) & 0x7FFFFFFFu, __float_as_uint(v.w) & 0x7FFFFFFFu);
        return max(m, max(a, b));
    };
    if (t < 3u) {
        odd[t] = kNoTile;
    }
    // A tile's entries pass through registers, each wave four key rows and
    // four value rows (4 wave + 0 .. 3), lane l dimensions 4 l .. 4 l + 3.
    // Rows past the chunk's last entry repeat it (behind every row's
    // position, so of weight 0).
    float4 key_in[4], value_in[4];
    const auto entry = [&](const float *cache, uint32_t key) {
        return reinterpret_cast<const float4 *>(cache + static_cast<size_t>(min(key, total - 1u)) * kKvHeads *
                                                            kHeadSize)[lane];
    };
    // the largest of the wave's four keys of a tile, and what takes its scale
    // back into LDS
    const auto largest_key = [&] {
        uint32_t big = 0;
#pragma unroll
        for (uint32_t u = 0; u < 4u; ++u) {
            big = largest(big, key_in[u]);
        }
        big = wave_max(big);
        key_unscale[wave] = unscale_of(scale_exponent(min(big, kScoreLimit)));
        return big;
    };
    const auto key_scale = [](uint32_t big) { return scale_of(scale_exponent(min(big, kScoreLimit))); };
    // key row 4 wave + u into LDS
    const auto stage_key = [&](uint32_t u, float scale) {
        const HalfPieces a = split_pair_f16(key_in[u].x * scale, key_in[u].y * scale);
        const HalfPieces b = split_pair_f16(key_in[u].z * scale, key_in[u].w * scale);
        unsigned char *to = key_lds + key_place(4u * wave + u, lane >> 1) + 8u * (lane & 1u);
        *reinterpret_cast<uint2 *>(to) = make_uint2(a.hi, b.hi);
        *reinterpret_cast<uint2 *>(to + kKeyPiece) = make_uint2(a.lo, b.lo);
    };
    // dimension 4 lane + d of the wave's four values into row 64 d + lane, at
    // the place of P^T's key order: keys 4 q .. 4 q + 3 and 16 + 4 q .. are
    // the eight of quarter q
    const auto stage_value = [&](uint32_t d) {
        const auto of = [&](uint32_t k) {
            const float4 &v = value_in[k];
            return d == 0 ? v.x : d == 1 ? v.y : d == 2 ? v.z : v.w;
        };
        const Pieces a = split_pair(of(0), of(1)), b = split_pair(of(2), of(3));
        unsigned char *to = value_lds + value_place(64u * d + lane, wave & 3u) + 8u * (wave >> 2);
#pragma unroll
        for (uint32_t k = 0; k < kPieces; ++k) {
            *reinterpret_cast<uint2 *>(to + k * kValuePiece) = make_uint2(a.p[k], b.p[k]);
        }
    };

    f32x4 out[16];
#pragma unroll
    for (uint32_t i = 0; i < 16u; ++i) {
        out[i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    }
    float maximum = -__builtin_huge_valf(), denominator = 0.0f;

    // A tile in floats: its entries to LDS (read again, so that none is held
    // through the products), then four at a time: a lane adds the products of its quarter of the row's
    // query (as q holds the dimensions), every quarter then has the row's
    // scores, and takes its 64 dimensions of the output through the online steps
    // of update_online_softmax (src/attention.cpp:15-35). The row's denominator
    // is the sum of its four lanes'. Some 30 us a tile, which the vector kernel
    // takes 100 for on a full chip, and 8 where every row of the wave is a NaN
    // already: nothing changes those.
    const auto tile_in_floats = [&](uint32_t key0) {
        float4 row_query[8][2];
#pragma unroll
        for (uint32_t s = 0; s < 8u; ++s) {
            const float4 *from = reinterpret_cast<const float4 *>(query + 32u * s + 8u * quarter);
            row_query[s][0] = from[0];
            row_query[s][1] = from[1];
        }
        float4 *const key_rows = reinterpret_cast<float4 *>(key_lds);
        float4 *const value_rows = reinterpret_cast<float4 *>(value_lds);
        constexpr uint32_t kRow = kHeadSize / 4u;
#pragma unroll
        for (uint32_t u = 0; u < 4u; ++u) {
            key_rows[(4u * wave + u) * kRow + lane] = entry(keys, key0 + 4u * wave + u);
            value_rows[(4u * wave + u) * kRow + lane] = entry(values, key0 + 4u * wave + u);
        }
        __syncthreads();
        // (a wave whose tokens all come before the tile has none)
        const uint32_t past = min(args.position + wave_token + kWaveTokens, total);
        const uint32_t end = past > key0 ? min(kKeys, past - key0) : 0u;
#pragma unroll 1
        for (uint32_t k0 = 0; k0 < end && !__all(denominator != denominator); k0 += 4u) {
            float dot[4];
#pragma unroll
            for (uint32_t u = 0; u < 4u; ++u) {
                const float4 *key = key_rows + (k0 + u) * kRow + 2u * quarter;
                float sum[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (uint32_t s = 0; s < 8u; ++s) {
#pragma unroll
                    for (uint32_t h = 0; h < 2u; ++h) {
                        const float4 a = row_query[s][h], b = key[8u * s + h];
                        sum[0] += a.x * b.x;
                        sum[1] += a.y * b.y;
                        sum[2] += a.z * b.z;
                        sum[3] += a.w * b.w;
                    }
                }
                dot[u] = (sum[0] + sum[1]) + (sum[2] + sum[3]);
            }
#pragma unroll
            for (uint32_t u = 0; u < 4u; ++u) {
                dot[u] += lane_xor<16>(dot[u]);
                dot[u] += lane_xor<32>(dot[u]);
            }
#pragma unroll
            for (uint32_t u = 0; u < 4u; ++u) {
                if (key0 + k0 + u <= seen) {
                    const float4 *value = value_rows + (k0 + u) * kRow + 4u * quarter;
                    const float score = dot[u] * 0.0625f;
                    const bool up = !(score <= maximum);
                    if (__any(up)) {
                        const float previous = up ? expf(maximum - score) : 1.0f;
                        maximum = up ? score : maximum;
                        denominator *= previous;
#pragma unroll
                        for (uint32_t i = 0; i < 16u; ++i) {
                            out[i] *= previous;
                        }
                    }
                    const float weight = up ? 1.0f : expf(score - maximum);
                    denominator += quarter == 0 ? weight : 0.0f;
#pragma unroll
                    for (uint32_t i = 0; i < 4u; ++i) {
#pragma unroll
                        for (uint32_t r = 0; r < 4u; ++r) {
                            const float4 v = value[16u * i + r];
                            out[i][r] += v.x * weight;
                            out[i + 4u][r] += v.y * weight;
                            out[i + 8u][r] += v.z * weight;
                            out[i + 12u][r] += v.w * weight;
                        }
                    }
                }
            }
        }
    };

    // runs of tiles on the matrix cores, each up to a tile that is not for them
    uint32_t tile = tile0;
    while (tile < tile_end) {
        // the row's query in pieces: step s holds dimensions 32 s + 8 quarter +
        // 0 .. 7
        u32x4 q[8][kKeyPieces];
        uint32_t big_query = 0;
        float4 query_in[8][2];
#pragma unroll
        for (uint32_t s = 0; s < 8u; ++s) {
            const float4 *from = reinterpret_cast<const float4 *>(query + 32u * s + 8u * quarter);
            query_in[s][0] = from[0];
            query_in[s][1] = from[1];
            big_query = largest(largest(big_query, query_in[s][0]), query_in[s][1]);
        }
        big_query = max(big_query, lane_xor_bits<16>(big_query));
        big_query = max(big_query, lane_xor_bits<32>(big_query));
        const uint32_t query_exponent = scale_exponent(min(big_query, kScoreLimit));
        const float query_scale = scale_of(query_exponent);
        // with 1 / sqrt(256)
        const float query_unscale = unscale_of(query_exponent) * 0.0625f;
#pragma unroll
        for (uint32_t s = 0; s < 8u; ++s) {
            const float4 a = query_in[s][0], b = query_in[s][1];
            const HalfPieces c0 = split_pair_f16(a.x * query_scale, a.y * query_scale);
            const HalfPieces c1 = split_pair_f16(a.z * query_scale, a.w * query_scale);
            const HalfPieces c2 = split_pair_f16(b.x * query_scale, b.y * query_scale);
            const HalfPieces c3 = split_pair_f16(b.z * query_scale, b.w * query_scale);
            q[s][0] = u32x4{c0.hi, c1.hi, c2.hi, c3.hi};
            q[s][1] = u32x4{c0.lo, c1.lo, c2.lo, c3.lo};
        }
#pragma unroll
        for (uint32_t u = 0; u < 4u; ++u) {
            key_in[u] = entry(keys, tile * kKeys + 4u * wave + u);
        }
#pragma unroll
        for (uint32_t u = 0; u < 4u; ++u) {
            value_in[u] = entry(values, tile * kKeys + 4u * wave + u);
        }
        __syncthreads();  // odd[] is set
        if (big_query >= kScoreLimit && big_query <= kInfinity) {
            odd[2] = 0;
        }
        const uint32_t first_key = largest_key();
#pragma unroll
        for (uint32_t u = 0; u < 4u; ++u) {
            stage_key(u, key_scale(first_key));
        }
        if (first_key >= kScoreLimit) {
            odd[0] = tile;
        }
        for (; tile < tile_end; ++tile) {
            const uint32_t key0 = tile * kKeys;
            __syncthreads();  // the tile's keys are staged; the last tile's values are free
            // the scores, this tile's values staged between their products
            const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
            // three sums a score (the small products, the large of even and of
            // odd steps): fewer roundings at its full size
            f32x4 small[2] = {zero, zero}, large[2][2] = {{zero, zero}, {zero, zero}};
            uint32_t big = 0;
#pragma unroll
            for (uint32_t s = 0; s < 8u; ++s) {
#pragma unroll
                for (uint32_t m = 0; m < 2u; ++m) {
                    const unsigned char *from = key_lds + key_place(16u * m + column, 4u * s + quarter);
                    const u32x4 hi = *reinterpret_cast<const u32x4 *>(from);
                    const u32x4 lo = *reinterpret_cast<const u32x4 *>(from + kKeyPiece);
                    small[m] = mfma_f16(lo, q[s][0], small[m]);
                    small[m] = mfma_f16(hi, q[s][1], small[m]);
                    large[m][s & 1u] = mfma_f16(hi, q[s][0], large[m][s & 1u]);
                }
                if ((s & 1u) == 0) {
                    big = largest(big, value_in[s >> 1]);
                    stage_value(s >> 1);
                }
            }
            if (big >= kBf16Overflow) {
                odd[1] = tile;
            }
            const bool odd_keys = uniform(odd[0]) == tile || uniform(odd[2]) == 0;
            const float unscale[2] = {key_unscale[quarter], key_unscale[4u + quarter]};
            __syncthreads();  // the tile's values are staged; its keys are free
            if (__builtin_expect(odd_keys || uniform(odd[1]) == tile, 0)) {  // the same for every wave
                break;
            }
            // the next tile's keys load under the softmax
#pragma unroll
            for (uint32_t u = 0; u < 4u; ++u) {
                key_in[u] = entry(keys, key0 + kKeys + 4u * wave + u);
            }
            // score[m][r] is key key0 + 16 m + 4 quarter + r
            f32x4 score[2];
            score[0] = ((large[0][0] + large[0][1]) + small[0]) * (query_unscale * unscale[0]);
            score[1] = ((large[1][0] + large[1][1]) + small[1]) * (query_unscale * unscale[1]);
            if (key0 + kKeys > args.position + wave_token + 1u) {  // some row of the wave ends before the tile does
#pragma unroll
                for (uint32_t r = 0; r < 8u; ++r) {
                    const uint32_t key = key0 + 16u * (r >> 2) + 4u * quarter + (r & 3u);
                    score[r >> 2][r & 3u] = key <= seen ? score[r >> 2][r & 3u] : -__builtin_huge_valf();
                }
            }
            float top = fmaxf(fmaxf(fmaxf(score[0][0], score[0][1]), fmaxf(score[0][2], score[0][3])),
                              fmaxf(fmaxf(score[1][0], score[1][1]), fmaxf(score[1][2], score[1][3])));
            top = fmaxf(top, lane_xor<16>(top));
            top = fmaxf(fmaxf(top, lane_xor<32>(top)), maximum);
            if (__any(top > maximum)) {
                const float factor = maximum == top ? 1.0f : expf(maximum - top);
                denominator *= factor;
#pragma unroll
                for (uint32_t i = 0; i < 16u; ++i) {
#pragma unroll
                    for (uint32_t r = 0; r < 4u; ++r) {
                        out[i][r] *= factor;
                    }
                }
                maximum = top;
            }
            // a row with no key yet has maximum -infinity: its weights are 0
            const float base = maximum == -__builtin_huge_valf() ? 0.0f : maximum;
            float weight[8];
#pragma unroll
            for (uint32_t r = 0; r < 8u; ++r) {
                const float s = score[r >> 2][r & 3u];
                weight[r] = weight_of(s == base ? 0.0f : s - base);
            }
            denominator += ((weight[0] + weight[1]) + (weight[2] + weight[3])) +
                           ((weight[4] + weight[5]) + (weight[6] + weight[7]));
            // the next tile's values load under this tile's, its keys are staged
            // between the products
#pragma unroll
            for (uint32_t u = 0; u < 4u; ++u) {
                value_in[u] = entry(values, key0 + kKeys + 4u * wave + u);
            }
            u32x4 p[kPieces];
            {
                const Pieces c0 = split_pair(weight[0], weight[1]), c1 = split_pair(weight[2], weight[3]);
                const Pieces c2 = split_pair(weight[4], weight[5]), c3 = split_pair(weight[6], weight[7]);
#pragma unroll
                for (uint32_t i = 0; i < kPieces; ++i) {
                    p[i] = u32x4{c0.p[i], c1.p[i], c2.p[i], c3.p[i]};
                }
            }
            uint32_t next_key = 0;
#pragma unroll
            for (uint32_t i = 0; i < 16u; ++i) {
                u32x4 v[kPieces];
#pragma unroll
                for (uint32_t k = 0; k < kPieces; ++k) {
                    v[k] = *reinterpret_cast<const u32x4 *>(value_lds + k * kValuePiece +
                                                            value_place(16u * i + column, quarter));
                }
                out[i] = product(v, p, out[i]);
                if (i == 0) {
                    next_key = largest_key();
                }
                if ((i & 3u) == 0) {
                    stage_key(i >> 2, key_scale(next_key));
                }
            }
            if (next_key >= kScoreLimit) {
                odd[0] = tile + 1u;
            }
        }
        if (__builtin_expect(tile < tile_end, 0)) {
            tile_in_floats(tile * kKeys);
            ++tile;
        }
    }
    denominator += lane_xor<16>(denominator);
    denominator += lane_xor<32>(denominator);
    if (wave_token + column / kHeads >= args.count) {
        return;
    }
    // out[i][r], row 16 i + 4 quarter + r of the staged values, is dimension
    // 4 (row % 64) + row / 64: i, i + 4, i + 8 and i + 12 hold four
    // consecutive dimensions
    const size_t row = static_cast<size_t>(token) * kQueryHeads + head;
    if (args.splits == 1u) {
        const float inverse = 1.0f / denominator;
        const float4 *gate = reinterpret_cast<const float4 *>(query + kHeadSize);
        float4 *to = reinterpret_cast<float4 *>(args.attended + row * kHeadSize);
#pragma unroll
        for (uint32_t i = 0; i < 4u; ++i) {
#pragma unroll
            for (uint32_t r = 0; r < 4u; ++r) {
                const uint32_t at = 16u * i + 4u * quarter + r;
                const float4 g = gate[at];
                to[at] = make_float4(out[i][r] * inverse * sigmoid_of(g.x), out[i + 4u][r] * inverse * sigmoid_of(g.y),
                                     out[i + 8u][r] * inverse * sigmoid_of(g.z),
                                     out[i + 12u][r] * inverse * sigmoid_of(g.w));
            }
        }
        return;
    }
    float *to = args.partial + (row * args.splits + split) * kPartialStride;
#pragma unroll
    for (uint32_t i = 0; i < 4u; ++i) {
#pragma unroll
        for (uint32_t r = 0; r < 4u; ++r) {
            float2 *pair_to = reinterpret_cast<float2 *>(to + 4u * (16u * i + 4u * quarter + r));
            pair_to[0] = make_float2(out[i][r], out[i + 4u][r]);
            pair_to[1] = make_float2(out[i + 8u][r], out[i + 12u][r]);
        }
    }
    if (quarter == 0) {
        to[kHeadSize] = maximum;
        to[kHeadSize + 1u] = denominator;
    }
}

}  // namespace

// A launch costs some 25 us before its first tile (its queries, its code), so
// short attentions stay with the vector kernel, 2.2 us per 1000 (token, key)
// pairs. Both kernels, us, with their combines: 128 tokens at position 0 (8,000
// pairs) 26 there, 34 here; 32 tokens at 500 and 16 at 1000 (16,000) 37 and
// 36, 37 and 33 here; 256 tokens at 0 (33,000) 68 and 38; 512 at 3584 3065 and
// 196. Fewer tokens than a block has were not compared and stay there.
bool attention_chunk_takes(uint32_t position, uint32_t count) {
    return count >= kRowTokens && size_t(count) * (size_t(position) + count / 2u) >= 16384u;
}

uint32_t attention_chunk_splits(uint32_t position, uint32_t count, size_t free_bytes) {
    // a block a CU (its registers fill one), each with two key tiles or more
    const uint32_t blocks = ceil_div(count, kRowTokens) * kKvHeads;
    const uint32_t tiles = ceil_div(size_t(position) + count, kKeys);
    uint32_t splits = 1;
    while (splits < kMaxSplits && blocks * splits * 2u <= 256u && tiles >= splits * 4u &&
           Workspace::round(size_t(count) * kQueryHeads * splits * 2u * kPartialStride * 4u) <= free_bytes) {
        splits *= 2u;
    }
    return splits;
}

void launch_attention_chunk(adi_hip_context *ctx, const float *query_gate, const float *keys, const float *values,
                            uint32_t position, uint32_t count, uint32_t splits, float *partial, float *attended) {
    static const bool raised = set_lds_limit(reinterpret_cast<const void *>(k_attention_chunk), kChunkLds);
    (void)raised;
    const ChunkArgs args{query_gate, keys, values, position, count, splits, partial, attended};
    launch(ctx, "attention_chunk", k_attention_chunk, dim3(ceil_div(count, kRowTokens) * kKvHeads * splits), dim3(kThreads),
           kChunkLds, args);
}

}  // namespace adi_hip
