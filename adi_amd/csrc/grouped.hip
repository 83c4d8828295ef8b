// grouped.hip -- MFMA grouped GEMMs for prefill microbatches
// (src/kernels.cpp:491-593, 703-800 with the batch kernels of
// src/expert_batch_impl.hpp and src/ne_batch_impl.hpp): the codes are decoded
// straight into the A operand of v_mfma_f32_32x32x16_f16, x_hat is the B
// operand as f16 hi/lo pairs staged once per block in LDS, accumulation is
// fp32.
//
// Expert codec. The K axis is laid out as the eight columns a codebook plane
// covers in each tile (XhatOut planes 2), so a lane's eight K values are the
// two half-states of one tile row: two gathers from the block's LDS plane.
// The wave gamma of a tile is folded into A in f16: hi = f16(gamma * V),
// lo = f16(gamma * V - hi) (one packed f16 multiply and one packed f16 fma;
// gamma and V are f16, so the product has at most 22 significant bits and
// hi + lo holds it). Three MFMA passes, hi*hi + hi*lo + lo*hi, keep the error
// near fp32 rounding.
//
// NE codec. The 4 KiB signed table gives V exactly in f16 (Wscale is applied
// to the fp32 row sums); two passes, V*hi + V*lo.
#include "grouped.hpp"

#include <type_traits>

namespace adi_hip {
namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// expert GEMM shape: 32 positions per item, tile rows kExpertRT per wave,
// 512 * kExpertGroups threads per block (one block per CU), MFMA passes per
// product (hi*hi + hi*lo + lo*hi)
constexpr int kExpertRT = 4;
constexpr int kExpertCB = 2;      // blocks of 32 positions per item (the later one may be empty)
constexpr int kExpertGroups = 1;  // wave groups of eight per block, each on its own item
constexpr int kExpertPasses = 3;
constexpr uint32_t kPlaneRows16 = kExpertRows * 8 / 16;   // 16-byte rows of a plane
constexpr uint32_t kSlotCapacity = 1024;

// The 16-bit window at bit r (r <= 48) of the 64-bit string of u16 words
// w0 w1 w2 w3, each read most-significant bit first, where d0 = w0 | w1 << 16
// and d1 = w2 | w3 << 16 (src/expert_trellis.hpp:81-105).
__device__ __forceinline__ uint32_t window64(uint32_t d0, uint32_t d1, uint32_t r) {
    const uint64_t bits = (static_cast<uint64_t>(d0 & 0xFFFFu) << 48) |
                          (static_cast<uint64_t>(d0 >> 16) << 32) |
                          (static_cast<uint64_t>(d1 & 0xFFFFu) << 16) | (d1 >> 16);
    return static_cast<uint32_t>(bits >> (48u - r)) & 0xFFFFu;
}

// w (w + 1) mod 2^16 in bits 0..15 for any 32-bit w whose low 16 bits are
// the state: v_mad_u32_u24 reads 24 bits of each factor, and the bits above
// bit 15 only add multiples of 2^16 (the compiler would otherwise pick the
// quarter-rate v_mad_u64_u32 for the unmasked product).
__device__ __forceinline__ uint32_t state_hash_low16(uint32_t w) {
    uint32_t p;
    asm("v_mad_u32_u24 %0, %1, %1, %1" : "=v"(p) : "v"(w));
    return p;
}

// ---- expert ---------------------------------------------------------------
//
// v_mfma_f32_32x32x16_f16 (on the box 1.6x the f16 rate of 16x16x32): lane l
// holds A[l % 32][8 (l / 32) .. + 7], B[8 (l / 32) .. + 7][l % 32], and D
// column l % 32, rows (r % 4) + 8 (r / 4) + 4 (l / 32) of register r.
//
// An item is one routed slot's 32 positions times 32 tile rows of one entry.
// A block runs kExpertGroups wave groups of eight, each on its own item; wave
// w of a group takes tile rows 4w .. 4w + 3 of it as two 32-row blocks. Lane
// l holds row l % 16 of tile row 2 rb + (l % 32) / 16 of its block rb, and of
// K pair c at K step kc the tile column 4 kc + 2 c + l / 32: its eight K
// values (in the codebook-plane order of XhatOut planes 2) are the two
// half-states of that row, two gathers from the LDS plane. A group loads each
// K step's x_hat hi and lo of its positions once into its LDS ring that its
// eight waves read; the block takes one barrier per K step (all items of a
// launch have the same K). Each wave loads its own trellis words, four K
// steps ahead.

constexpr uint32_t kBlockTileRows = kExpertRT * 8;  // tile rows of an item (a wave group's share)
constexpr uint32_t kBRowPitch = 80;  // bytes per B row in LDS: 64 of data, 16 of pad (no bank conflicts)
constexpr uint32_t kGammaRow = kMaxTileColumns + kBlockTileRows;  // halves per gamma row
constexpr int kFragments = 4;  // A fragments per K step: (row block, K pair)

typedef float f32x16 __attribute__((ext_vector_type(16)));

__device__ __forceinline__ f32x16 mfma32(half8 a, half8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}

// A buffer resource over `bytes` bytes at `base`: loads past the end return 0.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_over(const void *base, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), 0, bytes, 0x00020000);
}

// The trellis words of the lane's four tiles (fragment f = 2 rb + c) at one K
// step: its two stream dwords (row 15: dwords 10 and 11).
struct ExpertWords {
    uint2 w[kFragments];
};

// The byte selectors of a lane's 28-bit string (its states 2 trow and 2 trow +
// 1) in its two dwords, and of row 15's last byte in the tile's first dword.
struct ExpertString {
    uint32_t bytes, last;
};

// The selectors of tile row trow: its string starts at bit 24 trow of the
// tile's stream, a whole byte, so one v_perm_b32 takes its four bytes from two
// dwords (u16 words most significant byte first) and puts them in order. Row
// 15's string ends in the tile's first byte (src/expert_trellis.hpp:79-80).
__device__ __forceinline__ ExpertString expert_string(uint32_t trow) {
    constexpr uint32_t kOrder = 0x67452301u;  // nibble j: where stream byte j of the two dwords lies
    const uint32_t k = trow == 15u ? 5u : 3u * trow & 3u;
    ExpertString out{0u, trow == 15u ? 0x07060501u : 0x07060504u};
    for (uint32_t j = 0; j < 4u; ++j) {
        out.bytes = out.bytes << 8 | (k + j < 8u ? kOrder >> 4u * (k + j) & 15u : 0x0Cu);
    }
    return out;
}

// The first of the two dwords a lane of tile row trow loads (row 15: 10, with
// 11; its last byte comes from lane 0 of its row).
__device__ __forceinline__ uint32_t expert_dwords(uint32_t trow) { return trow == 15u ? 10u : (24u * trow) >> 5; }

// Everything about a wave's share of an item that does not change along K:
// per-lane byte offsets (a K step advances the scalar offset only), the
// lane's byte selectors and its gamma row in LDS.
struct ExpertWave {
    __amdgpu_buffer_rsrc_t words;
    uint32_t woff[kFragments];  // the lane's stream dword pair of fragment f at K step 0
    const uint2 *gammas;        // gamma row tsub + kh of the item, at the wave's first tile row
    ExpertString string;
};

__device__ __forceinline__ void expert_words(const ExpertWave &wv, uint32_t kc, ExpertWords &s) {
    const uint32_t kw = kc * 192u;  // 4 tiles of 48 bytes per K step
#pragma unroll
    for (int f = 0; f < kFragments; ++f) {
        s.w[f] = __builtin_bit_cast(uint2, __builtin_amdgcn_raw_buffer_load_b64(wv.words, wv.woff[f], kw, 0));
    }
}

// The lane's A fragments at one K step: hi = f16(gamma * V) and
// lo = f16(gamma * V - hi).
struct ExpertA {
    half8 hi[kFragments], lo[kFragments];
};

// The lane's two half-states of a tile row: their hashes (bit 15 negates
// component 0) and codebook entries.
struct ExpertEntries {
    uint32_t p0, p1;
    uint2 e0, e1;
};

__device__ __forceinline__ ExpertEntries expert_gather(ExpertString at, uint2 words, const uint2 *plane) {
    // row 15's last byte is in dword 0 of its tile, which lane 0 of the same
    // 16-lane row (the same tile) loaded first (row_ror:15 reads lane (i + 1)
    // mod 16)
    const uint32_t wrap = __builtin_amdgcn_update_dpp(0u, words.x, 0x12F, 0xF, 0xF, false);
    const uint32_t most = __builtin_amdgcn_perm(words.y, words.x, at.bytes);
    const uint32_t string = __builtin_amdgcn_perm(most, wrap, at.last);
    ExpertEntries out;
    out.p0 = state_hash_low16(string >> 16);
    out.p1 = state_hash_low16(string >> 4);
    out.e0 = plane[(out.p0 >> 1) & 0x3FFFu];
    out.e1 = plane[(out.p1 >> 1) & 0x3FFFu];
    return out;
}

// The lane's eight values times the tile's gamma, as hi + lo.
template <int PASSES>
__device__ __forceinline__ void expert_scale(const ExpertEntries &in, uint32_t gamma, uint32_t sign_mask, half8 &hi,
                                             half8 &lo) {
#pragma clang fp contract(off)
    const half8 v = __builtin_bit_cast(half8, u32x4{in.e0.x ^ (in.p0 & sign_mask), in.e0.y,
                                                    in.e1.x ^ (in.p1 & sign_mask), in.e1.y});
    const _Float16 g = __builtin_bit_cast(_Float16, static_cast<uint16_t>(gamma));
    const half8 gv = {g, g, g, g, g, g, g, g};
    hi = gv * v;
    if constexpr (PASSES == 3) {
        lo = __builtin_elementwise_fma(gv, v, -hi);
    }
}

// Decodes the lane's A fragments at K step kc (lo only when PASSES is 3).
template <int PASSES>
__device__ __forceinline__ void expert_decode(const ExpertWave &wv, uint32_t kc, uint32_t sign_mask,
                                              const uint2 *plane, const ExpertWords &s, ExpertA &a) {
    // gammas of the lane's tiles: fragment (rb, c) sits 2 rb + 2 c anti-diagonals
    // past the lane's first, so offsets 0, 2, 2, 4 of the lane's gamma row
    const uint2 g03 = wv.gammas[kc];
    const uint2 g47 = wv.gammas[kc + 1];
    const uint32_t gbits[kFragments] = {g03.x & 0xFFFFu, g03.y & 0xFFFFu, g03.y & 0xFFFFu, g47.x & 0xFFFFu};
#pragma unroll
    for (int f = 0; f < kFragments; ++f) {
        expert_scale<PASSES>(expert_gather(wv.string, s.w[f], plane), gbits[f], sign_mask, a.hi[f], a.lo[f]);
    }
}

// acc[rb][cb] += hi * bh + hi * bl + lo * bh over the two K pairs, for the
// item's first LIVE of its CB blocks of 32 positions (lo only when PASSES is
// 3). Positions past the slot in a live block carry another slot's x_hat:
// their output columns are computed and never stored.
template <int CB, int LIVE, int PASSES>
__device__ __forceinline__ void expert_multiply(const ExpertA &a, const half8 (&bh)[CB][2],
                                                const half8 (&bl)[CB][2], f32x16 (&acc)[2][CB]) {
    static_assert(LIVE >= 1 && LIVE <= CB, "live blocks of an item");
#pragma unroll
    for (int rb = 0; rb < 2; ++rb) {
#pragma unroll
        for (int cb = 0; cb < LIVE; ++cb) {
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                acc[rb][cb] = mfma32(a.hi[2 * rb + c], bh[cb][c], acc[rb][cb]);
            }
        }
    }
#pragma unroll
    for (int rb = 0; rb < 2; ++rb) {
#pragma unroll
        for (int cb = 0; cb < LIVE; ++cb) {
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                acc[rb][cb] = mfma32(a.hi[2 * rb + c], bl[cb][c], acc[rb][cb]);
            }
        }
    }
    if constexpr (PASSES == 3) {
#pragma unroll
        for (int rb = 0; rb < 2; ++rb) {
#pragma unroll
            for (int cb = 0; cb < LIVE; ++cb) {
#pragma unroll
                for (int c = 0; c < 2; ++c) {
                    acc[rb][cb] = mfma32(a.lo[2 * rb + c], bh[cb][c], acc[rb][cb]);
                }
            }
        }
    }
}

// ---- slots of at most 16 positions -------------------------------------------
//
// Most slots of a decode batch or of a default prefill micro-batch hold one to
// eight positions, where an item's time is its decode and the latency of each
// K step. Here a unit is one slot times four tile rows of one entry, run by
// one wave on its own with v_mfma_f32_16x16x32_f16 (sixteen columns, half the
// matrix time of the 32-column form): no block barrier, so the waves of a SIMD
// fill each other's waits, and the last units spread one to a CU. Lane l holds
// row l % 16 of a tile row and, at K step kc, tile column 4 kc + l / 16. A
// wave reads its x_hat columns from memory itself (2 KB a K step), loads four
// K steps ahead straight across units, and gathers the codebook entries of the
// next K step before it multiplies this one's. Both launches of a layer of 256
// experts: 45 tokens (1.8 positions a slot) 154 -> 108 us, 128 tokens with
// uniform routes (4 a slot) 204 -> 142, 128 with skewed ones 81 -> 77; what
// bounds it now is vector issue, about 100 instructions a K step and wave.
// Slots of 17 positions or more fill a 32-column item's matrix time and share
// its x_hat, so they stay block items.

constexpr uint32_t kSmallPositions = 16;
constexpr uint32_t kSmallTileColumns = 128;  // the widest matrix whose gamma rows fit the ring's LDS
// a unit's gamma rows, twice: entry i of row q is the gamma at anti-diagonal
// i + q past the unit's first tile row
constexpr uint32_t kSmallGammaRow = kSmallTileColumns / 4u + 1u;  // uint2 of four halves
constexpr uint32_t kSmallGammas = 2u * 4u * kSmallGammaRow;       // uint2 per wave

__host__ __device__ inline bool small_slots_supported(uint32_t tile_columns) {
    return tile_columns >= 16u && tile_columns <= kSmallTileColumns;  // whole groups of four K steps
}

struct SmallUnit {
    __amdgpu_buffer_rsrc_t words, x_hi, x_lo, gamma;
    float *z;            // of the unit's first position
    uint32_t x_off;      // the lane's x_hat row and K offset
    uint32_t tile_row;   // the unit's first
    uint32_t positions;
};

template <int PASSES>
__device__ __forceinline__ void expert_small_slots(const ExpertMfmaJobs &J, uint32_t half, uint32_t first_unit,
                                                   uint32_t second_unit, uint32_t stride, const uint2 *plane,
                                                   const uint16_t *slots, uint32_t slot_count, uint2 *gammas) {
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t column = lane & 15u, kq = lane >> 4;
    const uint32_t rows = J.expert[0].rows, tile_rows = J.expert[0].tile_rows, tc_shift = J.expert[0].tc_shift;
    const uint32_t tile_columns = 1u << tc_shift, steps = tile_columns / 4u;
    const uint32_t parts = (tile_rows + 3u) / 4u;
    const uint32_t units = slot_count * J.expert_count * parts;
    const uint32_t sign_mask = half == 0 ? 0x8000u : 0u;
    const ExpertString string = expert_string(column);
    const uint32_t lane_words = (kq * 12u + expert_dwords(column)) * 4u;
    if (first_unit >= units) {
        return;
    }
    const auto open = [&](uint32_t unit) {
        const uint32_t part = unit % parts, entry = unit / parts;
        const ExpertMfma &a = J.expert[entry % J.expert_count];
        const uint32_t slot = __builtin_amdgcn_readfirstlane(slots[entry / J.expert_count]);
        const uint4 info = J.slot_info != nullptr ? J.slot_info[slot] : make_uint4(0u, 0u, J.max_positions, 0u);
        const uint32_t mat = __builtin_amdgcn_readfirstlane(info.x);
        const uint32_t first = __builtin_amdgcn_readfirstlane(info.y);
        const uint32_t positions = __builtin_amdgcn_readfirstlane(info.z) - first;
        const uint32_t half_columns = a.columns >> 1;
        const size_t plane_elems = static_cast<size_t>(a.positions) * half_columns;
        SmallUnit out;
        out.words = buffer_over(a.trellis + mat * a.trellis_stride, (tile_rows << tc_shift) * 48u);
        out.x_hi = buffer_over(a.x_hi + half * plane_elems, static_cast<uint32_t>(plane_elems * 2u));
        out.x_lo = buffer_over(a.x_lo + half * plane_elems, static_cast<uint32_t>(plane_elems * 2u));
        out.gamma = buffer_over(a.gamma + mat * a.gamma_stride, (tile_rows + tile_columns) * 2u);
        out.z = a.z + half * a.z_split_stride + static_cast<size_t>(first) * rows;
        // columns past the slot repeat its last position and are never stored
        out.x_off = ((first + min(column, positions - 1u)) * half_columns + 8u * kq) * 2u;
        out.tile_row = 4u * part;
        out.positions = positions;
        return out;
    };
    // the gamma of anti-diagonal tile_row + e in slot R_t + C_t - 1 - d, one
    // less past the main anti-diagonal (src/codec_cache.cpp:117-147); past the
    // matrix 0, for tiles that are never stored
    const auto load_gamma = [&](const SmallUnit &u, uint32_t e) {
        const uint32_t d = u.tile_row + e;
        const uint32_t slot = tile_rows + tile_columns - 1u - d - (d >= tile_columns ? 1u : 0u);
        return static_cast<uint32_t>(__builtin_amdgcn_raw_buffer_load_b16(u.gamma, slot * 2u, 0, 0));
    };
    const auto store_gamma = [&](uint2 *to, uint32_t e, uint32_t g) {
        uint16_t *row = reinterpret_cast<uint16_t *>(to);
#pragma unroll
        for (uint32_t q = 0; q < 4u; ++q) {
            if (e - q < 4u * kSmallGammaRow) {  // e < q wraps: out of range
                row[q * 4u * kSmallGammaRow + e - q] = static_cast<uint16_t>(g);
            }
        }
    };
    // a unit's gamma rows: written by every lane as halves, read by others in
    // fours
    const auto store_gammas = [&](uint2 *to, uint32_t a, uint32_t b, uint32_t c) {
        store_gamma(to, lane, a);
        store_gamma(to, lane + 64u, b);
        store_gamma(to, lane + 128u, c);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };
    struct Step {
        ExpertWords words;
        half8 hi, lo;
    };
    const auto load_step = [&](const SmallUnit &u, uint32_t kc, Step &to) {
#pragma unroll
        for (uint32_t f = 0; f < kFragments; ++f) {
            const uint32_t tr = min(u.tile_row + f, tile_rows - 1u);
            to.words.w[f] = __builtin_bit_cast(
                uint2, __builtin_amdgcn_raw_buffer_load_b64(u.words, lane_words, ((tr << tc_shift) + 4u * kc) * 48u, 0));
        }
        to.hi = __builtin_bit_cast(half8, __builtin_amdgcn_raw_buffer_load_b128(u.x_hi, u.x_off, kc * 64u, 0));
        to.lo = __builtin_bit_cast(half8, __builtin_amdgcn_raw_buffer_load_b128(u.x_lo, u.x_off, kc * 64u, 0));
    };
    struct Gathered {
        ExpertEntries f[kFragments];
    };
    const auto gather = [&](const ExpertWords &w) {
        Gathered out;
#pragma unroll
        for (uint32_t f = 0; f < kFragments; ++f) {
            out.f[f] = expert_gather(string, w.w[f], plane);
        }
        return out;
    };

    uint32_t next_unit = second_unit;
    SmallUnit load = open(first_unit);
    uint32_t g0 = load_gamma(load, lane), g1 = load_gamma(load, lane + 64u), g2 = load_gamma(load, lane + 128u);
    Step ring[4];
#pragma unroll
    for (uint32_t s = 0; s < 4u; ++s) {
        load_step(load, s, ring[s]);
    }
    uint32_t load_kc = 4u;
    uint2 *gamma_now = gammas, *gamma_next = gammas + 4u * kSmallGammaRow;
    store_gammas(gamma_now, g0, g1, g2);
    SmallUnit now = load;
    bool more = false;  // `load` is past `now`
    uint32_t kc = 0;
    f32x4 acc[kFragments];
#pragma unroll
    for (uint32_t f = 0; f < kFragments; ++f) {
        acc[f] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    }
    Gathered entries = gather(ring[0].words);
    for (;;) {
        if (load_kc == steps) {
            more = next_unit < units;
            if (more) {
                load = open(next_unit);
                next_unit += stride;
                g0 = load_gamma(load, lane);
                g1 = load_gamma(load, lane + 64u);
                g2 = load_gamma(load, lane + 128u);
                load_kc = 0;
            } else {
                load_kc = steps - 4u;  // the last group again, unused
            }
        }
#pragma unroll
        for (uint32_t s = 0; s < 4u; ++s) {
            const Gathered next = gather(ring[(s + 1u) & 3u].words);
            const uint2 g = gamma_now[kq * kSmallGammaRow + kc + s];
            __builtin_amdgcn_sched_barrier(0);
            const uint32_t gamma[kFragments] = {g.x & 0xFFFFu, g.x >> 16, g.y & 0xFFFFu, g.y >> 16};
            half8 hi[kFragments], lo[kFragments];
#pragma unroll
            for (uint32_t f = 0; f < kFragments; ++f) {
                expert_scale<PASSES>(entries.f[f], gamma[f], sign_mask, hi[f], lo[f]);
            }
#pragma unroll
            for (uint32_t f = 0; f < kFragments; ++f) {
                acc[f] = __builtin_amdgcn_mfma_f32_16x16x32_f16(hi[f], ring[s].hi, acc[f], 0, 0, 0);
            }
#pragma unroll
            for (uint32_t f = 0; f < kFragments; ++f) {
                acc[f] = __builtin_amdgcn_mfma_f32_16x16x32_f16(hi[f], ring[s].lo, acc[f], 0, 0, 0);
            }
            if constexpr (PASSES == 3) {
#pragma unroll
                for (uint32_t f = 0; f < kFragments; ++f) {
                    acc[f] = __builtin_amdgcn_mfma_f32_16x16x32_f16(lo[f], ring[s].hi, acc[f], 0, 0, 0);
                }
            }
            load_step(load, load_kc + s, ring[s]);
            entries = next;
        }
        load_kc += 4u;
        kc += 4u;
        if (kc == steps) {
            // D register r of lane l: position l % 16, tile row's row 4 (l / 16) + r
            if (column < now.positions) {
#pragma unroll
                for (uint32_t f = 0; f < kFragments; ++f) {
                    if (now.tile_row + f < tile_rows) {
                        *reinterpret_cast<f32x4 *>(now.z + static_cast<size_t>(column) * rows +
                                                   (now.tile_row + f) * kTile + 4u * kq) = acc[f];
                    }
                }
            }
            if (!more) {
                return;
            }
            uint2 *const spent = gamma_now;
            gamma_now = gamma_next;
            gamma_next = spent;
            store_gammas(gamma_now, g0, g1, g2);
            now = load;
            kc = 0;
#pragma unroll
            for (uint32_t f = 0; f < kFragments; ++f) {
                acc[f] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            }
        }
    }
}

// Block b serves codebook plane (b / 8) % 2 as worker ((b / 16) * 8 + b % 8)
// (the two blocks that walk the same tiles share an XCD). Each block counts
// the items of every routed slot (position groups x row quarters) and scans
// the counts in LDS, so the blocks walk only real items, evenly. Items are
// numbered (entry, slot, position group, row quarter); a block takes them
// kExpertGroups at a time, and a group past the last item runs a copy of the
// last one without storing it.
template <int CB, int GROUPS, int PASSES>
__global__ __launch_bounds__(512 * GROUPS) void k_expert_mfma(ExpertMfmaJobs J) {
    static_assert(CB == 1 || CB == 2, "items of 32 or 64 positions");
    constexpr uint32_t kExpertThreads = 512 * GROUPS;
    constexpr uint32_t kExpertGroups = GROUPS;
    constexpr uint32_t kPositions = 32 * CB;              // per item
    // a thread's share of a K step's B rows: 8 bytes (32 positions) or 16 (64)
    using BChunk = std::conditional_t<CB == 1, uint2, uint4>;
    constexpr uint32_t kThreadsPerRow = CB == 1 ? 8u : 4u;
    constexpr uint32_t kChunkBytes = 64u / kThreadsPerRow;
    constexpr uint32_t kWaves = kExpertThreads / kWave;
    constexpr uint32_t kGroupThreads = 512;
    constexpr uint32_t kBRows = 2u * kPositions;          // (hi/lo, position) rows of B
    constexpr uint32_t kBSlot = kBRows * kBRowPitch;      // bytes per K step in the ring
    constexpr int kDepth = 4;                             // K steps of loads in flight
    // static LDS with the plane first: its address is a compile-time
    // constant, so a gather's address is the masked row offset alone
    __shared__ uint4 plane_lds[kPlaneRows16];
    __shared__ uint32_t starts[kSlotCapacity + 1];
    __shared__ uint64_t wave_sums[kWaves];
    __shared__ uint32_t small_count;
    // gamma rows of an item: row q entry i = gamma of the tile at
    // anti-diagonal tr_block + i + q; lane (w, tsub, kh) reads its tiles'
    // gammas at K step kc from row tsub + kh at entries 4w + 4kc .. + 7
    __shared__ uint2 gamma_rows[kExpertGroups][4][kGammaRow / 4];
    __shared__ uint4 b_ring[kExpertGroups][2][kBSlot / 16];
    static_assert(sizeof(b_ring) >= 8u * kExpertGroups * kSmallGammas * sizeof(uint2), "the waves' gamma rows");
    __shared__ uint16_t small_slots[kSlotCapacity];
    const uint32_t b = blockIdx.x;
    const uint32_t half = (b >> 3) & 1u;
    const uint32_t worker = ((b >> 4) << 3) | (b & 7u);
    const uint32_t workers = gridDim.x >> 1;
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t group = wave >> 3, gwave = wave & 7u;
    const uint32_t gthread = threadIdx.x & (kGroupThreads - 1u);
    {
        const uint4 *src = static_cast<const uint4 *>(J.expert_book) + half * kPlaneRows16;
        // indexes past the plane are clamped: those threads reload and rewrite
        // its last row, so no load is guarded
        constexpr uint32_t kPer = (kPlaneRows16 + kExpertThreads - 1) / kExpertThreads;
        uint4 v[kPer];
#pragma unroll
        for (uint32_t u = 0; u < kPer; ++u) {
            v[u] = src[min(u * kExpertThreads + threadIdx.x, kPlaneRows16 - 1u)];
        }
        // item counts per slot: each thread owns two consecutive slots; a
        // small slot counts 1 in the upper half instead
        const uint32_t quarters = J.row_groups;
        uint32_t count[2];
        bool small[2];
#pragma unroll
        for (uint32_t k = 0; k < 2; ++k) {
            const uint32_t s = 2u * threadIdx.x + k;
            uint4 info = make_uint4(0u, 0u, 0u, 0u);
            if (s < J.max_active) {
                info = J.slot_info != nullptr ? J.slot_info[s]
                                              : make_uint4(0u, 0u, s == 0 ? J.max_positions : 0u, 0u);
            }
            const uint32_t held = info.z > info.y ? info.z - info.y : 0u;
            small[k] = J.small_slots != 0u && held != 0u && held <= kSmallPositions;
            count[k] = small[k] ? 0u : (held + kPositions - 1u) / kPositions * quarters;
        }
        // block-wide exclusive scans (slot order): items in the lower half,
        // small slots in the upper
        const uint64_t own = (static_cast<uint64_t>(small[0]) + small[1]) << 32 | (count[0] + count[1]);
        uint64_t inclusive = own;
#pragma unroll
        for (int offset = 1; offset < 64; offset <<= 1) {
            const uint64_t other = __shfl_up(static_cast<unsigned long long>(inclusive), offset);
            if (lane >= static_cast<uint32_t>(offset)) {
                inclusive += other;
            }
        }
        if (lane == 63u) {
            wave_sums[wave] = inclusive;
        }
#pragma unroll
        for (uint32_t u = 0; u < kPer; ++u) {
            plane_lds[min(u * kExpertThreads + threadIdx.x, kPlaneRows16 - 1u)] = v[u];
        }
        __syncthreads();
        uint64_t before = 0;
        for (uint32_t w = 0; w < wave; ++w) {
            before += wave_sums[w];
        }
        const uint64_t exclusive = before + inclusive - own;
        if (2u * threadIdx.x < kSlotCapacity) {
            const uint32_t start = static_cast<uint32_t>(exclusive);
            starts[2u * threadIdx.x] = start;
            starts[2u * threadIdx.x + 1u] = start + count[0];
            uint32_t place = static_cast<uint32_t>(exclusive >> 32);
#pragma unroll
            for (uint32_t k = 0; k < 2; ++k) {
                if (small[k]) {
                    small_slots[place] = static_cast<uint16_t>(2u * threadIdx.x + k);
                    ++place;
                }
            }
        }
        if (threadIdx.x == kExpertThreads - 1u) {
            starts[kSlotCapacity] = static_cast<uint32_t>(before + inclusive);  // items per entry
            small_count = static_cast<uint32_t>((before + inclusive) >> 32);
        }
    }
    __syncthreads();
    const uint2 *plane = reinterpret_cast<const uint2 *>(plane_lds);
    const uint32_t per_entry = starts[kSlotCapacity];
    const uint32_t total = per_entry * J.expert_count;
    const uint32_t m = lane & 31u, kh = lane >> 5;   // MFMA row / column and K half
    const uint32_t trow = m & 15u, tsub = m >> 4;    // row within the tile, tile row within the block
    const uint32_t sign_mask = half == 0 ? 0x8000u : 0u;
    const ExpertString string = expert_string(trow);
    // the thread's share of its group's B loads: one chunk of one B row (B
    // rows are (hi/lo, position); wave w of the group loads rows
    // (64 / kThreadsPerRow) w .., so the hi/lo plane is wave-uniform: derived
    // from `gwave`, the buffer resource stays scalar)
    const uint32_t b_row = gthread / kThreadsPerRow, b_chunk = gthread % kThreadsPerRow;
    const uint32_t b_lo = gwave >> 2, b_n = b_row & (kPositions - 1u);
    char *ring = reinterpret_cast<char *>(b_ring[group]);
    const uint32_t b_store = b_row * kBRowPitch + b_chunk * kChunkBytes;
    auto load_b = [](__amdgpu_buffer_rsrc_t src, uint32_t off, uint32_t soff) {
        if constexpr (CB == 1) {
            return __builtin_bit_cast(BChunk, __builtin_amdgcn_raw_buffer_load_b64(src, off, soff, 0));
        } else {
            return __builtin_bit_cast(BChunk, __builtin_amdgcn_raw_buffer_load_b128(src, off, soff, 0));
        }
    };
    const uint32_t rounds = (total + kExpertGroups - 1u) / kExpertGroups;
    for (uint32_t round = worker; round < rounds; round += workers) {
        const uint32_t item_any = round * kExpertGroups + group;
        const bool live = item_any < total;
        const uint32_t item = live ? item_any : total - 1u;
        const uint32_t which = item / per_entry;
        const uint32_t local = item - which * per_entry;
        // the slot whose item range holds `local`: last s with starts[s] <= local
        uint32_t lo = 0, hi = J.max_active;
        while (hi - lo > 1u) {
            const uint32_t mid = (lo + hi) >> 1;
            if (starts[mid] <= local) {
                lo = mid;
            } else {
                hi = mid;
            }
        }
        const uint32_t slot = __builtin_amdgcn_readfirstlane(lo);
        const uint32_t within = local - starts[slot];
        const uint32_t rq = within % J.row_groups;
        const uint32_t pg = within / J.row_groups;
        // the slot is uniform: its entry comes through the scalar cache
        const uint4 info = J.slot_info != nullptr ? J.slot_info[slot]
                                                  : make_uint4(0u, 0u, J.max_positions, 0u);
        const uint32_t first = __builtin_amdgcn_readfirstlane(info.y);
        const uint32_t mat = __builtin_amdgcn_readfirstlane(info.x);
        const uint32_t end = __builtin_amdgcn_readfirstlane(info.z);
        const ExpertMfma &a = J.expert[which];
        const uint32_t p0 = first + pg * kPositions;
        const uint32_t tr_block = rq * kBlockTileRows;
        const uint32_t tr0 = tr_block + gwave * kExpertRT;
        const uint32_t half_columns = a.columns >> 1;
        const uint32_t tile_columns = 1u << a.tc_shift;
        const uint32_t steps = tile_columns / 4u;  // a power of two
        const uint32_t last = steps - 1u;
        // this thread's B row: position p0 + b_n (clamped to a real row past
        // the slot), hi or lo plane
        const size_t plane_elems = static_cast<size_t>(a.positions) * half_columns;
        const uint32_t x_bytes = static_cast<uint32_t>(plane_elems * 2u);
        const __amdgpu_buffer_rsrc_t xsrc =
            buffer_over((b_lo ? a.x_lo : a.x_hi) + half * plane_elems, x_bytes);
        const uint32_t bp = p0 + b_n;
        const uint32_t b_off = ((bp < end ? bp : p0) * half_columns + b_chunk * (kChunkBytes / 2u)) * 2u;
        ExpertWave wv;
        const uint32_t tiles = a.tile_rows << a.tc_shift;
        wv.words = buffer_over(a.trellis + mat * a.trellis_stride, tiles * 48u);
        const uint32_t dpair = expert_dwords(trow);
#pragma unroll
        for (int f = 0; f < kFragments; ++f) {
            const uint32_t rb = f >> 1, c = f & 1;
            const uint32_t tr = min(tr0 + 2u * rb + tsub, a.tile_rows - 1u);
            const uint32_t tile = (tr << a.tc_shift) + 2u * c + kh;
            wv.woff[f] = (tile * 12u + dpair) * 4u;
        }
        wv.gammas = gamma_rows[group][tsub + kh] + gwave;  // entry 4 * gwave
        wv.string = string;

        // the previous item's readers of the gamma rows and the ring are done
        __syncthreads();
        {
            // gamma of the tile at anti-diagonal d = tr_block + e sits in wave
            // slot R_t + C_t - 1 - d, one less past the main anti-diagonal
            // (src/codec_cache.cpp:117-147); slots past the matrix read 0 and
            // belong to tiles that are never stored
            const __amdgpu_buffer_rsrc_t gbuf =
                buffer_over(a.gamma + mat * a.gamma_stride, (a.tile_rows + tile_columns) * 2u);
            const uint32_t top = a.tile_rows + tile_columns - 1u;
            uint16_t *rows = reinterpret_cast<uint16_t *>(gamma_rows[group]);
            const uint32_t e = gthread;  // tile_columns + 35 <= 512
            const uint32_t d = tr_block + e;
            const uint32_t gslot = top - d - (d >= tile_columns ? 1u : 0u);
            const uint16_t g = __builtin_amdgcn_raw_buffer_load_b16(gbuf, gslot * 2u, 0, 0);
            if (e < tile_columns + kBlockTileRows + 3u) {
#pragma unroll
                for (uint32_t q = 0; q < 4u; ++q) {
                    const uint32_t i = e - q;  // wraps past zero: then out of range
                    if (i < kGammaRow) {
                        rows[q * kGammaRow + i] = g;
                    }
                }
            }
        }
        f32x16 acc[2][CB];
#pragma unroll
        for (int rb = 0; rb < 2; ++rb) {
#pragma unroll
            for (int cb = 0; cb < CB; ++cb) {
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    acc[rb][cb][r] = 0.0f;
                }
            }
        }
        // B of K step kc, as the MFMA operands of position block cb, K pair c
        // (the item's first LIVE blocks)
        auto read_b = [&]<int LIVE>(uint32_t ring_slot, half8 (&bh)[CB][2], half8 (&bl)[CB][2]) {
            const char *base = ring + ring_slot * kBSlot + m * kBRowPitch + kh * 16u;
#pragma unroll
            for (int cb = 0; cb < LIVE; ++cb) {
#pragma unroll
                for (int c = 0; c < 2; ++c) {
                    bh[cb][c] = *reinterpret_cast<const half8 *>(base + cb * 32u * kBRowPitch + c * 32u);
                    bl[cb][c] = *reinterpret_cast<const half8 *>(base + (kPositions + cb * 32u) * kBRowPitch + c * 32u);
                }
            }
        };
        // the K loop for an item whose first LIVE blocks of 32 positions hold
        // positions of its slot: each K step's A fragments are decoded once
        // and multiplied with every live block (the slot's later blocks skip
        // their MFMAs, not the decode)
        auto k_loop = [&]<int LIVE>() {
            if (steps % kDepth != 0) {
                // short K (under 4 steps): one step at a time
                for (uint32_t kc = 0; kc < steps; ++kc) {
                    const BChunk bv = load_b(xsrc, b_off, kc * 64u);
                    ExpertWords ws;
                    expert_words(wv, kc, ws);
                    *reinterpret_cast<BChunk *>(ring + b_store) = bv;
                    __syncthreads();
                    half8 bh[CB][2], bl[CB][2];
                    read_b.template operator()<LIVE>(0, bh, bl);
                    ExpertA fa;
                    expert_decode<PASSES>(wv, kc, sign_mask, plane, ws, fa);
                    expert_multiply<CB, LIVE, PASSES>(fa, bh, bl, acc);
                    __syncthreads();
                }
            } else {
                // B of step s waits in bv[s % 4] (registers) until step s - 1
                // writes it to ring slot s % 2; the words of step s wait in
                // ws[s % 4]. Loads past the last step reload it (in bounds,
                // unused), so the loop body has no branch.
                BChunk bv[kDepth];
                ExpertWords ws[kDepth];
#pragma unroll
                for (int u = 0; u < kDepth; ++u) {
                    __builtin_amdgcn_sched_barrier(0);
                    bv[u] = load_b(xsrc, b_off, u * 64u);
                    if (u < kDepth - 1) {
                        expert_words(wv, u, ws[u]);
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
                *reinterpret_cast<BChunk *>(ring + b_store) = bv[0];
                bv[0] = load_b(xsrc, b_off, min(static_cast<uint32_t>(kDepth), last) * 64u);
                __syncthreads();
                for (uint32_t kc = 0; kc < steps; kc += kDepth) {
#pragma unroll
                    for (int u = 0; u < kDepth; ++u) {
                        const uint32_t step = kc + u;
                        __builtin_amdgcn_sched_barrier(0);
                        // hand B of the next step to the ring and refill its registers
                        *reinterpret_cast<BChunk *>(ring + ((u + 1) & 1) * kBSlot + b_store) = bv[(u + 1) % kDepth];
                        bv[(u + 1) % kDepth] = load_b(xsrc, b_off, min(step + 1u + kDepth, last) * 64u);
                        expert_words(wv, min(step + kDepth - 1u, last), ws[(u + kDepth - 1) % kDepth]);
                        __builtin_amdgcn_sched_barrier(0);
                        half8 bh[CB][2], bl[CB][2];
                        read_b.template operator()<LIVE>(u & 1, bh, bl);
                        ExpertA fa;
                        expert_decode<PASSES>(wv, step, sign_mask, plane, ws[u], fa);
                        expert_multiply<CB, LIVE, PASSES>(fa, bh, bl, acc);
                        __syncthreads();
                    }
                }
            }
        };
        if constexpr (CB == 2) {
            if (p0 + 32u < end) {
                k_loop.template operator()<2>();
            } else {
                k_loop.template operator()<1>();
            }
        } else {
            k_loop.template operator()<1>();
        }
        // D register r of lane l: position 32 cb + l % 32, block row
        // (r % 4) + 8 (r / 4) + 4 kh
        float *z = a.z + half * a.z_split_stride;
#pragma unroll
        for (int cb = 0; cb < CB; ++cb) {
            const uint32_t p = p0 + 32u * cb + m;
            if (live && p < end) {
#pragma unroll
                for (int rb = 0; rb < 2; ++rb) {
#pragma unroll
                    for (int g = 0; g < 4; ++g) {
                        const uint32_t row = (tr0 + 2u * rb) * kTile + 8u * g + 4u * kh;
                        if (row < a.rows) {
                            *reinterpret_cast<f32x4 *>(z + static_cast<size_t>(p) * a.rows + row) =
                                f32x4{acc[rb][cb][4 * g], acc[rb][cb][4 * g + 1], acc[rb][cb][4 * g + 2],
                                      acc[rb][cb][4 * g + 3]};
                        }
                    }
                }
            }
        }
    }
    // the small slots, a unit a wave: first the workers that the last round of
    // items left idle take one a wave, then all take the rest in turn, worker
    // by worker, so that the last ones spread over the CUs
    if (small_count != 0u) {  // uniform over the block
        __syncthreads();      // the ring is free
        const uint32_t busy = rounds % workers, idle = busy == 0u ? 0u : workers - busy;
        const uint32_t stride = workers * kWaves;
        const uint32_t turn = idle * kWaves + worker + workers * wave;
        const bool extra = idle != 0u && worker >= busy;
        const uint32_t first_unit = extra ? worker - busy + idle * wave : turn;
        expert_small_slots<PASSES>(J, half, first_unit, extra ? turn : turn + stride, stride, plane, small_slots,
                                   small_count,
                                   reinterpret_cast<uint2 *>(&b_ring[0][0][0]) + wave * kSmallGammas);
    }
}

// ---- NE -------------------------------------------------------------------
//
// Also on v_mfma_f32_32x32x16_f16. A block of eight waves takes one item: 32
// positions x 16 tile rows (256 rows) of one NE entry over one K slice; wave w
// takes tile rows 2w, 2w + 1 as one 32-row block. Lane l holds row l % 16 of
// tile row 2w + (l % 32) / 16 and, of K pair c at K step kc, columns
// 8 (l / 32) .. + 7 of tile column 2 kc + c: NE states 8 (l % 16) +
// 4 (l / 32) + 0..3, four lookups of the signed table (two f16 each). The
// block loads each K step's x_hat hi and lo of its 32 positions once into an
// LDS ring (one barrier per K step); each wave loads its trellis words four K
// steps ahead.

constexpr uint32_t kNeThreads = 512;
constexpr uint32_t kNeWaves = kNeThreads / kWave;
constexpr uint32_t kNeItemTileRows = 2 * kNeWaves;   // 256 rows per item
constexpr uint32_t kNeBSlot = 64 * kBRowPitch;      // (hi/lo, position) rows of one K step

// The lane's trellis dwords of its two fragments (K pair c) at one K step.
struct NeWords {
    uint32_t d0[2], d1[2];
};

__global__ __launch_bounds__(kNeThreads) void k_ne_mfma(NeMfmaJobs J) {
    __shared__ uint32_t table[1024];
    __shared__ uint4 b_ring[2][kNeBSlot / 16];
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // item (row group, K slice, position group, entry), fastest first
    uint32_t rest = blockIdx.x;
    const uint32_t rg = rest % J.row_groups;
    rest /= J.row_groups;
    const uint32_t ks = rest % J.k_slices;
    rest /= J.k_slices;
    const uint32_t pg = rest % J.position_groups;
    const uint32_t which = rest / J.position_groups;
    const NeMfma &a = J.ne[which];
    const uint32_t steps = (a.columns >> 5) / J.k_slices;  // K steps of 32 columns, a power of two
    const uint32_t k0 = ks * steps;
    const uint32_t last = steps - 1u;
    const uint32_t p0 = pg * 32u;
    // the table: eight bytes per thread, stored once the first loads are out
    const uint2 tv = reinterpret_cast<const uint2 *>(J.ne_book)[threadIdx.x];
    // B staging: thread t copies 8 bytes of B row t / 8 (rows 0..31 hi, 32..63
    // lo, so the plane is wave-uniform); positions past the batch repeat p0
    const uint32_t b_row = threadIdx.x >> 3, b_chunk = threadIdx.x & 7u;
    const uint32_t bp = p0 + (b_row & 31u);
    const uint32_t b_pos = bp < a.batch ? bp : p0;
    const __amdgpu_buffer_rsrc_t xsrc =
        buffer_over(wave >= 4u ? a.x_lo : a.x_hi, a.batch * a.columns * 2u);
    const uint32_t b_off = (b_pos * a.columns + b_chunk * 4u) * 2u + k0 * 64u;
    char *ring = reinterpret_cast<char *>(b_ring);
    const uint32_t b_store = b_row * kBRowPitch + b_chunk * 8u;
    auto load_b = [&](uint32_t kc) {
        return __builtin_bit_cast(uint2, __builtin_amdgcn_raw_buffer_load_b64(xsrc, b_off, kc * 64u, 0));
    };
    // the lane's trellis words: row trow of tile row tr, dwords dw and dw + 1
    // (row 15's second wraps to dword 0, src/ne_trellis.hpp:196-200)
    const uint32_t m = lane & 31u, kh = lane >> 5;
    const uint32_t trow = m & 15u;
    const uint32_t tr_block = rg * kNeItemTileRows + 2u * wave;
    const uint32_t tr = min(tr_block + (m >> 4), a.tile_rows - 1u);
    const uint32_t dw = 2u * trow + kh, dn = dw == 31u ? 0u : dw + 1u;
    const __amdgpu_buffer_rsrc_t wsrc = buffer_over(a.trellis, (a.tile_rows << a.tc_shift) * 128u);
    const uint32_t w0 = ((tr << a.tc_shift) * 32u + dw) * 4u;
    const uint32_t w1 = ((tr << a.tc_shift) * 32u + dn) * 4u;
    auto load_words = [&](uint32_t kc, NeWords &w) {
#pragma unroll
        for (uint32_t c = 0; c < 2; ++c) {
            const uint32_t soff = (2u * (k0 + kc) + c) * 128u;  // tile column 2 kc + c
            w.d0[c] = __builtin_amdgcn_raw_buffer_load_b32(wsrc, w0, soff, 0);
            w.d1[c] = __builtin_amdgcn_raw_buffer_load_b32(wsrc, w1, soff, 0);
        }
    };
    f32x16 acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        acc[r] = 0.0f;
    }
    // one K step: the two A fragments from the table, B from ring slot `slot`
    auto multiply = [&](uint32_t slot, const NeWords &w) {
        const char *base = ring + slot * kNeBSlot + m * kBRowPitch + kh * 16u;
#pragma unroll
        for (uint32_t c = 0; c < 2; ++c) {
            const half8 bh = *reinterpret_cast<const half8 *>(base + c * 32u);
            const half8 bl = *reinterpret_cast<const half8 *>(base + 32u * kBRowPitch + c * 32u);
            uint32_t v[4];
#pragma unroll
            for (uint32_t q = 0; q < 4; ++q) {
                // state hash in v_mad_u32_u24: the window's bits above bit 15
                // only add multiples of 2^16
                v[q] = table[(state_hash_low16(window64(w.d0[c], w.d1[c], 8u * q)) >> 6) & 0x3FFu];
            }
            const half8 av = __builtin_bit_cast(half8, u32x4{v[0], v[1], v[2], v[3]});
            acc = mfma32(av, bh, acc);
            acc = mfma32(av, bl, acc);
        }
    };
    constexpr uint32_t kDepth = 4;
    if (steps % kDepth != 0) {
        // short K (under 4 steps): one step at a time
        table[threadIdx.x * 2u] = tv.x;
        table[threadIdx.x * 2u + 1u] = tv.y;
        for (uint32_t kc = 0; kc < steps; ++kc) {
            const uint2 bv = load_b(kc);
            NeWords w;
            load_words(kc, w);
            *reinterpret_cast<uint2 *>(ring + b_store) = bv;
            __syncthreads();
            multiply(0, w);
            __syncthreads();
        }
    } else {
        // B of step s waits in bv[s % 4] until step s - 1 writes it to ring
        // slot s % 2; the words of step s wait in ws[s % 4]. Loads past the
        // last step reload it (in bounds, unused).
        uint2 bv[kDepth];
        NeWords ws[kDepth];
#pragma unroll
        for (uint32_t u = 0; u < kDepth; ++u) {
            bv[u] = load_b(u);
            if (u < kDepth - 1) {
                load_words(u, ws[u]);
            }
        }
        table[threadIdx.x * 2u] = tv.x;
        table[threadIdx.x * 2u + 1u] = tv.y;
        *reinterpret_cast<uint2 *>(ring + b_store) = bv[0];
        bv[0] = load_b(min(kDepth, last));
        __syncthreads();
        for (uint32_t kc = 0; kc < steps; kc += kDepth) {
#pragma unroll
            for (uint32_t u = 0; u < kDepth; ++u) {
                const uint32_t step = kc + u;
                __builtin_amdgcn_sched_barrier(0);
                *reinterpret_cast<uint2 *>(ring + ((u + 1) & 1) * kNeBSlot + b_store) = bv[(u + 1) % kDepth];
                bv[(u + 1) % kDepth] = load_b(min(step + 1u + kDepth, last));
                load_words(min(step + kDepth - 1u, last), ws[(u + kDepth - 1) % kDepth]);
                __builtin_amdgcn_sched_barrier(0);
                multiply(u & 1, ws[u]);
                __syncthreads();
            }
        }
    }
    // D register r of lane l: position l % 32, row (r % 4) + 8 (r / 4) + 4 kh
    // of the wave's 32-row block
    const uint32_t p = p0 + m;
    if (p < a.batch) {
        float *z = a.z + static_cast<size_t>(ks) * a.batch * a.rows + static_cast<size_t>(p) * a.rows;
#pragma unroll
        for (uint32_t g = 0; g < 4; ++g) {
            const uint32_t row = tr_block * kTile + 8u * g + 4u * kh;
            if (row < a.rows) {
                *reinterpret_cast<f32x4 *>(z + row) =
                    f32x4{acc[4 * g], acc[4 * g + 1], acc[4 * g + 2], acc[4 * g + 3]} * a.weight_scale;
            }
        }
    }
}

// The same product for many positions. An item of k_ne_mfma decodes its weights
// for 32 positions only, and reads x_hat from LDS once a wave and 32 rows: for
// hundreds of positions the table lookups and those reads bound it. Here a
// block of eight waves takes 64 RB rows x 128 positions and stages of 64
// columns: every thread decodes RB runs of eight weights into LDS, once for the
// 128 positions, and copies 64 bytes of x_hat; the waves, two by four, then
// multiply 32 RB rows by 32 positions from LDS. A stage is decoded and stored
// while the one before it is multiplied (two buffers, one barrier a stage), and
// its words and x_hat are loaded a stage earlier still. A and B lie in LDS as
// 64-lane fragments of 16-byte pieces, rows XORed so that stores and reads
// spread over the banks.
//
// Bound by LDS: at 8192 x 2048 and 512 positions its accesses take 52% and the
// matrix instructions 40% of the waves' 34 us (46 us a launch; k_ne_mfma 60),
// about a quarter of the launch is the start and the write-back of Z. Stages
// loaded one instead of two ahead: 49 us; half the waves multiplying while the
// others decode: 48.
constexpr uint32_t kWidePositions = 128;

template <uint32_t RB>
__global__ __launch_bounds__(kNeThreads) void k_ne_wide(NeMfmaJobs J) {
    constexpr uint32_t kTileRows = 4u * RB;  // a block's
    constexpr uint32_t kAPieces = 2u * RB * 4u * 64u, kBPieces = 4u * 4u * 2u * 64u;
    __shared__ uint32_t table[1024];
    __shared__ u32x4 a_lds[2][kAPieces];
    __shared__ u32x4 b_lds[2][kBPieces];
    const uint32_t t = threadIdx.x, lane = t & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(t >> 6);
    // item (row group, K slice, position group, entry), fastest first. With
    // eight K slices or more the slices come first: block b runs on XCD b % 8,
    // so an XCD then reads x_hat and weights of its slices only, where eight row
    // groups first had every XCD read all of x_hat (512 x 2048, 256 positions:
    // 20.0 us a call, 17.3; k_ne_mfma 18.3).
    const bool by_slice = J.k_slices >= 8u;
    const uint32_t slice_shift = __builtin_ctz(J.k_slices);  // (a power of two)
    uint32_t rest = by_slice ? blockIdx.x >> slice_shift : blockIdx.x;
    const uint32_t rg = rest % J.row_groups;
    rest /= J.row_groups;
    const uint32_t ks = (by_slice ? blockIdx.x : rest) & (J.k_slices - 1u);
    rest = by_slice ? rest : rest >> slice_shift;
    const uint32_t pg = rest % J.position_groups;
    const uint32_t which = rest / J.position_groups;
    const NeMfma &a = J.ne[which];
    const uint32_t stages = (a.columns >> 6) / J.k_slices;
    const uint32_t p0 = pg * kWidePositions;
    const uint2 tv = reinterpret_cast<const uint2 *>(J.ne_book)[t];
    // run i of the thread: dword t % 32 (row (t % 32) / 2, columns 8 (t % 2) ..)
    // of the tile in tile column (t / 32) % 4 and tile row t / 128 + 4 i; its
    // second dword wraps within the tile (src/ne_trellis.hpp:196-200)
    const uint32_t dword = t & 31u, tc = (t >> 5) & 3u;
    const __amdgpu_buffer_rsrc_t wsrc = buffer_over(a.trellis, (a.tile_rows << a.tc_shift) * 128u);
    uint32_t w_off[RB], a_slot[RB];
#pragma unroll
    for (uint32_t i = 0; i < RB; ++i) {
        const uint32_t tr = (t >> 7) + 4u * i;
        const uint32_t row = ((tr & 1u) << 4) | (dword >> 1), kh = dword & 1u;
        w_off[i] = ((min(rg * kTileRows + tr, a.tile_rows - 1u) << a.tc_shift) + tc) * 128u;
        a_slot[i] = ((tr >> 1) * 4u + tc) * 64u + kh * 32u + (row ^ (kh << 2));
    }
    // x_hat: 16 bytes (piece t % 8 of the stage's 128) of positions t / 8 and
    // t / 8 + 64, both planes; positions past the batch repeat p0
    const uint32_t piece = t & 7u;
    const uint32_t x_bytes = a.batch * a.columns * 2u;
    const __amdgpu_buffer_rsrc_t hi_src = buffer_over(a.x_hi, x_bytes), lo_src = buffer_over(a.x_lo, x_bytes);
    uint32_t x_off[2], b_slot[2];
#pragma unroll
    for (uint32_t i = 0; i < 2; ++i) {
        const uint32_t pos = (t >> 3) + 64u * i;
        x_off[i] = ((p0 + pos < a.batch ? p0 + pos : p0) * a.columns + 8u * piece) * 2u;
        b_slot[i] = ((pos >> 5) * 4u + (piece >> 1)) * 128u + (piece & 1u) * 32u + ((pos & 31u) ^ piece);
    }
    struct Stage {
        uint32_t d0[RB], d1[RB];
        u32x4 hi[2], lo[2];
    };
    const auto load_stage = [&](uint32_t stage) {
        Stage out;
        const uint32_t at = ks * stages + stage;
#pragma unroll
        for (uint32_t i = 0; i < RB; ++i) {
            out.d0[i] = __builtin_amdgcn_raw_buffer_load_b32(wsrc, w_off[i] + dword * 4u, at * 512u, 0);
            out.d1[i] = __builtin_amdgcn_raw_buffer_load_b32(wsrc, w_off[i] + ((dword + 1u) & 31u) * 4u, at * 512u, 0);
        }
#pragma unroll
        for (uint32_t i = 0; i < 2; ++i) {
            out.hi[i] = __builtin_amdgcn_raw_buffer_load_b128(hi_src, x_off[i], at * 128u, 0);
            out.lo[i] = __builtin_amdgcn_raw_buffer_load_b128(lo_src, x_off[i], at * 128u, 0);
        }
        return out;
    };
    const auto store_stage = [&](const Stage &s, uint32_t buffer) {
#pragma unroll
        for (uint32_t i = 0; i < 2; ++i) {
            b_lds[buffer][b_slot[i]] = s.hi[i];
            b_lds[buffer][b_slot[i] + 64u] = s.lo[i];
        }
#pragma unroll
        for (uint32_t i = 0; i < RB; ++i) {
            u32x4 v;
#pragma unroll
            for (uint32_t q = 0; q < 4; ++q) {
                v[q] = table[(state_hash_low16(window64(s.d0[i], s.d1[i], 8u * q)) >> 6) & 0x3FFu];
            }
            a_lds[buffer][a_slot[i]] = v;
        }
    };
    const uint32_t m = lane & 31u, kh = lane >> 5;
    const uint32_t wave_rows = wave & 1u, wave_positions = wave >> 1;
    f32x16 acc[RB];
#pragma unroll
    for (uint32_t rb = 0; rb < RB; ++rb) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            acc[rb][r] = 0.0f;
        }
    }
    struct Fragments {
        half8 hi, lo, a[RB];
    };
    const auto read = [&](uint32_t buffer, uint32_t c) {
        Fragments out;
        const u32x4 *b = b_lds[buffer] + (wave_positions * 4u + c) * 128u + kh * 32u + (m ^ (2u * c + kh));
        out.hi = __builtin_bit_cast(half8, b[0]);
        out.lo = __builtin_bit_cast(half8, b[64]);
#pragma unroll
        for (uint32_t rb = 0; rb < RB; ++rb) {
            out.a[rb] = __builtin_bit_cast(
                half8, a_lds[buffer][((wave_rows * RB + rb) * 4u + c) * 64u + kh * 32u + (m ^ (kh << 2))]);
        }
        return out;
    };
    const auto multiply = [&](uint32_t buffer) {
        Fragments f = read(buffer, 0);
#pragma unroll
        for (uint32_t c = 0; c < 4; ++c) {
            Fragments ahead = f;
            if (c < 3u) {
                ahead = read(buffer, c + 1u);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (uint32_t rb = 0; rb < RB; ++rb) {
                acc[rb] = mfma32(f.a[rb], f.hi, acc[rb]);
            }
#pragma unroll
            for (uint32_t rb = 0; rb < RB; ++rb) {
                acc[rb] = mfma32(f.a[rb], f.lo, acc[rb]);
            }
            __builtin_amdgcn_sched_barrier(0);
            f = ahead;
        }
    };
    // the words and x_hat of stage s wait in ring[s % 2]; loads past the last
    // stage repeat it, unused
    const uint32_t last = stages - 1u;
    Stage ring[2] = {load_stage(0), load_stage(min(1u, last))};
    table[2u * t] = tv.x;
    table[2u * t + 1u] = tv.y;
    __syncthreads();
    store_stage(ring[0], 0);
    ring[0] = load_stage(min(2u, last));
    __syncthreads();
    const auto step = [&](uint32_t stage, Stage &from) {  // `from` holds the stage after
        store_stage(from, (stage + 1u) & 1u);
        __builtin_amdgcn_sched_barrier(0);  // the loads stay ahead of the products
        from = load_stage(min(stage + 3u, last));
        __builtin_amdgcn_sched_barrier(0);
        multiply(stage & 1u);
        __syncthreads();
    };
    for (uint32_t stage = 0; stage + 2u < stages; stage += 2u) {
        step(stage, ring[1]);
        step(stage + 1u, ring[0]);
    }
    if (stages > 1u) {  // stages is a power of two
        step(stages - 2u, ring[1]);
    }
    multiply(last & 1u);
    // D register r of lane l: position l % 32, row (r % 4) + 8 (r / 4) + 4 kh
    // of the 32-row block
    const uint32_t p = p0 + 32u * wave_positions + m;
    if (p < a.batch) {
        float *z = a.z + static_cast<size_t>(ks) * a.batch * a.rows + static_cast<size_t>(p) * a.rows;
#pragma unroll
        for (uint32_t rb = 0; rb < RB; ++rb) {
#pragma unroll
            for (uint32_t g = 0; g < 4; ++g) {
                const uint32_t row =
                    (rg * kTileRows + 2u * (wave_rows * RB + rb)) * kTile + 8u * g + 4u * kh;
                if (row < a.rows) {
                    *reinterpret_cast<f32x4 *>(z + row) =
                        f32x4{acc[rb][4 * g], acc[rb][4 * g + 1], acc[rb][4 * g + 2], acc[rb][4 * g + 3]} *
                        a.weight_scale;
                }
            }
        }
    }
}

// Whether k_ne_wide takes a product: whole stages in every K slice, and at most
// an eighth of its positions padding more than k_ne_mfma's, about what it gains
// (8192 x 2048: 64 positions 16.1 us and 17.3, 128 23.0 and 19.1, 512 60 and 46;
// whole calls of 97, 128, 256 and 512 positions: 512 x 2048 15.4, 15.7, 18.3,
// 20.6 us and 14.3, 14.8, 17.3, 19.3; 2048 x 512 14.3, 14.6, 17.2, 20.6 and
// 13.3, 13.9, 16.5, 19.4; 2048 x 4096 23.0, 24.8, 29.9, 45.8 and 19.7, 21.3,
// 27.4, 40.3).
bool wide_takes(uint32_t columns, uint32_t batch, uint32_t k_slices) {
    const uint32_t narrow = ceil_div(batch, 32u) * 32u, wide = ceil_div(batch, kWidePositions) * kWidePositions;
    return columns / 64u >= k_slices && 8u * narrow >= 7u * wide;
}

}  // namespace

uint32_t ne_mfma_slices(uint32_t rows, uint32_t columns, uint32_t batch) {
    const uint32_t items = ceil_div(rows, kNeItemTileRows * kTile) * ceil_div(batch, 32u);
    uint32_t slices = 1;
    // about one block per CU, each with at least four K steps of 32 columns
    while (items * slices < 256u && columns / 32u / (slices * 2u) >= 4u) {
        slices *= 2u;
    }
    return slices;
}

void launch_expert_mfma(adi_hip_context *ctx, ExpertMfmaJobs &J) {
    require(J.expert_count >= 1 && J.expert_count <= 2, "MFMA GEMM: one or two expert entries");
    require(J.expert_book != nullptr, "MFMA GEMM: expert codebook missing");
    require(J.max_active >= 1 && J.max_active <= kSlotCapacity, "MFMA GEMM: routed slots out of range");
    require(J.slot_info != nullptr || J.max_active == 1, "MFMA GEMM: routed slots need a slot table");
    const ExpertMfma &e = J.expert[0];
    require(expert_mfma_supports(e.rows, e.columns), "MFMA GEMM: expert matrix shape out of range");
    for (uint32_t i = 0; i < J.expert_count; ++i) {
        ExpertMfma &x = J.expert[i];
        require(x.rows == e.rows && x.columns == e.columns, "MFMA GEMM: expert entries differ in shape");
        x.tile_rows = x.rows / kTile;
        x.tc_shift = log2_of(x.columns / kTile);
    }
    J.row_groups = ceil_div(e.rows / kTile, kBlockTileRows);  // row quarters of an item
    J.position_groups = ceil_div(J.max_positions, 32u * kExpertCB);
    J.items = J.expert_count * J.max_active * J.position_groups * J.row_groups;  // upper bound
    J.small_slots = small_slots_supported(e.columns / kTile) ? 1u : 0u;
    const uint32_t cap = ctx->cu_count >= 16 ? ctx->cu_count / 16 * 16 : 16u;
    const uint32_t needed = 16u * ceil_div(ceil_div(J.items, kExpertGroups), 8u);
    const uint32_t blocks = needed < cap ? needed : cap;
    auto kernel = k_expert_mfma<kExpertCB, kExpertGroups, kExpertPasses>;
    launch(ctx, "expert_mfma", kernel, dim3(blocks), dim3(512 * kExpertGroups), 0, J);
}

void launch_ne_mfma(adi_hip_context *ctx, NeMfmaJobs &J) {
    require(J.ne_count >= 1 && J.ne_count <= 2, "MFMA GEMM: one or two NE entries");
    require(J.ne_book != nullptr, "MFMA GEMM: NE codebook missing");
    const NeMfma &n = J.ne[0];
    require(n.columns >= 32 && n.rows >= 16, "MFMA GEMM: NE matrix below 16 x 32");
    require(is_power_of_two(n.columns) && n.rows % kTile == 0,
            "MFMA GEMM: NE columns must be a power of two and rows whole tiles");
    require(size_t(n.batch) * n.columns * 2u < (size_t(1) << 32) &&
                size_t(n.rows / kTile) * (n.columns / kTile) * 128u < (size_t(1) << 32),
            "MFMA GEMM: NE operands beyond 4 GiB");
    for (uint32_t i = 0; i < J.ne_count; ++i) {
        NeMfma &x = J.ne[i];
        require(x.rows == n.rows && x.columns == n.columns && x.batch == n.batch,
                "MFMA GEMM: NE entries differ in shape");
        require(aligned_to(x.x_hi, 16) && aligned_to(x.x_lo, 16) && aligned_to(x.z, 16),
                "MFMA GEMM: NE x_hat and Z must be 16-byte aligned");
        x.tile_rows = x.rows / kTile;
        x.tc_shift = log2_of(x.columns / kTile);
    }
    J.row_groups = ceil_div(n.rows / kTile, kNeItemTileRows);
    J.position_groups = ceil_div(n.batch, 32u);
    J.k_slices = ne_mfma_slices(n.rows, n.columns, n.batch);
    auto kernel = k_ne_mfma;
    if (wide_takes(n.columns, n.batch, J.k_slices)) {
        // two row blocks a wave where one would take more than one block a CU
        // (8192 x 2048, 512 positions: 46 us against 58; 4096 rows: 40, 31)
        J.position_groups = ceil_div(n.batch, kWidePositions);
        J.row_groups = ceil_div(n.rows, 64u);
        const bool two = J.ne_count * J.position_groups * J.row_groups * J.k_slices > static_cast<uint32_t>(ctx->cu_count);
        J.row_groups = two ? ceil_div(n.rows, 128u) : J.row_groups;
        kernel = two ? k_ne_wide<2> : k_ne_wide<1>;
    }
    J.items = J.ne_count * J.position_groups * J.row_groups * J.k_slices;
    launch(ctx, "ne_mfma", kernel, dim3(J.items), dim3(kNeThreads), 0, J);
}

}  // namespace adi_hip
