// Paged GQA decode attention for the shapes decode_split_mfma (decode_attention.h) does not take:
// any block size, any head_dim that is a multiple of 8 up to 256, FP32 pools, FP32 queries, any
// number of query heads per KV head, records and pools aligned to 4 bytes only.
//
// HBM-bound when it goes well: each K/V row is read once for (up to 16 of) the query heads that
// share its KV head, and the contractions run on the matrix cores. Work is cut into tiles of 16
// consecutive tokens of a sequence, whatever the block size: a lane finds each of its tokens'
// rows through the split's block ids, held in LDS. A wave takes one tile at a time, the waves of
// a workgroup round-robin over the split's tiles; lane l is (g, n) = (l / 16, l % 16):
//   QK: S^T[token][head], A = K (lane (g, n): token n), B = q^T (head n).
//   PV: O[head][dim], A = P (lane (g, n): head n, tokens 4g + r: the QK result as it stands),
//       B = V (tokens 4g + r, dims kVDims n .. +kVDims; MFMA e makes dims kVDims n' + e).
// Two forms of the arithmetic:
//   BF16 queries over BF16 or FP8 pools: v_mfma_f32_16x16x32_bf16 for QK (the products are exact
//   in FP32); the FP32 weights go to PV as three BF16 parts (24 bits together) in two 16x16x32
//   steps: the k index 8g + i of the first is token 4g + i's first part for i < 4 and its second for
//   i >= 4; the other step takes the third.
//   FP32 queries or pools: v_mfma_f32_16x16x4_f32 throughout, FP32 as it stands.
// Rows of tokens past the split or the sequence are read from a row of zeros instead, so the loads
// need no branches and a zero weight never meets a NaN.
//
// Measured on MI355X, per layer, against one wave per (sequence, query head, split) walking its
// tokens one at a time (decode_split_generic, which keeps head_dims that are no multiple of 8 and
// odd alignments): FP32 pool, 32 query heads of 128 dims, batch 4 at 700-2,500 tokens 517 -> 19 us
// (3.4 TB/s of K and V); BF16, 64 dims, batch 16 at 300-6,000 tokens 908 -> 22 us (4.5 TB/s), the
// merge launch apart. About 6 us of that is the chain from the launch to the first tile and from
// the last to the partials; at long contexts the loads set the pace.
#ifndef LAYOVER_AMD_DECODE_TILES_H
#define LAYOVER_AMD_DECODE_TILES_H

#include <type_traits>

#include "decode_attention.h"

namespace lk {

constexpr uint32_t kTilesMaxDim = 256;

// A row of zeros, as long as the longest row (256 FP32 dims).
static __device__ __align__(16) const uint32_t zero_row[kTilesMaxDim] = {};

// Loads that need only 4-byte alignment (2 for the halves of a word).
typedef uint32_t u32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));
typedef uint32_t u32x2_a4 __attribute__((ext_vector_type(2), aligned(4)));

template <int kBytes>
__device__ __forceinline__ void load_words(uint32_t* to, const uint8_t* from) {
    if constexpr (kBytes == 16) {
        const u32x4_a4 w = *reinterpret_cast<const u32x4_a4*>(from);
#pragma unroll
        for (int i = 0; i < 4; ++i) to[i] = w[i];
    } else if constexpr (kBytes == 8) {
        const u32x2_a4 w = *reinterpret_cast<const u32x2_a4*>(from);
        to[0] = w[0];
        to[1] = w[1];
    } else if constexpr (kBytes == 4) {
        to[0] = *reinterpret_cast<const uint32_t*>(from);
    } else {
        static_assert(kBytes == 2, "pieces are 2, 4, 8 or 16 bytes");
        to[0] = *reinterpret_cast<const uint16_t*>(from);
    }
}

// kD: head_dim rounded up to 32, 64, 128 or 256.
template <int KV, int QF, int kD>
struct TileShape {
    static constexpr bool kF32 = QF == LK_F32 || KV == LK_F32;  // FP32 arithmetic
    static constexpr uint32_t kElem = KV == LK_FP8_RECORD ? 1 : (KV == LK_F32 ? 4 : 2);
    // K: lane (g, n) loads kChunk dims from 4 kChunk j + kChunk g of token n, for each step j.
    static constexpr uint32_t kChunk = KV == LK_F32 ? 4 : 8;
    static constexpr uint32_t kSteps = kD / (4 * kChunk);
    static constexpr uint32_t kChunkWords = kChunk * kElem / 4;
    // V: lane (g, n) loads dims kVDims n .. +kVDims of tokens 4g + r, in pieces that lie wholly
    // below or past head_dim (a multiple of 8).
    static constexpr uint32_t kVDims = kD / 16;
    static constexpr uint32_t kPiece = KV == LK_F32 ? (kVDims < 4 ? kVDims : 4) : (kVDims < 8 ? kVDims : 8);
    static constexpr uint32_t kPieces = kVDims / kPiece;
    static constexpr uint32_t kPieceBytes = kPiece * kElem;
    static constexpr uint32_t kPieceWords = kPieceBytes < 4 ? 1 : kPieceBytes / 4;
    // Tiles in flight per wave, as the registers allow.
    static constexpr int kRing = kD == 256 ? 1 : 2;
};

template <int KV, int QF, int kD>
struct TokenTile {
    using Shape = TileShape<KV, QF, kD>;
    uint32_t k[Shape::kSteps][Shape::kChunkWords];
    uint32_t v[4][Shape::kPieces * Shape::kPieceWords];
    int32_t k_shift;      // FP8: of token n's group
    int32_t shifts[4];    // FP8: of tokens 4g + r, K low half, V high half
};

// A shift the FP8 fast path takes: the code becomes BF16 unscaled and 2^shift goes into the score
// or the weight. Others are decoded exactly with the shift included.
__device__ __forceinline__ bool tile_shift_is_plain(int32_t shift) { return shift >= -64 && shift <= 64; }

// Two E4M3 codes (the low or high half of `word`) times 2^shift as a BF16 pair, as decode_e4m3 gives
// them (largest finite value on overflow, signed zero below BF16's normals, 0x7FC0 for NaN), in a
// few float operations: the product of a 4-bit significand and a power of two is exact.
__device__ __forceinline__ uint32_t scaled_fp8_pair(uint32_t word, bool high, int32_t shift) {
    const codec_f32x2 codes = high ? __builtin_amdgcn_cvt_pk_f32_fp8(int(word), true) : __builtin_amdgcn_cvt_pk_f32_fp8(int(word), false);
    auto bits_of = [&](float code) __attribute__((always_inline)) {
        const uint32_t bits = __float_as_uint(__builtin_amdgcn_ldexpf(code, shift));
        uint32_t magnitude = bits & 0x7FFFFFFFu;
        const bool nan = magnitude > 0x7F800000u;
        magnitude = magnitude < 0x00800000u ? 0u : min(magnitude, 0x7F7F0000u);
        return nan ? 0x7FC00000u : (bits & 0x80000000u) | magnitude;
    };
    return bits_of(codes.x) >> 16 | bits_of(codes.y);
}

// kWhole: head_dim is kD itself.
template <int KV, int QF, int kD, bool kWhole>
__global__ __launch_bounds__(kD == 256 && (KV == LK_F32 || QF == LK_F32) ? 256 : 512) void decode_split_tiles(DecodeArgs a) {
    using Shape = TileShape<KV, QF, kD>;
    using Tile = TokenTile<KV, QF, kD>;
    constexpr bool kF32 = Shape::kF32;
    constexpr uint32_t kElem = Shape::kElem, kChunk = Shape::kChunk, kSteps = Shape::kSteps, kVDims = Shape::kVDims;
    // Dynamic LDS: the split's block ids and (FP8) shifts, then the merge of the waves' states.
    extern __shared__ __align__(16) uint32_t lds_words[];
    const uint32_t waves = blockDim.x / kWave;
    const uint32_t lane = threadIdx.x % kWave;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const uint32_t g = lane / 16, n = lane % 16;

    // KV head (and chunk of 16 query heads) fastest, then the split, then the sequence.
    const uint32_t chunks = (a.groups + kMaxHeads - 1) / kMaxHeads;
    const uint32_t units = a.kv_heads * chunks;
    const uint32_t unit = blockIdx.x % units;
    const uint32_t split = (blockIdx.x / units) % a.splits;
    const uint32_t seq = blockIdx.x / (units * a.splits);
    const uint32_t kv_head = unit / chunks;
    const uint32_t head0 = kv_head * a.groups + (unit % chunks) * kMaxHeads;  // first query head
    const uint32_t heads = min(kMaxHeads, a.groups - (unit % chunks) * kMaxHeads);

    // The ids (and FP8 shifts) are loaded before the length is known, bounded by the table alone.
    const uint32_t first = split * a.bps;
    const uint32_t listed = min(a.bps, a.table_width - first);
    const uint64_t head_tile = uint64_t(a.layer) * a.kv_heads + kv_head;
    const uint64_t v_group = uint64_t(a.layers) * a.kv_heads + head_tile;
    const uint64_t group_elems = uint64_t(a.slots) * a.head_dim;
    const uint64_t block_elems = 2ull * a.layers * a.kv_heads * group_elems;
    uint32_t* s_ids = lds_words;
    uint32_t* s_shifts = lds_words + a.bps;
    const int32_t* row_ids = a.table + uint64_t(seq) * a.table_stride + first;
    const int32_t my_id = row_ids[threadIdx.x < listed ? threadIdx.x : 0];
    const int32_t length = a.lengths[uint64_t(seq) * a.lengths_stride];
    const uint32_t nblocks = blocks_of(length, a.slots);
    const bool writes_out = a.out != nullptr;
    if (first >= nblocks && !writes_out) return;
    const uint32_t count = first < nblocks ? min(a.bps, nblocks - first) : 0;
    const uint32_t tokens = min(uint32_t(length) - first * a.slots, count * a.slots);  // of this split
    // At most 256 ids and at least 256 threads.
    if (threadIdx.x < count) {
        s_ids[threadIdx.x] = uint32_t(my_id);
        if constexpr (KV == LK_FP8_RECORD) {
            const uint16_t* shifts = reinterpret_cast<const uint16_t*>(a.pool + uint64_t(uint32_t(my_id)) * a.block_bytes + block_elems);
            s_shifts[threadIdx.x] = uint32_t(shifts[head_tile]) | uint32_t(shifts[v_group]) << 16;
        }
    }

    // B operand of QK: query head n, the dims lane group g of K holds for each step; zero for
    // heads past the group and dims past head_dim.
    constexpr uint32_t kQWords = kF32 ? kChunk : 4;  // per step: FP32 values, or BF16 pairs
    uint32_t qt[kSteps][kQWords];
#pragma unroll
    for (uint32_t j = 0; j < kSteps; ++j) {
        const uint32_t dim = 4 * kChunk * j + kChunk * g;
#pragma unroll
        for (uint32_t i = 0; i < kQWords; ++i) qt[j][i] = 0;
        if (n < heads && dim < a.head_dim) {
            const uint64_t at = (uint64_t(seq) * a.query_heads + head0 + n) * a.head_dim + dim;
            const uint8_t* q = static_cast<const uint8_t*>(a.q) + at * (QF == LK_F32 ? 4 : 2);
            if constexpr (QF == LK_F32) {
#pragma unroll
                for (uint32_t i = 0; i < kQWords; i += 4) load_words<16>(qt[j] + i, q + 4 * i);
            } else if constexpr (kF32) {
                uint32_t w[kQWords / 2];
                load_words<2 * kQWords>(w, q);
#pragma unroll
                for (uint32_t i = 0; i < kQWords; ++i) qt[j][i] = i % 2 ? w[i / 2] & 0xFFFF0000u : w[i / 2] << 16;
            } else {
                load_words<16>(qt[j], q);
            }
        }
    }
    __syncthreads();

    const uint32_t tiles = (tokens + kTileTokens - 1) / kTileTokens;
    const uint32_t mine = tiles > wave ? (tiles - wave + waves - 1) / waves : 0;
    const uint32_t row_bytes = a.head_dim * kElem;
    const uint64_t k_base = head_tile * group_elems * kElem, v_base = v_group * group_elems * kElem;
    const uint8_t* zeros = reinterpret_cast<const uint8_t*>(zero_row);
    // Block and slot of a token of this split (token / slots by a multiply: tokens of a split are
    // below 2^18 and slots at most 1,024, so the rounded-up reciprocal is exact).
    auto block_of = [&](uint32_t token) __attribute__((always_inline)) { return a.slots == 1 ? token : __umulhi(token, a.slots_inverse); };

    // Row of token n of a tile (K, then V): lane (g, n) finds it, the V loads take their four
    // tokens' from the lanes that have them. The addresses are made opaque so that the choice
    // between a row and the zeros stays a select.
    const uint64_t zeros_at = reinterpret_cast<uint64_t>(zeros);
    uint32_t from_lane[4];
#pragma unroll
    for (uint32_t r = 0; r < 4; ++r) from_lane[r] = 4 * (4 * g + r);
    // Dims past head_dim: their lanes read dims that exist instead; K's are masked off when used, V's
    // make outputs that nothing stores.
    auto dim_of = [&](uint32_t dim) __attribute__((always_inline)) { return kWhole || dim < a.head_dim ? dim : 0; };
    auto fetch = [&](Tile& tile, uint32_t i) __attribute__((always_inline)) {
        const uint32_t token = kTileTokens * (wave + i * waves) + n;
        const bool live = i < mine && token < tokens;
        const uint32_t safe = live ? token : 0;
        const uint32_t block = block_of(safe), slot = safe - block * a.slots;
        uint64_t k_row = reinterpret_cast<uint64_t>(a.pool) + uint64_t(s_ids[block]) * a.block_bytes + (k_base + slot * row_bytes);
        uint64_t v_row = k_row + (v_base - k_base);
        asm volatile("" : "+v"(k_row), "+v"(v_row));
        k_row = live ? k_row : zeros_at;
        v_row = live ? v_row : zeros_at;
        uint32_t packed_shifts = 0;
        if constexpr (KV == LK_FP8_RECORD) {
            packed_shifts = s_shifts[block];
            tile.k_shift = int32_t(int16_t(uint16_t(packed_shifts)));
        }
        const uint8_t* k_at = reinterpret_cast<const uint8_t*>(k_row);
#pragma unroll
        for (uint32_t j = 0; j < kSteps; ++j) load_words<kChunk * kElem>(tile.k[j], k_at + dim_of(4 * kChunk * j + kChunk * g) * kElem);
#pragma unroll
        for (uint32_t r = 0; r < 4; ++r) {
            const uint32_t lo = uint32_t(__builtin_amdgcn_ds_bpermute(int(from_lane[r]), int(uint32_t(v_row))));
            const uint32_t hi = uint32_t(__builtin_amdgcn_ds_bpermute(int(from_lane[r]), int(uint32_t(v_row >> 32))));
            const uint8_t* v_at = reinterpret_cast<const uint8_t*>(uint64_t(hi) << 32 | lo);
            if constexpr (KV == LK_FP8_RECORD) tile.shifts[r] = __builtin_amdgcn_ds_bpermute(int(from_lane[r]), int(packed_shifts));
#pragma unroll
            for (uint32_t p = 0; p < Shape::kPieces; ++p)
                load_words<Shape::kPieceBytes>(tile.v[r] + p * Shape::kPieceWords, v_at + dim_of(kVDims * n + Shape::kPiece * p) * kElem);
        }
    };

    float m = -INFINITY, l = 0.0f;
    f32x4 o[kVDims];
#pragma unroll
    for (uint32_t e = 0; e < kVDims; ++e) o[e] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

    // kProducts: PV in FP32 products of the whole weights (see the second pass below).
    auto consume = [&](Tile& tile, uint32_t i, auto products) __attribute__((always_inline)) {
        constexpr bool kProducts = kF32 || decltype(products)::value;
        const uint32_t token0 = kTileTokens * (wave + i * waves);
        // K and V as FP32 words or BF16 pairs. FP8 codes become BF16 unscaled, or (any shift of the
        // tile out of the plain range: a wave-uniform branch) are decoded with their shifts.
        constexpr uint32_t kPairs = kVDims / 2;
        constexpr uint32_t kValueWords = KV == LK_F32 ? kVDims : (KV == LK_FP8_RECORD && kPairs < 2 ? 2 : kPairs);
        uint32_t kb[kSteps][4], vw[4][kValueWords];
        bool exact = false;
        if constexpr (KV == LK_FP8_RECORD) {
            constexpr uint32_t kCodeWords = kVDims < 4 ? 1 : kVDims / 4;
            auto convert = [&](auto decoded) __attribute__((always_inline)) {
                auto pair = [&](uint32_t word, bool high, int32_t shift) __attribute__((always_inline)) {
                    if constexpr (decltype(decoded)::value) return scaled_fp8_pair(word, high, shift);
                    else return fp8_pair(word, high, false, 0);
                };
#pragma unroll
                for (uint32_t j = 0; j < kSteps; ++j)
#pragma unroll
                    for (int x = 0; x < 4; ++x) kb[j][x] = pair(tile.k[j][x / 2], x % 2 == 1, tile.k_shift);
#pragma unroll
                for (int r = 0; r < 4; ++r)
#pragma unroll
                    for (uint32_t x = 0; x < 2 * kCodeWords; ++x) vw[r][x] = pair(tile.v[r][x / 2], x % 2 == 1, tile.shifts[r] >> 16);
            };
            bool plain = true;
#pragma unroll
            for (int r = 0; r < 4; ++r)
                plain = plain && tile_shift_is_plain(int16_t(uint16_t(tile.shifts[r]))) && tile_shift_is_plain(tile.shifts[r] >> 16);
            exact = !__all(plain);
            if (__builtin_expect(exact, 0)) {
                asm volatile("" ::: "memory");
                convert(std::true_type{});
            } else {
                convert(std::false_type{});
            }
        } else {
#pragma unroll
            for (uint32_t j = 0; j < kSteps; ++j)
#pragma unroll
                for (int x = 0; x < 4; ++x) kb[j][x] = tile.k[j][x];
#pragma unroll
            for (int r = 0; r < 4; ++r)
#pragma unroll
                for (uint32_t x = 0; x < kValueWords; ++x) vw[r][x] = tile.v[r][x];
        }

        if constexpr (!kWhole) {
#pragma unroll
            for (uint32_t j = 0; j < kSteps; ++j)
#pragma unroll
                for (int x = 0; x < 4; ++x) kb[j][x] = 4 * kChunk * j + kChunk * g < a.head_dim ? kb[j][x] : 0u;
        }

        f32x4 s = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (uint32_t j = 0; j < kSteps; ++j) {
            if constexpr (!kF32) {
                s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(kb[j][0], kb[j][1], kb[j][2], kb[j][3]),
                                                            as_bf16x8(qt[j][0], qt[j][1], qt[j][2], qt[j][3]), s, 0, 0, 0);
            } else {
#pragma unroll
                for (uint32_t c = 0; c < kChunk; ++c) {
                    const float value = KV == LK_F32 ? __uint_as_float(kb[j][c]) : (c % 2 ? bf16_hi(kb[j][c / 2]) : bf16_lo(kb[j][c / 2]));
                    s = __builtin_amdgcn_mfma_f32_16x16x4f32(value, __uint_as_float(qt[j][c]), s, 0, 0, 0);
                }
            }
        }

        float score[4], v_factor[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            float factor = a.scale_log2;
            v_factor[r] = 1.0f;
            if constexpr (KV == LK_FP8_RECORD) {
                if (!exact) {
                    factor *= pow2(int16_t(uint16_t(tile.shifts[r])));
                    v_factor[r] = pow2(tile.shifts[r] >> 16);
                }
            }
            score[r] = token0 + 4 * g + r < tokens ? s[r] * factor : -INFINITY;
        }
        const float top = max_over_lane_groups(fmaxf(fmaxf(score[0], score[1]), fmaxf(score[2], score[3])));
        // The running max is raised only when a score passes it by more than 2^8 (see
        // decode_split_mfma).
        if (__builtin_expect(__any(top > m + kRescaleThreshold), 0)) {
            asm volatile("" ::: "memory");
            const float next = top > m + kRescaleThreshold ? top : m;
            const float alpha = merge_weight(m, next);
            m = next;
            l *= alpha;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float factor = __shfl(alpha, int(4 * g + r), kWave);
#pragma unroll
                for (uint32_t e = 0; e < kVDims; ++e) o[e][r] *= factor;
            }
        }
        float p[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            p[r] = score[r] == -INFINITY ? 0.0f : exp2_fast(score[r] - m);
            l += p[r];
            p[r] *= v_factor[r];
        }

        if constexpr (kProducts) {
#pragma unroll
            for (int r = 0; r < 4; ++r)
#pragma unroll
                for (uint32_t e = 0; e < kVDims; ++e) {
                    const float value = KV == LK_F32 ? __uint_as_float(vw[r][e]) : (e % 2 ? bf16_hi(vw[r][e / 2]) : bf16_lo(vw[r][e / 2]));
                    o[e] = __builtin_amdgcn_mfma_f32_16x16x4f32(p[r], value, o[e], 0, 0, 0);
                }
        } else {
            // The weights as three BF16 parts, cut (not rounded) from the top: exact, and none negative.
            uint32_t part[3][2];
#pragma unroll
            for (int half = 0; half < 2; ++half) {
                float x0 = p[2 * half], x1 = p[2 * half + 1];
#pragma unroll
                for (int k = 0; k < 3; ++k) {
                    part[k][half] = __builtin_amdgcn_perm(__float_as_uint(x1), __float_as_uint(x0), 0x07060302u);
                    x0 -= bf16_lo(part[k][half]);
                    x1 -= bf16_hi(part[k][half]);
                }
            }
            // Both steps are the same instruction: with 16x16x16 on the result of 16x16x32 the first
            // step's product was missing from the sum (no wait states stand between the two in the
            // assembly; the cause was not established).
            const bf16x8 p_top = as_bf16x8(part[0][0], part[0][1], part[1][0], part[1][1]);
            const bf16x8 p_low = as_bf16x8(part[2][0], part[2][1], 0u, 0u);
#pragma unroll
            for (uint32_t e = 0; e < kVDims; ++e) {
                const uint32_t select = (e & 1) ? 0x07060302u : 0x05040100u;
                const uint32_t b01 = __builtin_amdgcn_perm(vw[1][e / 2], vw[0][e / 2], select);
                const uint32_t b23 = __builtin_amdgcn_perm(vw[3][e / 2], vw[2][e / 2], select);
                const bf16x8 values = as_bf16x8(b01, b23, b01, b23);
                o[e] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(p_top, values, o[e], 0, 0, 0);
                o[e] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(p_low, values, o[e], 0, 0, 0);
            }
        }
    };

    // A ring of register tiles, each refilled as soon as it is consumed (past the wave's last
    // tile with zeros, so that no load is conditional).
    constexpr int kRing = Shape::kRing;
    Tile ring[kRing];
    if (mine > 0) {
#pragma unroll
        for (int d = 0; d < kRing; ++d) fetch(ring[d], uint32_t(d));
        for (uint32_t i = 0; i < mine; i += kRing) {
#pragma unroll
            for (int d = 0; d < kRing; ++d) {
                if (i + d < mine) consume(ring[d], i + d, std::false_type{});
                fetch(ring[d], i + d + kRing);
            }
        }
    }
    // Zero parts of a weight (its low ones often are, and half of p_low is) make NaN of an infinite V, where
    // the weight itself makes the infinity: BF16 pools with a NaN in a sum take their tiles again, as
    // products in FP32, and a NaN that stays is the result's own. (FP8 codes hold no infinity.)
    if constexpr (!kF32 && KV == LK_BF16) {
        bool nan = false;
#pragma unroll
        for (uint32_t e = 0; e < kVDims; ++e)
#pragma unroll
            for (int r = 0; r < 4; ++r) nan = nan || o[e][r] != o[e][r];
        if (__builtin_expect(__any(nan), 0)) {
            m = -INFINITY;
            l = 0.0f;
#pragma unroll
            for (uint32_t e = 0; e < kVDims; ++e) o[e] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            for (uint32_t i = 0; i < mine; ++i) {
                fetch(ring[0], i);
                consume(ring[0], i, std::true_type{});
            }
        }
    }

    // The waves' states meet in LDS, at most 128 dims at a time.
    constexpr uint32_t kPass = kD < 128 ? kD : 128, kPasses = kD / kPass, kPassDims = kVDims / kPasses;
    float* s_acc = reinterpret_cast<float*>(lds_words + (KV == LK_FP8_RECORD ? 2 : 1) * a.bps);  // [waves][heads][kPass]
    float* s_m = s_acc + waves * heads * kPass;                                                 // [waves][heads]
    float* s_l = s_m + waves * heads;
    l += __shfl_xor(l, 16, kWave);
    l += __shfl_xor(l, 32, kWave);
    if (g == 0 && n < heads) {
        s_m[wave * heads + n] = m;
        s_l[wave * heads + n] = l;
    }
#pragma unroll
    for (uint32_t pass = 0; pass < kPasses; ++pass) {
        if (pass > 0) __syncthreads();
        // Entry (wave, head, kPassDims n + e) of this pass is dim kVDims n + kPassDims pass + e.
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            if (4 * g + r < heads) {
#pragma unroll
                for (uint32_t e = 0; e < kPassDims; ++e) s_acc[(wave * heads + 4 * g + r) * kPass + kPassDims * n + e] = o[kPassDims * pass + e][r];
            }
        }
        __syncthreads();
        for (uint32_t idx = threadIdx.x; idx < heads * kPass; idx += blockDim.x) {
            const uint32_t h = idx / kPass, at = idx % kPass;
            const uint32_t d = kVDims * (at / kPassDims) + kPassDims * pass + at % kPassDims;
            float best = -INFINITY;
            for (uint32_t w = 0; w < waves; ++w) best = fmaxf(best, s_m[w * heads + h]);
            float sum = 0.0f, lsum = 0.0f;
            for (uint32_t w = 0; w < waves; ++w) {
                const float weight = merge_weight(s_m[w * heads + h], best);
                sum += s_acc[(w * heads + h) * kPass + at] * weight;
                lsum += s_l[w * heads + h] * weight;
            }
            if (d >= a.head_dim) continue;
            const uint64_t row = uint64_t(seq) * a.query_heads + head0 + h;
            if (writes_out) {  // the row's only split
                const float value = sum * (1.0f / lsum);
                if constexpr (QF == LK_BF16) reinterpret_cast<uint16_t*>(a.out)[row * a.head_dim + d] = to_bf16(value);
                else reinterpret_cast<float*>(a.out)[row * a.head_dim + d] = value;
                continue;
            }
            const uint64_t slot = row * a.splits + split;
            a.partial_acc[slot * a.head_dim + d] = sum;
            if (d == 0) {
                a.partial_ml[2 * slot] = best;
                a.partial_ml[2 * slot + 1] = lsum;
            }
        }
    }
}

// Dynamic LDS of a launch: ids, FP8 shifts, then the merge.
inline uint32_t tiles_lds_bytes(const DecodeArgs& a, int kv, uint32_t waves) {
    const uint32_t pass = a.head_dim <= 32 ? 32 : (a.head_dim <= 64 ? 64 : 128);
    const uint32_t heads = a.groups < kMaxHeads ? a.groups : kMaxHeads;
    return 4 * ((kv == LK_FP8_RECORD ? 2 : 1) * a.bps + waves * heads * (pass + 2));
}

}  // namespace lk

#endif  // LAYOVER_AMD_DECODE_TILES_H
