// Parameter blocks of the prefill kernels (prefill.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "common.h"

namespace plamo {

enum GemmEpilogue { GEMM_F32 = 0, GEMM_BF16 = 1, GEMM_SWIGLU = 2, GEMM_RAW = 3 };

struct GemmParams {
    const uint16_t* w;      // plain BF16 [m][k] or .p12 payload
    const uint32_t* table;  // .p12 block table
    const uint16_t* x;      // BF16 [tokens][k]
    float* y;               // F32: [tokens][m]
    uint16_t* y16;          // BF16: [tokens][m]; SWIGLU: [tokens][6144]
    int m, k, tokens;
};

struct RowsNormParams {
    const int32_t* tokens_in;  // embedding mode when set
    const uint16_t* embed;
    const uint16_t* in;        // residual mode: projection output [T][1536] BF16
    const uint16_t* g_post;
    float post_offset;
    uint16_t* x;               // residual stream [T][1536] BF16 (updated in place; every value
                               // is BF16-rounded, so the BF16 copy is lossless)
    const uint16_t* g_next;
    uint16_t* xn;              // next-norm output BF16 [T][1536] (optional)
    int tokens;                // set by launch_rows_norm
};

// Rows of one prefill pass that belong to one KV lane: rows token0 .. token0 + tokens - 1 are its
// tokens from position p0 on, and its query blocks (of 8 tokens) start at first_block.
struct PrefillSegment {
    int token0, tokens, first_block;
    uint32_t lane;  // KV slice, counted from the one the pass's keys and values point to
};
constexpr int PREFILL_SEGMENTS = MAX_ROWS;
struct PrefillSegments {
    int n;
    PrefillSegment s[PREFILL_SEGMENTS];
    // The segment of row t, or of query block b.  Its values are selected, not its index: kernel
    // arguments read at a computed index are a load that waits for the index.
    __host__ __device__ PrefillSegment of_token(int t) const {
        PrefillSegment g = s[0];
#pragma unroll
        for (int k = 1; k < PREFILL_SEGMENTS; ++k)
            if (k < n && t >= s[k].token0) g = s[k];
        return g;
    }
    __host__ __device__ PrefillSegment of_block(int b) const {
        PrefillSegment g = s[0];
#pragma unroll
        for (int k = 1; k < PREFILL_SEGMENTS; ++k)
            if (k < n && b >= s[k].first_block) g = s[k];
        return g;
    }
    // A single segment is the pass: its rows from 0 on, of the first KV slice.  Kernels then look
    // nothing up and move no pointer (flash of 3 global queries 8.1 -> 7.9 us, 61 local ones 8.76 ->
    // 8.67).
    bool valid() const { return n > 1 || (n == 1 && s[0].token0 == 0 && s[0].first_block == 0 && s[0].lane == 0); }
};

struct QkPrepParams {
    const uint16_t* qkv;       // [T][2304] BF16
    const uint16_t* q_norm;
    const uint16_t* k_norm;
    uint16_t* q16;             // out: [T][16][128] BF16, normalised and rotated queries
    uint16_t* keys;            // lane slice [capacity][128]
    uint16_t* values;
    uint16_t* keys_rot;        // local layers: lane slice [rot_rows][128] (null: none)
    uint32_t rot_rows;
    uint32_t capacity, p0;
    int tokens;
    PrefillSegments seg;
    int full;
    const uint32_t* local_rope;   // [2064][64] BF16 (cos | sin << 16)
    const uint32_t* global_rope;  // [context][64]
};

// Flash prefill splits the key tiles of a query block (8 tokens x 16 heads) over up to
// FLASH_PARTS workgroups; their partial results meet in a workspace.
constexpr int FLASH_PARTS = 3;
constexpr int FLASH_PART_TILES = 11;         // 64-key tiles a part aims at
__host__ __device__ inline int flash_blocks(int tokens) { return (tokens + 7) / 8; }
inline int flash_blocks(const PrefillSegments& g) { return g.s[g.n - 1].first_block + flash_blocks(g.s[g.n - 1].tokens); }
// One segment: `tokens` rows of the first KV slice.
inline PrefillSegments one_segment(int tokens) { return PrefillSegments{1, {{0, tokens, 0, 0u}}}; }
// workspace floats: per block and part, O^T [128 columns][128 dims] and (m, l) per column
// Key tiles (64 keys) that query block qb of a call attends to, and the parts they are split
// into (contiguous tile ranges, part q from q * tiles / parts).
__host__ __device__ inline int flash_block_tiles(int tokens, uint32_t p0, int full, int qb) {
    const int t0 = qb * 8, t1 = t0 + 8 < tokens ? t0 + 8 : tokens;
    const uint32_t plo = p0 + uint32_t(t0), khi = p0 + uint32_t(t1 - 1);
    const uint32_t klo = full ? 0u : (plo > uint32_t(WINDOW - 1) ? plo - uint32_t(WINDOW - 1) : 0u);
    return int((khi + 1 - klo + 63) / 64);
}
__host__ __device__ inline int flash_block_parts(int tiles) {
    const int parts = (tiles + FLASH_PART_TILES - 1) / FLASH_PART_TILES;
    return parts < FLASH_PARTS ? parts : FLASH_PARTS;
}
// The order in which workgroups take the (query block, part) items of a call: item w of the
// launch is item[w] (qb << 2 | part).  n = 0: workgroup w takes part w / blocks of block
// blocks - 1 - w % blocks (and returns if the block has fewer parts).
constexpr int FLASH_SCHEDULE_MAX = 780;  // the items of a 2048-token pass of four segments, at most
struct FlashSchedule {
    uint32_t n;
    uint16_t item[FLASH_SCHEDULE_MAX];
};
inline size_t flash_part_o_floats(int blocks) { return size_t(blocks) * FLASH_PARTS * 128 * 128; }
inline size_t flash_part_ml_floats(int blocks) { return size_t(blocks) * FLASH_PARTS * 128 * 2; }

struct FlashParams {
    const uint16_t* q;         // [T][16][128] BF16, normalised and rotated
    const uint16_t* keys;      // lane slice [capacity][128]
    const uint16_t* values;
    const uint32_t* local_rope;   // local layers: keys rotate with chunk-relative coordinates
    const uint16_t* keys_rot;  // local layers: lane slice [rot_rows][128] of keys rotated at their
                               // own position (null: rotate every key)
    uint32_t rot_rows;
    uint16_t* out;             // [T][2048] BF16
    uint32_t capacity, p0;
    PrefillSegments seg;
    int full;
    int blocks;                // query blocks of the pass (set by launch_flash_prefill)
    float* part_o;             // flash_part_o_floats(blocks)
    float* part_ml;            // flash_part_ml_floats(blocks)
    uint32_t* tickets;         // one per block, zero between launches
    const uint32_t* qsa_mask;  // global layers with QSA: token t's selected blocks of four keys
                               // (bit b of word t * qsa_words + b / 32); null: every key
    uint32_t qsa_words;
};

void launch_gemm(bool packed, GemmEpilogue epi, const GemmParams& p, hipStream_t s);
void launch_rows_norm(const RowsNormParams& p, int tokens, hipStream_t s);
void launch_qk_prep(const QkPrepParams& p, hipStream_t s);
void launch_flash_prefill(const FlashParams& p, hipStream_t s);
// Every segment's last row of `a` and `b` ([rows][1536] BF16) to rows 0 .. n - 1 of `a_out` and `b_out`.
void launch_gather_last(const uint16_t* a, const uint16_t* b, const PrefillSegments& seg, uint16_t* a_out, uint16_t* b_out,
                        hipStream_t s);

}  // namespace plamo
