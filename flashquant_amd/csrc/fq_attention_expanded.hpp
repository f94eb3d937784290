// Parameter blocks, plan and launcher of the attention over expanded keys and values (fq_attention_expanded.hip), shared with the
// host entry points in fq_fused_attention.hip.
#pragma once

#include <cstddef>
#include <cstdint>

namespace fq {

struct ExpandParams {
    const uint8_t* k_packed;    // (pairs, cap, D/2), a pair being one (batch, KV head)
    const float* k_norms;
    const uint8_t* v_packed;
    const float* v_norms;
    const float* centroids_k;
    const float* centroids_v;
    const float* rotation;
    int rot_col_major;
    int64_t k_cap, v_cap;
    int keys, tiles;            // keys of a pair, and the tiles they fill
    int pair0, pairs;           // the pairs of this launch
    uint8_t* images;            // (pair, tile): TileCfg
    int* flags;                 // (pair, tile, side, block of 32 tokens): whether it holds rows of long norms
    int* exps;                  // the same, by token: the binary orders by which a row is stored smaller
};

struct AttendParams {
    const uint16_t* q;
    uint16_t* out;
    const uint8_t* images;
    const int* flags;
    const int* exps;
    int H_Q, H_KV, G, N_Q, N_KV;
    int causal;
    float scale_log2e;
    int tiles, pair0, pairs, W;
    int round_slots;            // CUs
    bool out_wide;
};

// Whether a call over contiguous keys runs on expanded ones, and the workspace that takes.  Expanding costs about 9 ns a tile of
// keys or values beyond the launch (6 us, most of it its start), and saves 15 us of rotations and 0.2 us a tile of every workgroup of
// 256 rows, so what counts is how many workgroups share a pair's keys.  Measured (bf16, causal, batch x query heads over KV heads x
// tokens; us here / on the kernel that dequantises): 128 coordinates 1 x 32 over 8 x 40 14 / 18, 1 x 32 over 8 x 700 28 / 41, 4 x 64
// over 8 x 4000 1138 / 1489, 256 coordinates 1 x 16 over 4 x 65 18 / 49, 64 coordinates 4 x 16 over 4 x 1500 43 / 66.  It stays there
//   * with 64 coordinates and few tokens, where the two launches cost what the one does (4 x 32 over 8 x 65 11.7 / 10.5, x 130 12.7
//     / 12.1);
//   * with few workgroups on the keys of very many pairs (4 x 32 heads of their own x 300 34 / 28, x 700 60 / 70);
//   * with many keys for few queries, which it cuts into pieces (33 queries over 8000 keys, 32 heads over 8, 154 / 37).
struct ExpandedPlan {
    int keys = 0, tiles = 0;        // of a pair
    int64_t per_chunk = 0;          // pairs whose images the workspace holds at a time; 0: not on this path
    size_t images = 0, flags = 0, bytes = 0;
};
constexpr int64_t kImageBytes = int64_t(1) << 30;      // images at a time: beyond it the pairs take turns
inline ExpandedPlan plan_expanded(int64_t pairs, int64_t n_q, int64_t n_kv, int G, int D, bool causal) {
    ExpandedPlan e;
    const int64_t tt = D == 256 ? 32 : 64;
    const int64_t keys = causal && n_kv > n_q ? n_q : n_kv, tiles = (keys + tt - 1) / tt, per_pair = tiles * (4 * tt * D);
    if (per_pair > kImageBytes) return e;
    const int64_t W = ((n_q + 31) / 32 * G + 3) / 4, most = int64_t(1) << 23;      // workgroups of a pair, of a launch
    const int64_t blocks = (keys + 63) / 64;
    if (n_q <= (D == 64 ? 128 : 16) || W > most) return e;
    if (W < 5 && pairs * blocks > 256) return e;
    if (blocks > 4 * W + 4 || (!causal && blocks > 12 && pairs * W < 128)) return e;
    e.keys = int(keys);
    e.tiles = int(tiles);
    e.per_chunk = kImageBytes / per_pair < most / W ? kImageBytes / per_pair : most / W;
    if (e.per_chunk > pairs) e.per_chunk = pairs;
    e.images = size_t(e.per_chunk * per_pair);
    e.flags = (size_t(e.per_chunk * tiles) * (tt / 32) * 8 + 255) / 256 * 256;
    e.bytes = e.images + e.flags + size_t(e.per_chunk * tiles * 2 * tt) * 4;
    return e;
}

int launch_attention_expanded(const ExpandParams& e, const AttendParams& a, int D, int dtype, int64_t pairs, int64_t per_chunk,
                              void* stream);

}  // namespace fq
