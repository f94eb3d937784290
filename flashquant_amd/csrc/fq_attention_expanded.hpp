// Parameter blocks, plan and launcher of the attention over expanded keys and values (fq_attention_expanded.hip), shared with the
// host entry points in fq_fused_attention.hip.
#pragma once

#include <cstddef>
#include <cstdint>

#if defined(__HIPCC__)
#include <hip/hip_runtime.h>
#ifndef FQ_HD
#define FQ_HD __host__ __device__ __forceinline__
#endif
#elif !defined(FQ_HD)
#define FQ_HD inline
#endif

namespace fq_host {
int device_cu_count();
}

namespace fq {

// One piece of a workgroup's work, written by the plan (fq_attention_expanded.hip): 128 rows over a part of their keys.
struct WorkPiece {
    int seq, q_first, NQ, NKV;
    int x, pieces, tile_base, slot;     // x: workgroup of the sequence | piece << 20; slot: of its first piece
};
struct WorkPlan {
    int* counts;                // pieces, workgroups in several pieces
    WorkPiece* items;
    WorkPiece* splits;
    int max_items, max_slots;   // of a KV head: places, pieces of workgroups that have several
    int cus, cu_slots;          // CUs, and workgroups that run at a time
};

// The keys: pairs of (batch, KV head) one behind the other, or sequences in the paged cache.
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
    uint8_t* images;            // (tile): TileCfg; tiles of a pair, or (tile, KV head) of a sequence, one behind the other
    int* flags;                 // (tile, side, block of 32 tokens): whether it holds rows of long norms
    int* exps;                  // the same, by token: the binary orders by which a row is stored smaller
    const int32_t* cu_seqlens_q;
    const int32_t* seq_lens;
    const int32_t* block_table;
    const uint8_t* cache;
    int max_blocks, num_blocks, bs_log2;
    // the plan of the second launch, if it has one
    bool planned;
    int num_seqs, H_KV, G, N_Q, causal;
    WorkPlan plan;
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
    bool paged;
    WorkPlan plan;              // items == nullptr: the workgroups of all pairs, in one piece
    float* part;                // slots of pieces
};

// Whether a call over contiguous keys runs on expanded ones, and the workspace that takes.  Expanding costs about 9 ns a tile of
// keys or values beyond the launch (6 us, most of it its start), and saves 15 us of rotations and 0.2 us a tile of every workgroup of
// 256 rows, so what counts is how many workgroups share a pair's keys.  Measured (bf16, causal, batch x query heads over KV heads x
// tokens; us here / on the kernel that dequantises): 128 coordinates 1 x 32 over 8 x 40 14 / 18, 1 x 32 over 8 x 700 28 / 41, 4 x 64
// over 8 x 4000 1138 / 1489, 256 coordinates 1 x 16 over 4 x 65 18 / 49, 64 coordinates 4 x 16 over 4 x 1500 43 / 66.  It stays there
//   * with 64 coordinates and few tokens, where the two launches cost what the one does (4 x 32 over 8 x 65 11.7 / 10.5, x 130 12.7
//     / 12.1);
//   * with few workgroups on the keys of very many pairs (4 x 32 heads of their own x 300 34 / 28, x 700 60 / 70), at 128 coordinates and
//     one workgroup a pair of as few as 56 (7 x 16 heads of their own x 20 15.6 / 14.3, 3 x 16 x 20 14.0 / 14.0);
//   * with many keys for few queries, which it cuts into pieces (33 queries over 8000 keys, 32 heads over 8, 154 / 37).
struct ExpandedPlan {
    int keys = 0, tiles = 0;        // of a pair; paged: tiles of all sequences at most
    int64_t per_chunk = 0;          // pairs whose images the workspace holds at a time; 0: not on this path
    int max_items = 0, max_slots = 0, cus = 0, cu_slots = 0;      // WorkPlan; no items: no plan
    size_t images = 0, flags = 0, exps = 0, plan = 0, bytes = 0;
};
constexpr int64_t kImageBytes = int64_t(1) << 30;      // images at a time: beyond it the pairs take turns
inline size_t round_256(size_t n) { return (n + 255) / 256 * 256; }
// The parts of the workspace, for `tiles` tiles in all.
inline void lay_out(ExpandedPlan& e, int64_t tiles, int H_KV, int D) {
    const int64_t tt = D == 256 ? 32 : 64;
    e.images = size_t(tiles) * size_t(4 * tt * D);
    e.flags = round_256(size_t(tiles) * (tt / 32) * 8);
    e.exps = round_256(size_t(tiles) * 2 * tt * 4);
    e.plan = e.max_items > 0 ? round_256(256 + (size_t(e.max_items) + e.max_slots / 2 + 1) * sizeof(WorkPiece)) : 0;
    e.bytes = e.images + e.flags + e.exps + e.plan + size_t(e.max_slots) * H_KV * 4 * (32 * D + 64) * 4;
}
// What a batch takes with pieces of at most `piece` tiles (those of the kernel: 32 keys at 256 coordinates), in ns, for the choice
// between them: the longest piece, slowed down while it shares its CU, or the share of a place; and what the rows of `split` pieces
// cost in the combine, written and read.  Tiles as measured on an empty chip, and beside a second workgroup twice that; rows at 3.5
// TB/s.  16 heads over 4 of 256 coordinates x 3001 tokens stay whole (144 us, 136 to 150 by card; in pieces of the share 151 beside the 144), 32
// over 8 of 128 x 1500 too (46 and 53); 8 over 1 x 4000 run in pieces (82 whole, 71).
constexpr int kPieceTiles = 4;                  // the shortest pieces, in tiles of 64 keys
struct PieceCost {
    int tile, rows;
};
FQ_HD PieceCost piece_cost(int D) { return D == 64 ? PieceCost{700, 19} : (D == 128 ? PieceCost{1100, 38} : PieceCost{1250, 76}); }
FQ_HD int64_t batch_ns(int64_t piece, int64_t share, int64_t items, int64_t split, int cus, int D, bool alike) {
    const PieceCost c = piece_cost(D);
    int64_t ns = c.tile * piece;
    if (D != 256 && items > cus) ns += c.tile * (piece < share ? piece : share) * 6 / 10;
    int64_t all = D == 256 ? c.tile * share : c.tile * share * 19 / 10;
    // Pieces of one length do not fill a last round of places (5291 queries over 12,235 keys without a mask, 4 heads over 1 of 256, 520 us
    // in two pieces a workgroup, 413 in three, 473 on the kernel that dequantises).
    if (alike && D == 256) all = c.tile * piece * ((items + cus - 1) / cus);
    return (ns > all ? ns : all) + (split > 0 ? 7000 + split * c.rows : 0);
}
// Tiles of `workgroups` workgroups, the first of which has `first` and the last `last` (2^38 where a batch is as large as it may be).
FQ_HD int64_t work_of(int64_t workgroups, int first, int last) { return (workgroups * (int64_t(first) + last) + 1) / 2; }
// The share of one of `places` of all KV heads' tiles.
FQ_HD int64_t share_of_work(int64_t work, int H_KV, int places) { return (work * H_KV + places - 1) / places; }
// The candidates: the longest workgroup's tiles in 1, 2, 3, 4, 6, 8, 12 and 16.
constexpr int kPieceChoices = 8;
FQ_HD int piece_choice(int i, int longest, int least) {
    const int n = i < 4 ? i + 1 : (i & 1 ? 8 : 6) * (i < 6 ? 1 : 2), piece = (longest + n - 1) / n;
    return piece > least ? piece : least;
}
// Room for the plan: the pieces of workgroups that have several are at most four times the workgroups that run at a time.
inline void add_plan(ExpandedPlan& e, int64_t workgroups, int H_KV, int D, int cus, bool split) {
    e.cus = cus;
    e.cu_slots = (D == 256 ? 1 : 2) * cus;
    e.max_slots = split ? 4 * cus / H_KV + 2 : 0;
    e.max_items = int(workgroups) + e.max_slots;
}
// The workgroups of a pair (128 rows each) and the tiles that they see, by numbers alone: counting them one by one for every choice
// cost the host 46 us a call (32 query heads over one KV head x 4096 tokens, alone 216 us, 201 before keys were expanded, 175 this way).
struct ContiguousWork {
    int64_t W, tiles;
    int step;                       // units from the first that sees a tile more to the next
    bool causal;
    int64_t with(int64_t t) const { return t > tiles ? 0 : (causal ? W - (t - 1) * step / 4 : W); }     // workgroups of t tiles and more
    int64_t all() const {
        int64_t n = 0;
        if (!causal) return W * tiles;
        for (int64_t t = 1; t <= tiles; ++t) n += with(t);
        return n;
    }
    int64_t items(int64_t piece) const {                    // pieces of at most `piece` tiles
        int64_t n = 0;
        for (int64_t t = 1; t <= tiles; t += piece) n += with(t);
        return n;
    }
    int64_t split(int64_t piece) const { return items(piece) - (W - with(piece + 1)); }      // those of workgroups that have several
};
inline ExpandedPlan plan_expanded(int64_t B, int H_KV, int64_t n_q, int64_t n_kv, int G, int D, bool causal) {
    ExpandedPlan e;
    if (n_q <= (D == 64 ? 192 : 16)) return e;
    const int64_t pairs = B * H_KV;
    const int64_t tt = D == 256 ? 32 : 64;
    const int64_t keys = causal && n_kv > n_q ? n_q : n_kv, tiles = (keys + tt - 1) / tt, per_pair = tiles * (4 * tt * D);
    if (per_pair > kImageBytes) return e;
    const int64_t W = ((n_q + 31) / 32 * G + 3) / 4, most = int64_t(1) << 23;      // workgroups of a pair, of a launch
    const int64_t blocks = (keys + 63) / 64;
    if (W > most) return e;
    if (W < 5 && pairs * blocks >= (D == 128 && (n_q + 31) / 32 * G <= 4 ? 56 : 128)) return e;
    if (blocks > 4 * W + 4 || (!causal && blocks > 12 && pairs * W < 128)) return e;
    e.keys = int(keys);
    e.tiles = int(tiles);
    e.per_chunk = kImageBytes / per_pair < most / W ? kImageBytes / per_pair : most / W;
    if (e.per_chunk > pairs) e.per_chunk = pairs;
    // In pieces where that is faster, the workgroups being few enough to be counted
    const int cus = fq_host::device_cu_count();
    if (e.per_chunk == pairs && B <= 256 && pairs * W <= 8 * cus && tiles > kPieceTiles) {
        const ContiguousWork work{W, tiles, int(tt / 32) * G, causal};
        const int64_t places = (D == 256 ? 1 : 2) * int64_t(cus), share = share_of_work(work.all(), int(pairs), int(places));
        int64_t whole = 0, best = 0;
        for (int i = 0; i < kPieceChoices; ++i) {
            const int64_t piece = piece_choice(i, int(tiles), kPieceTiles * 64 / int(tt)), items = work.items(piece);
            const int64_t ns = batch_ns(piece, share, pairs * items, pairs * work.split(piece), cus, D, !causal);
            if (i == 0) whole = best = ns;
            best = ns < best ? ns : best;
        }
        if (20 * best < 19 * whole) add_plan(e, B * W, H_KV, D, cus, true);
    }
    lay_out(e, e.per_chunk * tiles, H_KV, D);
    return e;
}

// The same for paged batches, of which the host knows the number of sequences, the tokens, the most of a sequence and the longest
// context possible.  It stays on the other kernel too
//   * with few queries under a wide block table (3 of its columns to 10 rows of a KV head);
//   * at 128 coordinates where that kernel runs all sequences in one round of its workgroups (256 rows each) and the keys are many for it.
//     Its round of up to 4 units of 32 rows a workgroup takes 15 us and more, of 5 to 8 units 23, several rounds 30.  Measured (bf16;
//     sequences x tokens, query heads over KV heads; us here / there): up to 4 units, from 32 blocks of 64 keys on, 12 x 6, 16 over 16,
//     17.4 / 15.3, 13 x 83, 16 over 16, 24.0 / 19.1, and below that 2 x 10, 8 over 8, 15.8 / 15.3; up to 8 units, from 384 blocks on (192
//     where every sequence has only one), 12 x 214, 16 over 16, 36.3 / 28.7, 57 x 17, 32 over 4, 24.9 / 23.4, and below that 2 of 213 (up
//     to 252), 4 over 4, 19.4 / 26.4; up to 12 units, from 640 blocks on, 8 x 380, 16 over 16, 35.4 / 32.5, 4 x 300, 32 over 32, 32.6 /
//     31.3, and below that 16 x 300, 8 over 8, 31.9 / 31.2.
// Of 18,000 batches of 1 to 256 sequences that the first line leaves 941 ran more than 3 % slower here (the worst 8 chunks of 93, 32 over
// 32, 37.1 / 25.5); the others leave 29 of them and refuse 130 that would have run more than 3 % faster here.  What is left is mostly
// chunks of 64 coordinates that two launches more do not pay for (2 % of those; 407 over 1551 tokens, 8 over 1, 32.3 / 26.9), which no line
// on these sizes tells from ones that gain.
inline bool one_round_is_faster(int64_t num_seqs, int64_t total_q, int64_t max_q, int64_t max_kv, int H_KV, int G, int D) {
    const int64_t cus = fq_host::device_cu_count(), pairs = num_seqs * H_KV, units = (max_q + 31) / 32 * G, blocks = (max_kv + 63) / 64;
    if (D != 128) return false;
    if (units <= 8) return pairs <= cus && pairs * blocks >= (units <= 4 ? 32 : (blocks == 1 ? 192 : 384));
    // workgroups of that kernel: a sequence has half a block of 32 queries and half a workgroup more than its tokens fill
    const int64_t most = num_seqs * ((units + 7) / 8), about = ((total_q / 16 + num_seqs) * G / 8 + num_seqs) / 2;
    return units <= 12 && (about < most ? about : most) * H_KV <= cus && pairs * blocks >= 640;
}
inline ExpandedPlan plan_expanded_paged(int64_t num_seqs, int64_t total_q, int64_t max_q, int64_t max_kv, int H_KV, int G, int D) {
    ExpandedPlan e;
    const int64_t tt = D == 256 ? 32 : 64, tiles = num_seqs * ((max_kv + tt - 1) / tt);
    if (num_seqs > 256 || total_q <= 0 || tiles * H_KV * (4 * tt * D) > 0x7fffffff) return e;
    if (10 * total_q * G < 3 * num_seqs * max_kv || (D == 64 && total_q < 256 * num_seqs)) return e;
    if (one_round_is_faster(num_seqs, total_q, max_q, max_kv, H_KV, G, D)) return e;
    const int64_t workgroups = (total_q / 32 + num_seqs) * G / 4 + num_seqs;
    if (workgroups * H_KV > (int64_t(1) << 23) || workgroups >= (1 << 20)) return e;
    e.tiles = int(tiles);
    e.per_chunk = 1;
    add_plan(e, workgroups, H_KV, D, fq_host::device_cu_count(), max_kv > 128 * kPieceTiles);
    lay_out(e, tiles * H_KV, H_KV, D);
    return e;
}

// `e` and `a` hold the operands; the rest is filled in from the plan.
int launch_attention_expanded(ExpandParams e, AttendParams a, const ExpandedPlan& ep, int D, int dtype, void* workspace, void* stream);

}  // namespace fq
