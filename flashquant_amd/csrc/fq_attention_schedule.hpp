// Order and split of the workgroups of the fused attention kernel.
//
// A workgroup's time is a fixed part (the two rotations, about eight tiles' worth) plus its key tiles, and
// under a causal mask or in a batch of prompts, later chunks and single queries the tiles differ by two orders of
// magnitude.  Nothing on the host knows the lengths, so every workgroup works out from them which piece of the work is
// its own:
//   * work is handed out longest first (the workgroups of a KV-head group in the order of their linear index), so that
//     the short ones fill the end of the launch (up to kOrderSeqs sequences);
//   * where a sequence's keys are long for its few queries (`split_w`, `max_pieces`, set by the host from what it
//     knows), they are cut into pieces of about the share of a CU; the pieces leave partial results, combined by a
//     launch of their own.
// So the bits of a row depend on the batch around it (the pieces on the lengths, their sum, the longest context that the host
// allows for and the number of CUs): within rounding, and the same for the same call.
// Measured (MI355X, bf16, 32 query heads over 8 KV heads of 128): a batch of 12 with six prompts, three later chunks and
// three single queries, 10,556 new tokens, 467 us in grid order and 385 us longest first; one query over 4 x 2500 tokens of a
// ring buffer 67 us in one workgroup per KV head, 22 us in 8 pieces (20 with the combine's columns shared), over 1 x 16,384 tokens 31 us in 32 pieces (369 us
// before the kernel cut contexts).
// Everything here is arithmetic on the lengths alone: the same in every workgroup and in the combine launch.
#pragma once

#include <cstdint>

#if defined(__HIPCC__)
#define FQ_HD __host__ __device__ __forceinline__
#else
#define FQ_HD inline
#endif

namespace fq {

// The shortest piece, in tiles of 64 keys.  Pieces go to CUs that have nothing else to do, so a piece costs its rows in
// the combine (2 KB a query head block of few queries) and not its prologue.  One query over a ring buffer of 4 x 2500 tokens,
// 32 heads over 8: 30.2 us with at least 8 tiles a piece, 28.5 with 6, 26.0 with 5 and 25.9 with 4; 1 x 1300 tokens 34.5, 28.5,
// 27.1 and 25.8; 8 heads over 1 of 256 coordinates, 1 x 2000 tokens, 2 queries 78.5, 72.0, 67.9 and 58.1.  (Each is 1.5 to 2.5
// us less now that the host works out the pieces of contiguous keys.)
constexpr int kSplitMinTiles = 4;

// Batches of more sequences than this are not ordered.  Every workgroup finds its own item, and the search for the longest
// ones reads all lengths about seven times (the first 64 once): 20 us at 1024 sequences, where a workgroup's own time is 30 to 60.
// Beyond it a workgroup counts through the sequences once, or, where the grid has at most two places for every workgroup that
// the batch can need, its place says which sequence it is.  bf16, in us, ordered / not ordered, 32 query heads over 8 of 128, 8
// over 1 of 128, 16 over 4 of 256: 256 sequences, sixteen of them prompts of 32 to 512 tokens, the others one query over 100 to
// 2000, 433 / 437, 92 / 113, 587 / 736; 384 of them 709 / 657, 127 / 155, 917 / 1069; 512 988 / 882, 169 / 187, 1228 / 1366; 1024
// 1854 / 1337, 283 / 236, 1859 / 1737.  256 single queries over 100 to 1000 257 / 246, 56 / 48, 340 / 409, 1024 1637 / 982,
// 234 / 180, 1727 / 1542; 256 prompts of 30 to 300 tokens 687 / 590, 162 / 174, 817 / 865, 512 1686 / 1125, 383 / 327, 1693 / 1618.
// In the order of the grid, all sequences with as many workgroups as the longest, 1024 single queries took 2060.
constexpr int kOrderSeqs = 256;

// One sequence as the kernel sees it.
struct SeqShape {
    int NQ, NKV, qoff;       // queries, keys, position of the first query among the keys
    int units, W;            // (32 positions x one query head) units, workgroups of 8 units
    int all_tiles;
};

FQ_HD SeqShape make_seq_shape(int NQ, int NKV, int qoff, int G, int max_w) {
    SeqShape s;
    s.NQ = NQ > 0 ? NQ : 0;
    s.NKV = NKV;
    s.qoff = qoff;
    s.units = ((s.NQ + 31) >> 5) * G;
    s.W = (s.units + 7) >> 3;
    s.W = s.W < max_w ? s.W : max_w;
    s.all_tiles = (NKV + 63) >> 6;
    return s;
}

// Key tiles that the furthest row of workgroup x sees; does not decrease with x.
FQ_HD int tiles_of(const SeqShape& s, int x, int G, bool causal) {
    if (!causal) return s.all_tiles;
    const int last_unit = 8 * x + 7 < s.units - 1 ? 8 * x + 7 : s.units - 1;
    int pos = 32 * (last_unit / G) + 31;
    pos = pos < s.NQ - 1 ? pos : s.NQ - 1;
    const int t = ((s.qoff + pos) >> 6) + 1;
    return t < s.all_tiles ? t : s.all_tiles;
}

// First workgroup of the sequence with at least T tiles (W when there is none).
FQ_HD int first_with(const SeqShape& s, int T, int G, bool causal) {
    if (T <= 0) return 0;
    if (T > s.all_tiles) return s.W;
    if (!causal) return 0;
    const int64_t P = 64 * int64_t(T - 1) - s.qoff;      // the position whose row sees T tiles
    if (P <= 0) return 0;
    if (P > s.NQ - 1) return s.W;
    const int64_t b = P > 31 ? P / 32 : 0;               // its block of 32 positions: ceil((P - 31) / 32)
    const int64_t x = b * G / 8;                         // first x whose last unit 8 x + 7 reaches unit b G
    return x < s.W ? int(x) : s.W;
}

// What splitting saves and costs, in ns: a tile of 64 keys of the longest workgroup; what a sequence's rows cost in the combine
// however few they are; 256 rows that are combined, and each of their pieces, written and read.  Fitted on 1775 paged batches of equal sequences (1, 3 and 8
// of them, 1 to 1000 queries over 400 to 4000 keys, four head counts), each run in pieces and in one: with 33 queries and more
// the combine took 3 and 5 us up to 16 workgroups' worth of pieces and 8 and 17 us at 128 (64 and 128 coordinates).  At 256
// pieces won in all of them: the rows go through the combine there whether they are split or not.
struct SplitCost {
    int tile, fixed, rows, piece;
};
FQ_HD SplitCost split_cost(int D) {
    return D == 64 ? SplitCost{1400, 3000, 60, 15} : (D == 128 ? SplitCost{2100, 5000, 20, 70} : SplitCost{5200, 0, 0, 0});
}

// What the pieces of a batch follow from: the tiles of a CU's share of all work, and the rows that may have to be combined,
// in workgroups' worth of 256.
struct BatchWork {
    int share, slots;
};

// Pieces that every workgroup's keys of this sequence are cut into.  The plan allows them by the longest context possible, of
// which the sequence may have little: with more than 16 queries (those of fewer always gained) pieces have to save more
// than they cost.  Without this a paged batch with a table of 4096 tokens lost: 3 prompts of 400 tokens, 16 heads over 4
// of 128, 41 us in one piece and 57 in two; 8 of 400 on one KV head of 64 25 and 36.
FQ_HD int pieces_of(const SeqShape& s, const BatchWork& b, int split_w, int max_pieces, int G, bool causal, int D) {
    if (max_pieces < 2 || s.W == 0 || s.W > split_w) return 1;
    const int tiles = tiles_of(s, s.W - 1, G, causal);
    int n = (tiles + b.share / 2) / b.share;
    n = n < max_pieces ? n : max_pieces;
    if (n < 2) return 1;
    const SplitCost c = split_cost(D);
    if (s.NQ > 16 && int64_t(c.tile) * tiles * (n - 1) <= int64_t(n) * (c.fixed + int64_t(b.slots) * (c.rows + c.piece * n))) return 1;
    return n;
}

// The share of one of `slots` CUs: `tile_sum` tiles of all workgroups.
FQ_HD int share_of(uint32_t tile_sum, int slots) {
    const int s = int((tile_sum + uint32_t(slots) - 1) / uint32_t(slots));
    return s > kSplitMinTiles ? s : kSplitMinTiles;
}

// Whether any batch around this sequence could make it run in pieces.
FQ_HD bool may_split(const SeqShape& s, int split_w, int max_pieces, int G, bool causal, int D) {
    return pieces_of(s, BatchWork{kSplitMinTiles, 0}, split_w, max_pieces, G, causal, D) > 1;
}

// Workgroups x of the sequence whose pieces have at least T tiles: x >= this.
FQ_HD int first_piece_with(const SeqShape& s, int T, int pieces, int G, bool causal) {
    if (T <= 0) return 0;
    const int64_t whole = int64_t(T - 1) * pieces + 1;
    return whole > s.all_tiles ? s.W : first_with(s, int(whole), G, causal);
}

// What the host allows: workgroups per sequence that may be split and pieces per workgroup.  The first kind of batch
// leaves more than half of the CUs without work (few prompts, or the chunks of a few): every workgroup may be split as
// far as a round of workgroups goes, if the tiles saved (1.4, 2.1 and 5.2 us each at 64, 128 and 256 coordinates) outweigh the
// combine launch (6 us, 12 at 256) and its traffic (132 KB a workgroup and piece at 128, written and read): 16 heads over 4 of
// 64 coordinates, 5 queries over 520 keys 16.6 us in one piece, 19.9 in two; a prompt of 520 tokens at 256 88.1 and 90.5.  The second kind (`prompts`: sequences
// of one known length under a causal mask) is about one round of workgroups, the longest with twice the average work: two
// pieces, if half of the longest workgroup outweighs that traffic and the second prologues too.  (Whether the shares are
// uneven enough pieces_of decides; more workgroups than 4/3 of a round never are.)  8 heads x 6000 tokens of 256 coordinates,
// one KV head, 188 workgroups: 538 us in one piece, 336 us in two; 16 heads x 3001 tokens on 4 KV heads 307 and 220 us (203 later; with room for their expanded keys
// and values such prompts take another kernel: 136).  Else only
// sequences of one workgroup (single queries of a mixed batch) are.
struct SplitPlan {
    int split_w, max_pieces;
};
inline SplitPlan plan_split(int num_seqs, int H_KV, int max_w, int64_t max_tiles, int cus, int D, bool prompts) {
    SplitPlan none{0, 1};
    if (max_tiles < 2 * kSplitMinTiles) return none;
    auto pieces = [&](int64_t items) {
        int64_t n = cus / (items > 0 ? items : 1);
        n = n < max_tiles / kSplitMinTiles ? n : max_tiles / kSplitMinTiles;
        return int(n < 32 ? n : 32);
    };
    const int64_t items = int64_t(num_seqs) * H_KV * max_w;
    const int n = pieces(items);
    const double tile = split_cost(D).tile * 1e-3, slot = 0.033 * (D / 64), prologue = D == 256 ? 40.0 : 15.0;
    if (n >= 2) {
        const double saved = tile * double(max_tiles) * (1.0 - 1.0 / n), cost = (D == 256 ? 12.0 : 6.0) + slot * double(items) * n;
        if (saved > 1.3 * cost) return {max_w, n};
    } else if (prompts && 3 * items <= 4 * int64_t(cus)) {
        const double saved = tile * double(max_tiles) / 2, cost = 6.0 + slot * double(items) * 2 + prologue * double(items) / cus;
        if (saved > 1.3 * cost) return {max_w, 2};
    }
    if (max_w > 1) {
        const int n1 = pieces(int64_t(num_seqs) * H_KV);
        if (n1 >= 2) return {1, n1};
    }
    return none;
}

}  // namespace fq
